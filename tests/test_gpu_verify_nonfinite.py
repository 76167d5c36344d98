"""Non-finite V scales in the verify kernels: a key that a query does not see may
hold any scale, and a visible key's NaN or infinity reaches the outputs of the
queries that see it (of the dims it scales), and no others."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from superl8_serve_amd import ops
from tests.kvcase import make_case
from tests.kvgpu import CODEBOOK, alloc, append, assert_close, t, to_np

pytestmark = pytest.mark.gpu

LAYOUTS = [("int8", 64), ("int8", 128), ("int8", 256), ("k8v3", 128), ("k8v3", 256)]
ROWS = [5, 20, 50]  # queries of 4 heads: one 32-row wave, a 128-row workgroup, more (256-row ones at head_dim 128)
PREFIX, BS = np.array([400, 150]), 32
BAD = (np.inf, np.nan, -np.inf)


def _case(kind, d, nq, window):
    case = make_case(70 + d + nq, 2, 8, 2, d, BS, PREFIX + nq)
    cache = alloc(kind, case.num_blocks, 2, BS, d)
    append(kind, t(case.k), t(case.v), cache, t(case.slots))
    q = t(np.random.default_rng(71).standard_normal((2, 8, nq, d)).astype(np.float16))
    fn = ops.attn_paged_verify if kind == "int8" else ops.attn_paged_verify_k8v3
    extra = () if kind == "int8" else (t(CODEBOOK),)
    width = case.block_table.shape[1] * BS

    def run():
        out = fn(q, *cache, *extra, t(case.block_table), t(PREFIX.astype(np.int32)), BS, max_context_len=width,
                 scale=case.scale, window=window)
        torch.cuda.synchronize()
        return to_np(out.float())

    return case, cache, run


@pytest.mark.parametrize("kind,d", LAYOUTS)
@pytest.mark.parametrize("nq", ROWS)
@pytest.mark.parametrize("window", [None, 61])
def test_scales_of_unseen_keys_change_nothing(kind, d, nq, window):
    """Past a row's last key, and below its window: bit-identical outputs."""
    case, cache, run = _case(kind, d, nq, window)
    clean = run()
    for b, p in enumerate(PREFIX):
        ends = -(-(p + nq) // BS) * BS
        below = range(0 if window is None else p - window)
        for pos in [*below, *range(p + nq, ends)]:
            blk, off = int(case.block_table[b, pos // BS]), pos % BS
            cache[1][blk, :, off] = cache[3][blk, :, off] = BAD[pos % 3]
    assert np.array_equal(run(), clean)


@pytest.mark.parametrize("kind,d", LAYOUTS)
@pytest.mark.parametrize("nq", ROWS)
@pytest.mark.parametrize("window", [None, 61])
@pytest.mark.parametrize("bad", BAD)
@pytest.mark.parametrize("draft", [-10, 2])  # a prefix key, and one that only queries from the third on see
def test_visible_scale_reaches_its_queries(kind, d, nq, window, bad, draft):
    case, cache, run = _case(kind, d, nq, window)
    clean = run()
    pos = int(PREFIX[0]) + draft
    scale = cache[3][int(case.block_table[0, pos // BS]), 0]
    scale[pos % BS] = bad if kind == "int8" else torch.tensor([1.0] * (d // 128 - 1) + [bad])
    got, first, dims = run(), max(draft, 0), 0 if kind == "int8" else d - 128
    assert np.isnan(got[0, :4, first:, dims:]).all() and np.isfinite(got[0, :4, first:, :dims]).all()
    assert np.array_equal(got[1], clean[1]) and np.array_equal(got[0, 4:], clean[0, 4:])
    if first:
        assert_close(got[0, :4, :first], clean[0, :4, :first].astype(np.float64), "queries before the draft")
