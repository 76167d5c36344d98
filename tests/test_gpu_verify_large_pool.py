"""Verify over pools past 4 GiB a layer, which run the 16-row kernel (tiles
through descriptors rebased per tile) at every head_dim and layout, against the
oracle on a compact copy of the blocks in use: chains and trees of several query
blocks, windows, fresh drafts, and key splits."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import kv_oracle as O
from superl8_serve_amd import _lib, ops
from tests.kvcase import make_case
from tests.kvgpu import CODEBOOK, alloc, append, assert_close, layer, t, to_np
from tests.test_gpu_limits import _edge_ids

pytestmark = pytest.mark.gpu

HQ, HKV, BS = 8, 2, 32
PREFIX = np.array([700, 33, 0, 511])


def _tree(rng, n):
    masks = np.zeros(n, np.uint64)
    for i in range(n):
        masks[i] = (masks[int(rng.integers(0, i))] if i else np.uint64(0)) | (np.uint64(1) << np.uint64(i))
    return masks.view(np.int64)


@pytest.mark.parametrize("kind,d", [("int8", 64), ("int8", 128), ("int8", 256), ("k8v3", 128), ("k8v3", 256)])
def test_verify_of_a_pool_past_4_gib(kind, d):
    nblk = (1 << 32) // (HKV * BS * d) + 70
    cache = alloc(kind, nblk, HKV, BS, d)
    lib = _lib.load()
    fn = ops.attn_paged_verify if kind == "int8" else ops.attn_paged_verify_k8v3
    extra = () if kind == "int8" else (t(CODEBOOK),)
    half = (1 << 31) // (HKV * BS * d)
    try:
        for nq, tree, window, fresh, splits in [
            (5, False, None, False, 0), (40, True, None, False, 1), (40, False, None, False, 3),
            (5, False, 61, False, 1), (40, True, 300, False, 2), (5, True, 61, True, 1), (40, False, 300, True, 3),
        ]:
            what = f"{kind} D={d} nq={nq} tree={tree} window={window} fresh={fresh} splits={splits}"
            case = make_case(800 + d + nq, len(PREFIX), HQ, HKV, d, BS, PREFIX + nq, outlier_channels=2)
            ids = _edge_ids(case, nblk, (2 * half, 2 * half - 1, half, 0, nblk - 2), np.random.default_rng(801))
            table = ids[case.block_table].astype(np.int32)
            append(kind, t(case.k), t(case.v), cache, t((ids[case.slots // BS] * BS + case.slots % BS).astype(np.int32)))
            host = layer(kind, tuple(to_np(x.index_select(0, t(ids))) for x in cache))
            qv = np.random.default_rng(802).standard_normal((len(PREFIX), HQ, nq, d)).astype(np.float16)
            lens = np.array([nq, nq - 2, nq, 1], np.int32)
            mask = np.stack([_tree(np.random.default_rng(803 + b), nq) for b in range(len(PREFIX))]) if tree else None
            starts = np.concatenate([[0], np.cumsum(case.lens)])
            idx = np.stack([starts[b] + PREFIX[b] + np.arange(nq) for b in range(len(PREFIX))])
            drafts = (case.k[idx], case.v[idx]) if fresh else None
            kw = dict(zip(("k_draft", "v_draft"), map(t, drafts))) if fresh else {}
            _lib.check(lib.s8kv_verify_set_splits(splits), "set_splits")
            out = fn(t(qv), *cache, *extra, t(table), t(PREFIX.astype(np.int32)), BS, query_lens=t(lens),
                     tree_mask=None if mask is None else t(mask), max_context_len=int(case.lens.max()),
                     scale=case.scale, window=window, **kw)
            torch.cuda.synchronize()
            ref = O.paged_verify(qv, host, case.block_table, PREFIX, case.scale, query_lens=lens, tree_mask=mask,
                                 window=window, fresh_drafts=drafts)
            got = to_np(out.float())
            for b, n in enumerate(lens):
                assert not got[b, :, n:].any(), f"{what}: row {b}, outputs past its {n} queries"
            assert_close(got, ref, what)
    finally:
        lib.s8kv_verify_set_splits(0)
        del cache
        torch.cuda.empty_cache()
