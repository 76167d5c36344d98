"""Rows of the decode cut into many slices, or fewer than the grid holds.

The combine of a split row reads its partials 16 at a time: rows of one below,
exactly and one above such a batch, and of several, against the oracle; and
batches whose rows are too few or short for every workgroup to take a slice.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import kv_oracle as O
from tests import kvgpu as K
from tests.kvcase import make_case, oracle_fill_int8

pytestmark = pytest.mark.gpu


def _run(case, cache):
    out = K.decode("int8", K.t(case.q)[:, :, None, :], tuple(K.t(x) for x in cache), K.t(case.block_table),
                   K.t(case.lens.astype(np.int32)), case.block_size, int(case.lens.max()), case.scale)
    torch.cuda.synchronize()
    return out[:, :, 0, :]


@pytest.mark.parametrize("hq,d", [(1, 128), (4, 128), (16, 128), (2, 32), (8, 256)])
@pytest.mark.parametrize("segments", [2, 15, 16, 17, 33, 80])
def test_rows_of_many_partials(segments, hq, d, monkeypatch):
    """One KV head, slices of one tile: a row of 32 * segments - 5 tokens is
    that many partials; a second, shorter row shares the counters' line."""
    rows = [32 * segments - 5, 40]
    for name, value in (("WG_PER_HEAD", segments + 2), ("GHOST", 0), ("SLOT_SKEW", 0)):
        monkeypatch.setenv(f"S8KV_DECODE_{name}", str(value))
    case = make_case(11, 2, hq, 1, d, 32, rows)
    cache = oracle_fill_int8(case)
    ref = O.paged_decode(case.q, O.LayerCache(*cache), case.block_table, case.lens, case.scale)
    first = _run(case, cache)
    K.assert_close(K.to_np(first.float()), ref, f"{segments} segments")
    for _ in range(3):  # (the workspace may hold the last call's words)
        assert torch.equal(_run(case, cache), first)


@pytest.mark.parametrize("kind", K.KINDS)
@pytest.mark.parametrize("rows", [[1], [31, 0, 33], [2900], [2000, 17], [700] * 9, [4, 5000, 4, 4]])
def test_least_slice_length(kind, rows, monkeypatch):
    """The default slicing gives a head fewer slices than the grid holds when
    its rows are few; the plan made for it gives the same output, and one
    slice per head the same within the rounding of the combine."""
    case = make_case(12, len(rows), 8, 2, 128, 32, rows)
    cache = K.alloc(kind, case.num_blocks, 2, 32, 128)
    K.append(kind, K.t(case.k), K.t(case.v), cache, K.t(case.slots))
    lens, table = K.t(case.lens.astype(np.int32)), K.t(case.block_table)
    q, longest = K.t(case.q)[:, :, None, :], int(case.lens.max())
    args = (table, lens, 32, longest, case.scale)
    new = [K.t(np.random.default_rng(3).standard_normal((len(rows), 2, 128)).astype(np.float16)) for _ in range(2)]
    out = K.decode_append(kind, q, *new, cache, *args)
    plan = K.decode_plan(kind, cache, table, lens, 32, case.num_q_heads, longest)
    assert torch.equal(out, K.decode_append(kind, q, *new, cache, *args, plan=plan))
    ref = O.paged_decode(case.q, K.layer(kind, [K.to_np(x) for x in cache]), case.block_table, case.lens, case.scale)
    K.assert_close(K.to_np(out[:, :, 0, :].float()), ref, f"rows {rows}")
    monkeypatch.setenv("S8KV_DECODE_WG_PER_HEAD", "1")
    one = K.decode(kind, q, cache, *args)
    K.assert_close(K.to_np(one[:, :, 0, :].float()), ref, f"rows {rows}, one slice")
