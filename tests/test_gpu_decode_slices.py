"""Rows of the decode cut into many slices, or fewer than the grid holds.

The combine of a split row reads its partials 16 at a time: rows of one below,
exactly and one above such a batch, and of several, against the oracle.
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
