"""The verify kernels' units on the GPU against the oracle: every (sequence, KV
head, query block, key split) is computed by exactly one workgroup whatever the
number of pairs (dispatch takes them gcd(pairs, 8) at a time), and equal key
splits of rows of different lengths combine to the whole row's result."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import kv_oracle as O
from superl8_serve_amd import _lib, ops
from tests.kvcase import make_case
from tests.kvgpu import CODEBOOK, alloc, append, assert_close, layer, t, to_np

pytestmark = pytest.mark.gpu


def _tree(rng, n):
    """Ancestor bits of a random tree of n nodes."""
    masks = np.zeros(n, np.uint64)
    for i in range(n):
        masks[i] = np.uint64(1) << np.uint64(i)
        if i:
            masks[i] |= masks[int(rng.integers(0, i))]
    return masks.view(np.int64)


def _check(seed, kind, hq, hkv, d, bs, prefix, nq, what, query_lens=None, window=None, tree=False):
    prefix = np.asarray(prefix)
    case = make_case(seed, len(prefix), hq, hkv, d, bs, prefix + nq, outlier_channels=2 if d >= 128 else 0)
    cache = alloc(kind, case.num_blocks, hkv, bs, d)
    append(kind, t(case.k), t(case.v), cache, t(case.slots))
    qv = np.random.default_rng(seed + 1).standard_normal((len(prefix), hq, nq, d)).astype(np.float16)
    mask = np.stack([_tree(np.random.default_rng(seed + 2 + b), nq) for b in range(len(prefix))]) if tree else None
    fn = ops.attn_paged_verify if kind == "int8" else ops.attn_paged_verify_k8v3
    extra = () if kind == "int8" else (t(CODEBOOK),)
    out = fn(t(qv), *cache, *extra, t(case.block_table), t(prefix.astype(np.int32)), bs,
             query_lens=None if query_lens is None else t(np.asarray(query_lens, np.int32)),
             tree_mask=None if mask is None else t(mask), max_context_len=int(case.lens.max()), scale=case.scale,
             window=window)
    torch.cuda.synchronize()
    ref = O.paged_verify(qv, layer(kind, tuple(to_np(x) for x in cache)), case.block_table, prefix, case.scale,
                         query_lens=query_lens, window=window, tree_mask=mask)
    got = to_np(out.float())
    for b, n in enumerate([] if query_lens is None else query_lens):
        assert not got[b, :, n:].any(), f"{what}: row {b}, outputs past its {n} queries"
    assert_close(got, ref, what)


@pytest.mark.parametrize("batch,hkv", [(1, 1), (1, 4), (3, 1), (3, 2), (3, 4), (5, 3), (2, 8)])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_every_unit_of_any_pair_count(batch, hkv, d):
    """Several query blocks of 1, 3, 4, 6, 12, 15 and 16 pairs."""
    nq = 70
    _check(40 + batch * 8 + hkv, "int8", 4 * hkv, hkv, d, 16, [90 + 37 * b for b in range(batch)], nq,
           f"{batch} x {hkv} pairs, D={d}")


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("batch,hkv", [(1, 2), (7, 1), (8, 16)])  # (8, 16): enough pairs for 256-row blocks
def test_dense_units_of_any_pair_count(batch, hkv, d):
    rng = np.random.default_rng(60 + batch)
    lens = [400 - 53 * b for b in range(batch)]
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    hq = 4 * hkv
    q, k, v = (rng.standard_normal((cu[-1], h, d)).astype(np.float16) for h in (hq, hkv, hkv))
    out = to_np(ops.attn_varlen(t(q), t(k), t(v), t(cu), t(cu), max(lens), max(lens), causal=True,
                                scale=d ** -0.5).float())
    for b, n in enumerate(lens):
        qb, kb, vb = (torch.from_numpy(x[cu[b]:cu[b + 1]]).double().transpose(0, 1) for x in (q, k, v))
        kb, vb = kb.repeat_interleave(4, 0), vb.repeat_interleave(4, 0)
        s = (qb @ kb.transpose(1, 2)) * d ** -0.5
        s = s.masked_fill(~torch.ones((n, n), dtype=torch.bool).tril(), float("-inf"))
        assert_close(out[cu[b]:cu[b + 1]], (torch.softmax(s, -1) @ vb).transpose(0, 1).numpy(), f"sequence {b}")


@pytest.mark.parametrize("kind,d", [("int8", 128), ("int8", 64), ("int8", 256), ("k8v3", 128), ("k8v3", 256)])
@pytest.mark.parametrize("window", [None, 700])
@pytest.mark.parametrize("bs", [4, 32])
@pytest.mark.parametrize("splits", [0, 1])
def test_equal_splits_of_ragged_rows(kind, d, window, bs, splits):
    """The planned split of a batch of short and long rows with few queries:
    rows ending at, one below and one past a split's last key and tile, an
    empty prefix, and rows whose queries are fewer than the call's; and the
    same unsplit (at 4-token blocks more blocks than are looked up at a time)."""
    prefix, nq = [2600, 0, 511, 512, 513, 1023, 1024, 31, 33], 5
    lens = [5, 5, 1, 5, 0, 2, 5, 5, 3]
    lib = _lib.load()
    _lib.check(lib.s8kv_verify_set_splits(splits), "set_splits")
    try:
        _check(80 + d, kind, 8, 2, d, bs, prefix, nq, f"{kind} D={d} window={window}", query_lens=lens, window=window)
    finally:
        lib.s8kv_verify_set_splits(0)


@pytest.mark.parametrize("kind,d", [("int8", 64), ("int8", 128), ("k8v3", 128), ("int8", 256), ("k8v3", 256)])
@pytest.mark.parametrize("hq,nq", [(8, 8), (8, 9), (2, 32), (2, 33), (4, 1)])
def test_rows_around_one_wave(kind, d, hq, nq):
    """32 query rows a KV head (the narrow workgroups' most), one group more,
    and one query; trees and contexts from empty to a few tiles per wave."""
    _check(700 + d + nq, kind, hq, 2, d, 16, [0, 5, 128, 129, 300], nq, f"{kind} D={d} {hq}/2 heads x {nq}",
           query_lens=[nq, 1, nq, 0, nq], tree=True)


@pytest.mark.parametrize("kind,d", [("int8", 64), ("int8", 128), ("k8v3", 128), ("int8", 256), ("k8v3", 256)])
@pytest.mark.parametrize("bs,nq,tree", [(4, 40, False), (8, 64, True), (32, 64, True), (256, 33, False)])
@pytest.mark.parametrize("window", [None, 40])
def test_more_than_128_rows(kind, d, bs, nq, tree, window):
    """Rows enough for 8-wave workgroups (G 4, head_dim 128; else two blocks of 4): prefixes that start the drafts
    at every kind of place in a 32-key tile, one to three tiles in all, odd and
    even tile counts, more blocks than are looked up at a time (bs 4, 2,047
    keys and up), blocks smaller than a tile, and waves without a live row."""
    prefix = [0, 1, 31, 32, 33, 64, 95, 2047 + 5 * bs, 700]
    _check(300 + bs + nq, kind, 8, 2, d, bs, prefix, nq, f"{kind} D={d} bs={bs} nq={nq} tree={tree} window={window}",
           query_lens=[nq, nq, 1, nq - 1, nq, 9, nq, nq, 0], window=window, tree=tree)


@pytest.mark.parametrize("kind,d", [("int8", 64), ("int8", 128), ("k8v3", 128), ("int8", 256), ("k8v3", 256)])
@pytest.mark.parametrize("nq", [5, 20, 50])  # of 4 heads: one 32-row wave, a 128-row workgroup, more
@pytest.mark.parametrize("offset,pitch", [(1, 3), (4, 12), (8, 8)])
def test_q_rows_of_any_alignment(kind, d, nq, offset, pitch):
    """q as a view that starts `offset` elements into rows of d + `pitch`: the
    same bits as the aligned copy."""
    prefix = np.array([300, 150])
    case = make_case(95 + d, 2, 8, 2, d, 32, prefix + nq)
    cache = alloc(kind, case.num_blocks, 2, 32, d)
    append(kind, t(case.k), t(case.v), cache, t(case.slots))
    rows = t(np.random.default_rng(96).standard_normal((2, nq, 8, d + pitch)).astype(np.float16))
    view = rows[..., offset:offset + d].transpose(1, 2)
    fn = ops.attn_paged_verify if kind == "int8" else ops.attn_paged_verify_k8v3
    extra = () if kind == "int8" else (t(CODEBOOK),)
    outs = [fn(q, *cache, *extra, t(case.block_table), t(prefix.astype(np.int32)), 32,
               max_context_len=int(case.lens.max()), scale=case.scale) for q in (view, view.contiguous())]
    torch.cuda.synchronize()
    assert torch.isfinite(outs[0]).all() and torch.equal(*outs)


@pytest.mark.parametrize("kind,d", [("int8", 64), ("int8", 128), ("k8v3", 128), ("int8", 256), ("k8v3", 256)])
@pytest.mark.parametrize("nq", [5, 20, 50])  # of 4 heads: one 32-row wave, a 128-row workgroup, more
@pytest.mark.parametrize("bs", [16, 32, 64])
def test_block_id_past_the_pool_reads_zeros(kind, d, nq, bs):
    """The pool is the front of a larger allocation: a table entry naming the
    block after the pool's last gives the outputs of an all-zero block, not of
    what is stored there."""
    prefix = np.array([300, 150])
    case = make_case(90 + d, 2, 8, 2, d, bs, prefix + nq)
    n = case.num_blocks
    whole = alloc(kind, n + 3, 2, bs, d)
    append(kind, t(case.k), t(case.v), whole, t(case.slots))
    for x in whole:
        x[n:] = 3  # (past the pool below)
    spare = next(i for i in range(n) if i not in set(case.block_table.ravel()))
    cache = [x[:n] for x in whole]
    for x in cache:
        x[spare] = 0
    q = t(np.random.default_rng(91).standard_normal((2, 8, nq, d)).astype(np.float16))
    fn = ops.attn_paged_verify if kind == "int8" else ops.attn_paged_verify_k8v3
    extra = () if kind == "int8" else (t(CODEBOOK),)
    outs = []
    for block in (spare, n):
        table = case.block_table.copy()
        table[0, 1] = table[1, 0] = block
        out = fn(q, *cache, *extra, t(table), t(prefix.astype(np.int32)), bs,
                 max_context_len=int(case.lens.max()), scale=case.scale)
        torch.cuda.synchronize()
        outs.append(to_np(out))
    assert np.isfinite(outs[0]).all() and np.array_equal(*outs)


@pytest.mark.parametrize("kind,d", [("int8", 64), ("int8", 128), ("k8v3", 128), ("int8", 256), ("k8v3", 256)])
@pytest.mark.parametrize("nq", [5, 20, 50])  # of 4 heads: one 32-row wave, a 128-row workgroup, more
@pytest.mark.parametrize("given", ["none", "short"])
def test_call_without_its_workspace_runs_unsplit(kind, d, nq, given, monkeypatch):
    """No workspace, or one too small for any split: the bits of the unsplit
    call; and beyond 2^20 keys, where a split is a must, an error."""
    lib, inputs, asked = _lib.load(), ops._verify_inputs, []

    def withheld(*args, **kw):
        keep, head, tail, (ptr, size), geo, out = inputs(*args, **kw)
        asked.append(size)
        return keep, head, tail, (None, 0) if given == "none" else (ptr, min(size, 4096)), geo, out

    def run(max_ctx=None):
        out = fn(q, *cache, *extra, table, prefix, 64, max_context_len=max_ctx or int(case.lens.max()),
                 scale=case.scale)
        torch.cuda.synchronize()
        return out

    lens = np.array([9000, 33, 4100])
    case = make_case(98 + d, 3, 8, 2, d, 64, lens + nq, width=(1 << 20) // 64 + 1)
    cache = alloc(kind, case.num_blocks, 2, 64, d)
    append(kind, t(case.k), t(case.v), cache, t(case.slots))
    q = t(np.random.default_rng(99).standard_normal((3, 8, nq, d)).astype(np.float16))
    table, prefix = t(case.block_table), t(lens.astype(np.int32))
    fn = ops.attn_paged_verify if kind == "int8" else ops.attn_paged_verify_k8v3
    extra = () if kind == "int8" else (t(CODEBOOK),)
    split = run()
    lib.s8kv_verify_set_splits(1)
    try:
        whole = run()
    finally:
        lib.s8kv_verify_set_splits(0)
    monkeypatch.setattr(ops, "_verify_inputs", withheld)
    got = run()
    assert asked[0] > 0 and torch.equal(got, whole) and not torch.equal(split, whole)
    assert_close(to_np(got.float()), to_np(split.float()).astype(np.float64), f"{kind} D={d} unsplit")
    with pytest.raises(RuntimeError, match="workspace"):
        run((1 << 20) + 1)


def test_workspace_counts_the_split():
    """The workspace query plans the ragged batch's split too."""
    lib = _lib.load()
    assert lib.s8kv_verify_workspace_size(32, 32, 8, 128, 5, 8192) > 0
    assert lib.s8kv_verify_workspace_size(32, 32, 8, 128, 5, 500) == 0
