"""Performance cases of the paged KV-cache ops: what a serving engine asks of them.

A case is a dict of plain values.  ``prepare`` makes what the engine holds
before the call (the cache pool with its context, block tables, lengths, the
layer's q / k / v), ``run`` is one pass through the public ops, ``exact`` the
same outputs from plain torch in 64 bits, ``work`` the bytes and operations
that the pass cannot do without.

Kinds of pass:
  decode   one decode step of ``layers`` layers: append each row's token and
           attend (one launch per layer; ``planned``: after the step's slice
           plan; ``window`` > 0: append, then sliding-window attention)
  verify   append ``queries`` tokens per row and attend them over prefix and
           each other: chain (speculative drafts and prompt chunks are both
           causal chains) or tree
  prefill  causal attention of whole prompts over fresh fp16 K / V
  append   quantize-on-write of a prompt batch's K / V
  copy     block copies in every layer of a pool (copy-on-write)

Sizes that a case does not spell out (context lengths, trees, block ids) come
from its ``shape_seed``; values come from the seed given to ``prepare``.
"""

from __future__ import annotations

import math
import random

import torch

from superl8_serve_amd import ops

#: Lloyd-Max levels of N(0, 1) at 8 levels (Max 1960), the K8V3 codebook before its 1/sqrt(128).
LEVELS = (0.2451, 0.7560, 1.3439, 2.1520)
LLOYD_BLOCK = 128
OUTLIER_SCALE = 20.0  # 1 in 64 channels of K and V, as activations have them
DEV = "cuda"


def _decode(name, **kw):
    return {"name": name, "kind": "decode", "layout": "int8", "d": 128, "bs": 256, "layers": 1, "planned": False,
            "window": 0, **kw}


def _verify(name, **kw):
    return {"name": name, "kind": "verify", "layout": "int8", "d": 128, "bs": 256, "tree": False, "shared": False, **kw}


def listed():
    return [
        # one layer of a small model's decode step: a handful of users with short contexts
        _decode("decode_b8_short", batch=8, hq=16, hkv=8, lens="uniform", lo=128, hi=1024, shape_seed=1),
        # a single user deep in a long document
        _decode("decode_b1_long", batch=1, hq=32, hkv=8, lens="uniform", lo=30011, hi=30011, shape_seed=2),
        # the ordinary serving step: 64 users, contexts of a few thousand tokens, a plan shared by the layers
        _decode("decode_b64", batch=64, hq=32, hkv=8, lens="lognormal", lo=256, hi=8192, layers=4, planned=True,
                shape_seed=3),
        # long-context serving on the 3-bit V layout
        _decode("decode_k8v3_long", layout="k8v3", batch=32, hq=32, hkv=8, lens="uniform", lo=8192, hi=32768,
                planned=True, shape_seed=4),
        # a sliding-window layer with wide heads
        _decode("decode_window_d256", batch=32, hq=16, hkv=8, d=256, lens="uniform", lo=300, hi=8192, window=1024,
                shape_seed=5),
        # speculative decoding with a draft head: 4 drafts and the last token, checked as a chain
        _verify("chain_verify_b32", batch=32, hq=32, hkv=8, queries=5, lens="lognormal", lo=256, hi=8192,
                shape_seed=6),
        # speculative decoding with draft trees of 16 to 64 nodes
        _verify("tree_verify_b32", batch=32, hq=32, hkv=8, queries=64, tree=True, lens="uniform", lo=8192, hi=8192,
                shape_seed=7),
        # chunked prefill behind a shared system prompt
        _verify("chunk_b16", batch=16, hq=32, hkv=8, queries=512, shared=True, lens="uniform", lo=4096, hi=4096,
                shape_seed=8),
        # one long prompt's next chunk on a model with 256-wide heads, odd sizes
        _verify("chunk_b1_d256", batch=1, hq=16, hkv=4, d=256, queries=1999, lens="uniform", lo=6007, hi=6007,
                shape_seed=9),
        # a batch of ragged whole prompts
        {"name": "prefill_ragged", "kind": "prefill", "batch": 12, "hq": 32, "hkv": 8, "d": 128, "lens": "uniform",
         "lo": 200, "hi": 4000, "shape_seed": 10},
        # writing a prompt batch into the 3-bit V layout
        {"name": "append_k8v3", "kind": "append", "layout": "k8v3", "tokens": 24001, "hkv": 8, "d": 128, "bs": 256,
         "shape_seed": 11},
        # sequences leaving a shared prompt take private copies of its last block, in all layers
        {"name": "copy_on_write", "kind": "copy", "layout": "int8", "layers": 36, "pairs": 15, "blocks": 64, "hkv": 8,
         "d": 128, "bs": 256, "shape_seed": 12},
    ]


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        if w["bytes"] <= 2.5e9 and w["flops"] <= 4.8e11:  # no dearer than the listed chunk
            return case


def _log(rng, lo, hi):
    return min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def _draw(rng):
    kind = rng.choice(("decode", "decode", "verify", "verify", "verify", "prefill", "append", "copy"))
    layout = rng.choice(("int8", "int8", "k8v3"))
    heads = {"hkv": rng.choice((2, 4, 8))}
    d = rng.choice((128, 128, 128, 256, 64))
    if kind == "prefill":
        lo, hi = sorted((_log(rng, 16, 4096), _log(rng, 16, 4096)))
        return {"kind": kind, "batch": _log(rng, 1, 16), "hq": heads["hkv"] * rng.choice((1, 2, 4, 8)), **heads, "d": d,
                "lens": "uniform", "lo": lo, "hi": hi, "shape_seed": rng.randrange(1 << 30)}
    if layout == "k8v3" and d == 64:
        d = 128
    common = {"layout": layout, "d": d, "bs": rng.choice((16, 64, 256, 256)), **heads,
              "shape_seed": rng.randrange(1 << 30)}
    if kind == "append":
        return {"kind": kind, "tokens": _log(rng, 64, 32768), **common}
    if kind == "copy":
        return {"kind": kind, "layers": rng.randint(16, 48), "pairs": _log(rng, 1, 32), "blocks": 64, **common}
    hi = _log(rng, 160, 32768)
    rows = {"hq": heads["hkv"] * rng.choice((1, 2, 4, 4, 8)), "lens": rng.choice(("uniform", "lognormal")),
            "lo": max(1, hi // rng.choice((1, 2, 4, 16))), "hi": hi}
    if kind == "decode":
        window = rng.choice((0, 0, 0, 512, 4096))
        layers = 1 if window else rng.choice((1, 2))
        return {"kind": kind, "batch": _log(rng, 1, 64), "layers": layers, "planned": not window and rng.random() < 0.5,
                "window": window, **common, **rows}
    what = rng.choice(("chain", "chain", "tree", "chunk"))
    queries = {"chain": _log(rng, 2, 12), "tree": rng.randint(16, 64), "chunk": _log(rng, 64, 2048)}[what]
    return {"kind": kind, "batch": _log(rng, 1, 32), "queries": queries, "tree": what == "tree",
            "shared": what == "chunk" and rng.random() < 0.5, **common, **rows}


# ---------------------------------------------------------------------------
# Sizes of a case
# ---------------------------------------------------------------------------


def _shapes(case):
    """Context lengths (decode: with the new token; verify: the prefix), draft
    counts, ancestor masks and block tables of a case."""
    r = random.Random(case["shape_seed"])
    lo, hi, b = case["lo"], case["hi"], case["batch"]
    if case["lens"] == "lognormal":  # median a quarter of the longest
        lens = [min(hi, max(lo, int(round(math.exp(r.gauss(math.log(hi / 4), 0.75)))))) for _ in range(b)]
    else:
        lens = [r.randint(lo, hi) for _ in range(b)]
    s = {"lens": lens}
    if case["kind"] == "prefill":
        return s
    queries = case.get("queries", 0)
    counts = [queries] * b
    if case.get("tree"):
        counts = [r.randint(min(16, queries), queries) for _ in range(b)]
        s["masks"] = [_tree(r, n) for n in counts]
    s["counts"] = counts
    bs = case["bs"]
    shared = min(lens) // bs if case.get("shared") else 0  # whole blocks that every row starts with
    need = [-(-(n + queries) // bs) for n in lens]
    total = shared + sum(n - shared for n in need)
    ids = list(range(total + 3))
    r.shuffle(ids)
    table, at = [], shared
    for n in need:
        table.append(ids[:shared] + ids[at: at + n - shared])
        at += n - shared
    s.update(shared=shared, table=table, blocks=total + 3)
    return s


def _tree(r, n):
    """Ancestor bits of a random tree of n nodes, 1 to 4 children a node, in breadth-first order."""
    masks, frontier = [1], [0]
    while len(masks) < n:
        parent = frontier.pop(0)
        for _ in range(min(r.randint(1, 4), n - len(masks))):
            frontier.append(len(masks))
            masks.append(masks[parent] | 1 << len(masks))
    return masks


def _cell(case):
    """Cache bytes of one (token, KV head): int8 K and its scale, and V."""
    d = case["d"]
    return d + 4 + (d + 4 if case["layout"] == "int8" else 3 * d // 8 + 4 * (d // LLOYD_BLOCK))


def work(case):
    kind, d, hkv = case["kind"], case["d"], case["hkv"]
    if kind == "copy":
        return {"bytes": 2 * case["layers"] * case["pairs"] * hkv * case["bs"] * _cell(case), "flops": 0}
    if kind == "append":
        return {"bytes": case["tokens"] * (hkv * (4 * d + _cell(case)) + 4), "flops": 0}
    s, hq = _shapes(case), case["hq"]
    lens = s["lens"]
    if kind == "prefill":
        return {"bytes": sum(lens) * (2 * hq + 2 * hkv) * d * 2, "flops": sum(4 * d * hq * n * (n + 1) // 2 for n in lens)}
    if kind == "decode":
        seen = [min(n, case["window"] or n) for n in lens]
        layer = sum(seen) * hkv * _cell(case) + len(lens) * (4 * hq * d + hkv * (4 * d + _cell(case)))
        return {"bytes": case["layers"] * layer, "flops": case["layers"] * 4 * d * hq * sum(seen)}
    counts = s["counts"]
    if case["tree"]:
        pairs = sum(n * c + sum(bin(m).count("1") for m in ms) for n, c, ms in zip(lens, counts, s["masks"]))
    else:
        pairs = sum(n * c + c * (c + 1) // 2 for n, c in zip(lens, counts))
    held = sum(lens) - (len(lens) - 1) * s["shared"] * case["bs"]
    new = sum(counts)
    return {"bytes": (held + 2 * new) * hkv * _cell(case) + new * (4 * hkv * d + 4 * hq * d), "flops": 4 * d * hq * pairs}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


def _activations(gen, shape, outliers):
    x = torch.randn(shape, generator=gen, device=DEV)
    if outliers:
        ch = torch.randperm(shape[-1], generator=gen, device=DEV)[: max(1, shape[-1] // 64)]
        x[..., ch] *= OUTLIER_SCALE
    return x.half()


def _hadamard(d, dtype):
    h = torch.ones((1, 1), dtype=dtype, device=DEV)
    while h.shape[0] < d:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / math.sqrt(d)


def _rows_int8(x):
    """Symmetric int8 codes of each row and its scale, in x's precision."""
    scale = x.abs().amax(-1) / 127
    by = scale.float().to(x.dtype).clamp_min(1e-30)
    return (x / by.unsqueeze(-1)).round().clamp(-127, 127).to(torch.int8), scale


def _codebook():
    levels = [-v for v in reversed(LEVELS)] + list(LEVELS)
    return torch.tensor(levels, device=DEV) / math.sqrt(LLOYD_BLOCK)


def _rows_lloyd(x, codebook):
    """3-bit codes of each row's 128-value blocks and the blocks' norms, in x's precision."""
    blocks = x.reshape(*x.shape[:-1], -1, LLOYD_BLOCK)
    norm = blocks.square().sum(-1).sqrt()
    edges = ((codebook[1:] + codebook[:-1]) / 2).to(x.dtype)
    codes = torch.bucketize(blocks / norm.clamp_min(1e-30).unsqueeze(-1), edges)
    return codes.to(torch.uint8).reshape(x.shape), norm


def _pack(codes):
    """Bit-plane words: word 3 g + b holds bit b of codes 32 g .. 32 g + 31."""
    c = codes.reshape(*codes.shape[:-1], -1, 1, 32).long()
    bit = torch.arange(3, device=DEV).reshape(3, 1)
    words = ((c >> bit & 1) << torch.arange(32, device=DEV)).sum(-1)
    return torch.where(words >= 1 << 31, words - (1 << 32), words).int().flatten(-2)


def _pool(case, gen, layers, blocks):
    """A cache pool whose every row holds a quantized token."""
    hkv, d, bs = case["hkv"], case["d"], case["bs"]
    head = (layers, blocks, hkv, bs)
    pool = {"k_cache": torch.empty((*head, d), dtype=torch.int8, device=DEV),
            "k_scale": torch.empty(head, device=DEV)}
    if case["layout"] == "int8":
        pool |= {"v_cache": torch.empty_like(pool["k_cache"]), "v_scale": torch.empty(head, device=DEV)}
    else:
        pool |= {"v_packed": torch.empty((*head, 3 * d // 32), dtype=torch.int32, device=DEV),
                 "v_norm": torch.empty((*head, d // LLOYD_BLOCK), device=DEV)}
    had, book = _hadamard(d, torch.float32), _codebook()
    step = max(1, (1 << 25) // (hkv * bs * d))
    for layer in range(layers):
        for at in range(0, blocks, step):
            part = (layer, slice(at, min(blocks, at + step)))
            shape = tuple(pool["k_scale"][part].shape) + (d,)
            k = (_activations(gen, shape, True).float() @ had).half().float()
            pool["k_cache"][part], pool["k_scale"][part] = _rows_int8(k)
            v = _activations(gen, shape, True).float()
            if case["layout"] == "int8":
                pool["v_cache"][part], pool["v_scale"][part] = _rows_int8(v)
            else:
                codes, pool["v_norm"][part] = _rows_lloyd(v, book)
                pool["v_packed"][part] = _pack(codes)
    return pool


def _int32(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


def _slots(case, s, row, first, count):
    """Flat cache slots of `count` tokens of a row from position `first` on."""
    bs, blocks = case["bs"], s["table"][row]
    return [blocks[p // bs] * bs + p % bs for p in range(first, first + count)]


def prepare(case, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    kind, d, hkv = case["kind"], case["d"], case["hkv"]
    st = {"case": case}
    if kind == "copy":
        st["pool"] = _pool(case, gen, case["layers"], case["blocks"])
        ids = random.Random(case["shape_seed"]).sample(range(case["blocks"]), 2 * case["pairs"])
        st["src"], st["dst"] = ids[::2], ids[1::2]
        return st
    if kind == "append":
        blocks = -(-case["tokens"] // case["bs"]) + 3
        st["pool"] = _pool(case, gen, 1, blocks)
        order = random.Random(case["shape_seed"]).sample(range(blocks), blocks)
        st["slots"] = _int32([order[t // case["bs"]] * case["bs"] + t % case["bs"] for t in range(case["tokens"])])
        st["k"] = _activations(gen, (case["tokens"], hkv, d), True)
        st["v"] = _activations(gen, (case["tokens"], hkv, d), True)
        st["codebook"] = _codebook()
        return st
    s, hq, b = _shapes(case), case["hq"], case["batch"]
    lens = s["lens"]
    st["scale"] = 1.0 / math.sqrt(d)
    if kind == "prefill":
        ends = [0]
        for n in lens:
            ends.append(ends[-1] + n)
        st["cu"] = _int32(ends)
        st["longest"] = max(lens)
        st["q"] = _activations(gen, (ends[-1], hq, d), False)
        st["k"] = _activations(gen, (ends[-1], hkv, d), False)
        st["v"] = _activations(gen, (ends[-1], hkv, d), True)
        return st
    st["codebook"] = _codebook()
    layers = case.get("layers", 1)
    st["pool"] = _pool(case, gen, layers, s["blocks"])
    width = max(len(t) for t in s["table"])
    st["table"] = _int32([t + [0] * (width - len(t)) for t in s["table"]])
    longest = max(lens) + case.get("queries", 0)
    st["max_context_len"] = min(width * case["bs"], -(-longest // 128) * 128)
    if kind == "decode":
        st["lens"] = _int32(lens)
        # as a layer has them: [B, 1, H, D], the queries seen as [B, H, 1, D]
        st["q"] = [_activations(gen, (b, 1, hq, d), False).transpose(1, 2) for _ in range(layers)]
        st["k"] = [_activations(gen, (b, hkv, d), True) for _ in range(layers)]
        st["v"] = [_activations(gen, (b, hkv, d), True) for _ in range(layers)]
        st["slots"] = _int32([_slots(case, s, i, n - 1, 1)[0] for i, n in enumerate(lens)])
        return st
    queries = case["queries"]
    st["prefix"] = _int32(lens)
    st["q"] = _activations(gen, (b, queries, hq, d), False).transpose(1, 2)
    st["k"] = _activations(gen, (b * queries, hkv, d), True)
    st["v"] = _activations(gen, (b * queries, hkv, d), True)
    slots = [_slots(case, s, i, n, c) + [-1] * (queries - c) for i, (n, c) in enumerate(zip(lens, s["counts"]))]
    st["slots"] = _int32([x for row in slots for x in row])
    if case["tree"]:
        st["counts"] = _int32(s["counts"])
        masks = [m + [0] * (queries - len(m)) for m in s["masks"]]
        st["masks"] = torch.tensor([[x - (1 << 64) if x >> 63 else x for x in m] for m in masks], device=DEV)
    return st


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------


def _write(st, pool, k, v):
    if "v_cache" in pool:
        ops.quantize_kv_write_paged(k, v, pool["k_cache"], pool["k_scale"], pool["v_cache"], pool["v_scale"], st["slots"])
    else:
        ops.quantize_kv_write_paged_k8v3(k, v, pool["k_cache"], pool["k_scale"], pool["v_packed"], pool["v_norm"],
                                         st["codebook"], st["slots"])


def _cache_args(st, pool):
    if "v_cache" in pool:
        return pool["k_cache"], pool["k_scale"], pool["v_cache"], pool["v_scale"]
    return pool["k_cache"], pool["k_scale"], pool["v_packed"], pool["v_norm"], st["codebook"]


def _run_decode(st):
    case, pool = st["case"], st["pool"]
    bs, int8 = case["bs"], case["layout"] == "int8"
    how = {"max_context_len": st["max_context_len"], "scale": st["scale"]}
    outs = []
    if case["planned"]:
        how["plan"] = ops.attn_paged_decode_plan(pool["k_cache"][0], st["table"], st["lens"], bs, num_q_heads=case["hq"],
                                                 max_context_len=st["max_context_len"], layout=case["layout"])
    for layer in range(case["layers"]):
        view = {n: t[layer] for n, t in pool.items()}
        q, k, v = st["q"][layer], st["k"][layer], st["v"][layer]
        if case["window"]:
            _write(st, view, k, v)
            op = ops.attn_paged_decode_window if int8 else ops.attn_paged_decode_window_k8v3
            outs.append(op(q, *_cache_args(st, view), st["table"], st["lens"], bs, window=case["window"], **how))
        else:
            op = ops.attn_paged_decode_append if int8 else ops.attn_paged_decode_append_k8v3
            outs.append(op(q, k, v, *_cache_args(st, view), st["table"], st["lens"], bs, **how))
    return {"out": outs, **pool}


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "decode":
        return _run_decode(st)
    if kind == "prefill":
        return ops.attn_varlen(st["q"], st["k"], st["v"], st["cu"], st["cu"], st["longest"], st["longest"], causal=True,
                               scale=st["scale"])
    pool = st["pool"]
    if kind == "copy":
        ops.copy_blocks(list(pool.values()), st["src"], st["dst"])
        return pool
    view = {n: t[0] for n, t in pool.items()}
    _write(st, view, st["k"], st["v"])
    if kind == "append":
        return pool
    op = ops.attn_paged_verify if case["layout"] == "int8" else ops.attn_paged_verify_k8v3
    out = op(st["q"], *_cache_args(st, view), st["table"], st["prefix"], case["bs"], query_lens=st.get("counts"),
             tree_mask=st.get("masks"), max_context_len=st["max_context_len"], scale=st["scale"])
    return {"out": out, **pool}


def tolerance(case):
    """Attention outputs are fp16 (rounding alone: 2e-4 of the result's norm);
    cache bytes and copies are the same to the bit, new scales and norms 32-bit sums."""
    if case["kind"] == "copy":
        return "exact"
    if case["kind"] == "append":
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}
    return {"rel": 8e-4, "max": 8e-3, "differ": 0.0}


# ---------------------------------------------------------------------------
# The same outputs in 64 bits
# ---------------------------------------------------------------------------


def _exact_write(case, st, layer, k, v):
    """The layer's cache as 64-bit (K codes, K scales, V values, V scales or norms) with the new tokens in it."""
    pool, d, hkv, bs = st["pool"], case["d"], case["hkv"], case["bs"]
    live = st["slots"] >= 0
    slots = st["slots"][live].long()
    blk, off = slots // bs, slots % bs
    kc, ks = pool["k_cache"][layer].clone(), pool["k_scale"][layer].double()
    rotated = (k.double() @ _hadamard(d, torch.float64)).half().double()
    kc[blk, :, off], ks[blk, :, off] = (x[live] for x in _rows_int8(rotated))
    if case["layout"] == "int8":
        vc, vs = pool["v_cache"][layer].clone(), pool["v_scale"][layer].double()
        vc[blk, :, off], vs[blk, :, off] = (x[live] for x in _rows_int8(v.double()))
    else:
        words = pool["v_packed"][layer].reshape(-1, hkv, bs, d // 32, 3, 1)
        bits = words >> torch.arange(32, device=DEV, dtype=torch.int32) & 1
        vc = (bits[..., 0, :] + 2 * bits[..., 1, :] + 4 * bits[..., 2, :]).to(torch.uint8).flatten(-2)
        vs = pool["v_norm"][layer].double()
        vc[blk, :, off], vs[blk, :, off] = (x[live] for x in _rows_lloyd(v.double(), st["codebook"]))
    return kc, ks, vc, vs


def _exact_row(case, st, cache, blocks, first, n):
    """Rotated K and V in 64 bits of positions first .. n - 1 of one row, [Hkv, n - first, D] each."""
    kc, ks, vc, vs = cache
    blk = torch.tensor(blocks, device=DEV)

    def tokens(x):
        return x[blk].transpose(0, 1).flatten(1, 2)[:, first:n]

    k = tokens(kc).double() * tokens(ks).unsqueeze(-1)
    if case["layout"] == "int8":
        return k, tokens(vc).double() * tokens(vs).unsqueeze(-1)
    v = st["codebook"].double()[tokens(vc).long()]
    return k, (v.reshape(*v.shape[:-1], -1, LLOYD_BLOCK) * tokens(vs).unsqueeze(-1)).reshape(v.shape)


def _exact_attend(q, k, v, seen, scale):
    """q [Hq, S, D] over k, v [Hkv, n, D]; seen [S, n] or None: which keys each query sees."""
    hkv, g = k.shape[0], q.shape[0] // k.shape[0]
    out = torch.empty_like(q)
    for h in range(hkv):
        kt = k[h].T.contiguous()
        for i in range(g):
            y = q[h * g + i] @ kt * scale
            if seen is not None:
                y.masked_fill_(~seen, -math.inf)
            out[h * g + i] = torch.softmax(y, -1) @ v[h]
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "copy":
        return None
    st = prepare(case, seed)
    d = case["d"]
    if kind == "prefill":
        out = torch.empty(st["q"].shape, dtype=torch.float64, device=DEV)
        at = 0
        for n in _shapes(case)["lens"]:
            part = [st[x][at: at + n].transpose(0, 1).double() for x in ("q", "k", "v")]
            seen = torch.ones((n, n), dtype=torch.bool, device=DEV).tril()
            out[at: at + n] = _exact_attend(*part, seen, st["scale"]).transpose(0, 1)
            at += n
        return out
    scale_names = ("k_scale", "v_scale" if case["layout"] == "int8" else "v_norm")
    answer = dict.fromkeys(st["pool"])
    if kind == "append":
        cache = _exact_write(case, st, 0, st["k"], st["v"])
        return {**answer, scale_names[0]: cache[1][None], scale_names[1]: cache[3][None]}
    s, had = _shapes(case), _hadamard(d, torch.float64)
    layers = case.get("layers", 1)
    scales = [torch.empty(st["pool"][n].shape, dtype=torch.float64, device=DEV) for n in scale_names]
    outs = []
    for layer in range(layers):
        k, v, q = ((x[layer] if kind == "decode" else x) for x in (st["k"], st["v"], st["q"]))
        cache = _exact_write(case, st, layer, k, v)
        scales[0][layer], scales[1][layer] = cache[1], cache[3]
        qr = q.double() @ had
        out = torch.zeros(q.shape, dtype=torch.float64, device=DEV)
        for i, n in enumerate(s["lens"]):
            if kind == "decode":
                first = max(0, n - (case["window"] or n))
                part = _exact_row(case, st, cache, s["table"][i], first, n)
                out[i] = _exact_attend(qr[i], *part, None, st["scale"])
                continue
            c = s["counts"][i]
            part = _exact_row(case, st, cache, s["table"][i], 0, n + c)
            seen = torch.ones((c, n + c), dtype=torch.bool, device=DEV)
            if case["tree"]:
                rows = [[m >> j & 1 for j in range(c)] for m in s["masks"][i]]
                seen[:, n:] = torch.tensor(rows, dtype=torch.bool, device=DEV)
            else:
                seen[:, n:] = seen[:, n:].tril()
            out[i, :, :c] = _exact_attend(qr[i, :, :c], *part, seen, st["scale"])
        outs.append(out)
    return {**answer, "out": outs if kind == "decode" else outs[0], scale_names[0]: scales[0], scale_names[1]: scales[1]}
