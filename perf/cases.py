"""Performance cases of the attention library: what its users call, with their sizes.

Every case goes through the public Python front end (tmac_gguf.cpp_amd/tmac_attn.py, which
forwards to the C ABI).  The shapes are those of the benchmark configurations and the
tests: 14 query heads over 2 kv heads of 64 dims, 24 layers, 896-wide hidden state, and the
other head shapes the entry points take.  A case's `lens` number fixes its sequence lengths
(so its work is known without a seed); every value comes from the seed.

Kinds:
  ops     one layer of a batch-1 decode step as the engine's per-op loop issues it, eagerly:
          QKV projection with biases, RoPE of q and k, the two cache-row writes, attention,
          output projection (7 calls; latency and launches are what counts)
  step    a captured 24-layer decode step: position counter, then one fused layer call
          (RoPE + cache write + attention) per layer; with `proj` also the QKV projection
          before it and the output projection with the residual add behind it
  decode  one query token for each of n_seq sequences of equal length
  ragged  the same over a packed pool of sequences of different lengths
  paged   the same over 16-row pages in random order
  serve   the batched layer step of a serving loop over paged caches
  prefill a chunk of n_q prompt tokens per sequence after prefix rows (contiguous cache)
  prompt  the same over a paged cache
  any     batched decode at a head shape without kernels of its own
  gemv    one quantized weight matrix times a vector (output head, FFN down projection)
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "tmac_gguf.cpp_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import tmac_attn as tm  # noqa: E402

LAYERS, NH, NKV, HD = 24, 14, 2, 64
QD, KVD, G = NH * HD, NKV * HD, NH // NKV
BASE = 1e6
KV_DTYPE = {"f32": tm.TMAC_KV_F32, "bf16": tm.TMAC_KV_BF16, "f16": tm.TMAC_KV_F16, "q8": tm.TMAC_KV_Q8_0}
HEAD_BYTES = {"f32": 256, "bf16": 128, "f16": 128, "q8": 68}  # one (row, kv head) of 64 dims
QTYPE = {"q5_0": tm.TMAC_Q5_0, "q8_0": tm.TMAC_Q8_0, "q4_k": tm.TMAC_Q4_K, "q6_k": tm.TMAC_Q6_K}
QBLOCK = {"q5_0": (32, 22), "q8_0": (32, 34), "q4_k": (256, 144), "q6_k": (256, 210)}  # weights, bytes
ANY_SHAPES = [(14, 2, 128), (16, 2, 128), (12, 4, 96), (8, 8, 80), (14, 2, 32), (6, 3, 64), (5, 5, 256)]


def listed():
    return [
        # one token of an interactive session: the engine's own loop, one layer, op by op
        {"name": "ops_255", "kind": "ops", "past_len": 255},
        # one token of an interactive session: the whole 24-layer attention block as one graph
        {"name": "step_24x200_proj", "kind": "step", "pos": 200, "cap": 256, "proj": True},
        # offline batch decode at the benchmark's headline size (the largest case)
        {"name": "decode_f32_256x4096", "kind": "decode", "cache": "f32", "n_seq": 256, "n_pos": 4096},
        # the same batch with the quantized cache
        {"name": "decode_q8_256x4096", "kind": "decode", "cache": "q8", "n_seq": 256, "n_pos": 4096},
        # a few long documents of different lengths
        {"name": "ragged_f32_16x32768", "kind": "ragged", "cache": "f32", "n_seq": 16, "max_len": 32768, "lens": 4},
        # a serving batch on paged 16-bit caches, an odd number of sequences
        {"name": "paged_bf16_193x4096", "kind": "paged", "cache": "bf16", "n_seq": 193, "max_len": 4096, "lens": 7},
        # a serving loop's layer step, long contexts, paged fp32 caches
        {"name": "serve_f32_64x16384", "kind": "serve", "cache": "f32", "n_seq": 64, "max_len": 16384, "lens": 5},
        # chunked prefill of several prompts at the benchmark's size
        {"name": "prefill_f32_4x512_1536", "kind": "prefill", "cache": "f32", "n_seq": 4, "n_q": 512, "prefix": 1536},
        # one long prompt from its first token, odd length, paged 16-bit cache
        {"name": "prompt_bf16_1x2999", "kind": "prompt", "cache": "bf16", "n_seq": 1, "n_q": 2999, "prefix": 0},
        # the next turn of a conversation: a short chunk after a long cached prefix
        {"name": "prompt_q8_1x100_4000", "kind": "prompt", "cache": "q8", "n_seq": 1, "n_q": 100, "prefix": 4000},
        # a model with 128-wide heads: no kernels of its own, the any-shape path
        {"name": "any_14_2_128_32x2048", "kind": "any", "nh": 14, "nkv": 2, "hd": 128, "n_seq": 32, "n_pos": 2048},
        # the output head of one decode step
        {"name": "gemv_q8_0_151936x896", "kind": "gemv", "qtype": "q8_0", "rows": 151936, "cols": 896},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges, no larger than the largest listed case of its resource."""
    while True:
        kind = rng.choice(["ops", "step", "decode", "decode", "ragged", "ragged", "paged", "paged", "serve", "prefill",
                           "prompt", "prompt", "any", "gemv"])
        c = {"kind": kind}
        if kind == "ops":
            c["past_len"] = _log(rng, 1, 1024) - 1
        elif kind == "step":
            cap = _log(rng, 64, 4096)
            c.update(pos=rng.randrange(cap), cap=cap, proj=rng.random() < 0.5)
        elif kind == "decode":
            c.update(cache=rng.choice(["f32", "bf16", "f16", "q8"]), n_seq=_log(rng, 1, 300), n_pos=_log(rng, 16, 32768))
        elif kind in ("ragged", "paged", "serve"):
            c.update(cache=rng.choice(["f32", "bf16", "f16", "q8"]), n_seq=_log(rng, 1, 4096),
                     max_len=_log(rng, 40, 32768), lens=rng.randrange(1 << 30))
        elif kind in ("prefill", "prompt"):
            c.update(cache=rng.choice(["f32", "bf16", "f16", "q8"]), n_seq=_log(rng, 1, 8), n_q=_log(rng, 5, 3000),
                     prefix=rng.choice([0, _log(rng, 1, 8000)]))
        elif kind == "any":
            nh, nkv, hd = rng.choice(ANY_SHAPES)
            c.update(nh=nh, nkv=nkv, hd=hd, n_seq=_log(rng, 1, 64), n_pos=_log(rng, 16, 4096))
        else:
            qt = rng.choice(sorted(QTYPE))
            n = QBLOCK[qt][0]
            c.update(qtype=qt, rows=_log(rng, 64, 151936), cols=n * _log(rng, 256 // n, 4864 // n))
        w = work(c)
        rows = c["n_seq"] * c["max_len"] if "max_len" in c else 0
        if w["bytes"] <= (150e6 if kind in ("any", "gemv") else 1e9) and w["flops"] <= 16.2e9 and rows <= 1 << 21:
            return c


# ---------------------------------------------------------------- sizes

def _lens(case):
    """Sequence lengths of a ragged / paged case, uniform in 1..max_len, fixed by its `lens` number."""
    r = np.random.default_rng(case["lens"])
    return r.integers(1, case["max_len"] + 1, case["n_seq"]).astype(np.int32)


def _gemv_bytes(qt, rows, cols):
    n, b = QBLOCK[qt]
    return rows * (cols // n) * b


def work(case):
    """Bytes (each input once, each output once) and operations of one pass."""
    k = case["kind"]
    if k in ("ops", "step"):
        layers, rows = (1, case["past_len"] + 1) if k == "ops" else (LAYERS, case["pos"] + 1)
        proj = k == "ops" or case["proj"]
        b = rows * 4 * KVD * 2 + 4 * (2 * QD + 2 * KVD)
        f = 4 * HD * NH * rows
        if proj:
            b += _gemv_bytes("q5_0", 2 * QD + KVD, QD) + _gemv_bytes("q8_0", KVD, QD) + 4 * (3 * QD + 2 * KVD)
            f += 2 * QD * (2 * QD + 2 * KVD)
        return {"bytes": layers * b, "flops": layers * f}
    if k == "gemv":
        return {"bytes": _gemv_bytes(case["qtype"], case["rows"], case["cols"]) + 4 * (case["rows"] + case["cols"]),
                "flops": 2 * case["rows"] * case["cols"]}
    if k == "any":
        rows = case["n_seq"] * case["n_pos"]
        return {"bytes": rows * case["nkv"] * case["hd"] * 8 + 8 * case["n_seq"] * case["nh"] * case["hd"],
                "flops": 4 * case["hd"] * case["nh"] * rows}
    row = 2 * NKV * HEAD_BYTES[case["cache"]]
    if k in ("prefill", "prompt"):
        n, p = case["n_q"], case["prefix"]
        pairs = case["n_seq"] * (n * p + n * (n + 1) // 2)
        return {"bytes": case["n_seq"] * ((n + p) * row + n * QD * 8), "flops": 4 * HD * NH * pairs}
    rows = case["n_seq"] * case["n_pos"] if k == "decode" else int(_lens(case).sum())
    new = case["n_seq"] * (row + 8 * KVD) if k == "serve" else 0
    return {"bytes": rows * row + case["n_seq"] * QD * 8 + new, "flops": 4 * HD * NH * rows}


# ---------------------------------------------------------------- inputs

_shared = {}


def _ctx():
    """The program's one context, and the one stream all its calls go to."""
    if not _shared:
        _shared["ctx"] = tm.Context(0)
        _shared["stream"] = torch.cuda.Stream()
        try:  # the context looks kernels up in several modules and leaves the misses as the runtime's last error,
            torch.zeros(1, device="cuda")  # which torch's next launch reports once
        except RuntimeError:
            pass
    return _shared["ctx"], _shared["stream"].cuda_stream


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _cache(g, rows, name, nkv=NKV, hd=HD):
    """`rows` cache rows of N(0, 1) keys or values in the cache's own layout."""
    x = _randn(g, rows, nkv * hd)
    if name == "f32":
        return x
    if name in ("bf16", "f16"):
        return x.to(torch.bfloat16 if name == "bf16" else torch.float16)
    out = torch.empty(rows * nkv, 68, device="cuda", dtype=torch.uint8)
    step = 1 << 20
    x = x.view(rows * nkv, 2, 32)
    for i in range(0, rows * nkv, step):  # head rows: int8 q[64], fp16 d0, d1 (value = q * d)
        y = x[i:i + step]
        d = (y.abs().amax(-1, keepdim=True) / 127).to(torch.float16)
        q = torch.round(y / d.float()).clamp(-127, 127).to(torch.int8)
        out[i:i + step, :64] = q.reshape(-1, 64).view(torch.uint8)
        out[i:i + step, 64:] = d.reshape(-1, 2).contiguous().view(torch.uint8)
    return out


def _values(cache, name, nkv=NKV, hd=HD):
    """The values a cache holds, exactly: float64 [rows][nkv][hd]."""
    if name != "q8":
        return cache.double().view(-1, nkv, hd)
    q = cache[:, :64].contiguous().view(torch.int8).double().view(-1, 2, 32)
    d = cache[:, 64:].contiguous().view(torch.float16).double().view(-1, 2, 1)
    return (q * d).view(-1, nkv, hd)


def _weights(g, qt, rows, cols, layers=1):
    """Random quantized blocks with scales as trained weights have them."""
    n, b = QBLOCK[qt]
    nb = layers * rows * (cols // n)
    w = torch.randint(0, 256, (nb, b), generator=g, device="cuda", dtype=torch.uint8)
    at = {"q5_0": [0], "q8_0": [0], "q4_k": [0, 2], "q6_k": [208]}[qt]
    for a in at:
        hi = {"q5_0": 4e-3, "q8_0": 5e-4, "q4_k": 2e-4, "q6_k": 2e-5}[qt]
        d = (torch.rand(nb, 1, generator=g, device="cuda") * (hi * 0.875) + hi * 0.125).to(torch.float16)
        w[:, a:a + 2] = d.view(torch.uint8)
    return w


class _State:
    """What the program holds: its tensors by name, the case, and a captured graph where there is one."""

    def __init__(self, case, **tensors):
        self.case, self.graph = case, None
        self.__dict__.update(tensors)

    def __del__(self):
        if self.graph is not None:
            ctx, _ = _ctx()
            ctx.graph_destroy(self.graph)


def _pages(g, case, lens):
    """Block table over a pool that holds just these sequences, its pages in random order."""
    need = (lens.astype(np.int64) + 15) // 16
    max_pages = int((case.get("max_len", int(lens.max())) + 15) // 16)
    total = int(need.sum())
    perm = torch.randperm(total, generator=g, device="cuda").to(torch.int32)
    table = torch.zeros(len(lens), max_pages, device="cuda", dtype=torch.int32)
    n = torch.from_numpy(need).cuda()
    table[torch.arange(max_pages, device="cuda")[None, :] < n[:, None]] = perm
    return table, max_pages, total


def prepare(case, seed):
    g = _gen(seed)
    k = case["kind"]
    ctx, stream = _ctx()
    if k in ("ops", "step"):
        layers, cap = (1, case["past_len"] + 1) if k == "ops" else (LAYERS, case["cap"])
        ctx.rope_prepare(HD, BASE, cap)
        s = _State(case, kc=_randn(g, layers, cap, KVD), vc=_randn(g, layers, cap, KVD),
                   x=_randn(g, layers, QD), q=_randn(g, layers, QD), kn=_randn(g, layers, KVD),
                   vn=_randn(g, layers, KVD), out=torch.empty(layers, QD, device="cuda"))
        if k == "ops" or case["proj"]:
            s.wq, s.wk = _weights(g, "q5_0", QD, QD, layers), _weights(g, "q5_0", KVD, QD, layers)
            s.wv, s.wo = _weights(g, "q8_0", KVD, QD, layers), _weights(g, "q5_0", QD, QD, layers)
            s.bq, s.bk, s.bv = (0.1 * _randn(g, layers, n) for n in (QD, KVD, KVD))
            s.h0 = _randn(g, QD)
            s.h = torch.empty(QD, device="cuda")
        if k == "step":
            s.pos = torch.full((1,), case["pos"], device="cuda", dtype=torch.int32)
            torch.cuda.synchronize()
            _step(ctx, stream, s)  # once eagerly, as the library asks before a capture
            ctx.step_begin(stream)
            _step(ctx, stream, s)
            s.graph = ctx.step_end(stream)
    elif k == "gemv":
        s = _State(case, w=_weights(g, case["qtype"], case["rows"], case["cols"]), x=_randn(g, case["cols"]),
                   y=torch.empty(case["rows"], device="cuda"))
    elif k == "any":
        nh, nkv, hd, n = case["nh"], case["nkv"], case["hd"], case["n_seq"]
        s = _State(case, q=_randn(g, n, nh * hd), k=_randn(g, n * case["n_pos"], nkv * hd),
                   v=_randn(g, n * case["n_pos"], nkv * hd), out=torch.empty(n, nh * hd, device="cuda"))
    elif k in ("prefill", "prompt"):
        n, rows = case["n_seq"], case["prefix"] + case["n_q"]
        s = _State(case, q=_randn(g, n, case["n_q"], QD), out=torch.empty(n, case["n_q"], QD, device="cuda"))
        total = n * rows
        if k == "prompt":
            s.table, s.max_pages, s.n_pages = _pages(g, case, np.full(n, rows, np.int32))
            total = s.n_pages * 16
        s.k, s.v = _cache(g, total, case["cache"]), _cache(g, total, case["cache"])
    else:  # decode, ragged, paged, serve
        n = case["n_seq"]
        s = _State(case, q=_randn(g, n, QD), out=torch.empty(n, QD, device="cuda"))
        if k == "decode":
            total = n * case["n_pos"]
        else:
            lens = _lens(case)
            total = int(lens.sum())
            s.total = total
            s.lens = torch.from_numpy(lens).cuda()
            if k == "ragged":
                s.offs = torch.from_numpy(np.concatenate([[0], np.cumsum(lens[:-1], dtype=np.int64)])).cuda()
            else:
                s.table, s.max_pages, s.n_pages = _pages(g, case, lens)
                total = s.n_pages * 16
        s.k, s.v = _cache(g, total, case["cache"]), _cache(g, total, case["cache"])
        if k == "serve":
            ctx.rope_prepare(HD, BASE, case["max_len"])
            s.pos = s.lens - 1
            s.kn, s.vn = _randn(g, n, KVD), _randn(g, n, KVD)
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------- one pass

def _layer(t, i):
    return t.data_ptr() + i * (t[0].numel() * t.element_size())


def _per_layer(w, i):
    return w.data_ptr() + i * (w.numel() // LAYERS)


def _step(ctx, stream, s):
    c = s.case
    proj = c["proj"]
    p = lambda t: t.data_ptr()  # noqa: E731
    ctx.pos_update(p(s.pos), c["pos"], stream=stream)
    if proj:
        ctx.elem_op(2, p(s.h), p(s.h0), QD, stream=stream)  # the token's embedding into the hidden state
    for i in range(LAYERS):
        q, kn, vn, out = (_layer(t, i) for t in (s.q, s.kn, s.vn, s.out))
        if proj:
            ctx.fused_qkv(_per_layer(s.wq, i), _per_layer(s.wk, i), _per_layer(s.wv, i), _layer(s.x, i), q, kn, vn,
                          QD, KVD, KVD, QD, True, b_q=_layer(s.bq, i), b_k=_layer(s.bk, i), b_v=_layer(s.bv, i),
                          stream=stream)
        ctx.layer_attention_devpos(q, kn, vn, _layer(s.kc, i), _layer(s.vc, i), out, NH, NKV, HD, p(s.pos), c["cap"],
                                   BASE, stream=stream)
        if proj:
            ctx.matmul(tm.TMAC_Q5_0, QD, QD, _per_layer(s.wo, i), out, p(s.h), accumulate=True, stream=stream)


def run(s):
    c = s.case
    k = c["kind"]
    ctx, stream = _ctx()
    p = lambda t: t.data_ptr()  # noqa: E731
    if k == "step":
        ctx.graph_launch(s.graph, stream)
        return {"out": s.out, "k": s.kc, "v": s.vc, **({"h": s.h, "q": s.q} if c["proj"] else {})}
    if k == "ops":
        pos = c["past_len"]
        row = 4 * pos * KVD
        ctx.fused_qkv(p(s.wq), p(s.wk), p(s.wv), p(s.x), p(s.q), p(s.kn), p(s.vn), QD, KVD, KVD, QD, True, b_q=p(s.bq),
                      b_k=p(s.bk), b_v=p(s.bv), stream=stream)
        ctx.rope_op(p(s.q), NH, HD, pos, BASE, stream=stream)
        ctx.rope_op(p(s.kn), NKV, HD, pos, BASE, stream=stream)
        ctx.elem_op(2, p(s.kc) + row, p(s.kn), KVD, stream=stream)
        ctx.elem_op(2, p(s.vc) + row, p(s.vn), KVD, stream=stream)
        ctx.attention_op(p(s.q), p(s.kc), p(s.vc), p(s.out), NH, NKV, HD, pos, stream=stream)
        ctx.matmul(tm.TMAC_Q5_0, QD, QD, p(s.wo), p(s.out), p(s.h), stream=stream)
        return {"out": s.out, "h": s.h, "k": s.kc, "v": s.vc}
    if k == "gemv":
        ctx.matmul(QTYPE[c["qtype"]], c["rows"], c["cols"], p(s.w), p(s.x), p(s.y), stream=stream)
        return s.y
    if k == "any":
        ctx.decode_batched(p(s.q), p(s.k), p(s.v), p(s.out), c["n_seq"], c["nh"], c["nkv"], c["hd"], c["n_pos"],
                           c["n_pos"], stream=stream)
        return s.out
    dt = KV_DTYPE[c["cache"]]
    if k == "prefill":
        ctx.prefill(p(s.q), p(s.k), p(s.v), p(s.out), c["n_seq"], c["n_q"], c["prefix"], c["prefix"] + c["n_q"], NH, NKV,
                    HD, stream=stream, kv_dtype=dt)
    elif k == "prompt":
        ctx.prefill_paged(p(s.q), p(s.k), p(s.v), s.n_pages, p(s.table), s.max_pages, p(s.out), c["n_seq"], c["n_q"],
                          c["prefix"], NH, NKV, HD, stream=stream, kv_dtype=dt)
    elif k == "decode":
        ctx.decode_batched(p(s.q), p(s.k), p(s.v), p(s.out), c["n_seq"], NH, NKV, HD, c["n_pos"], c["n_pos"],
                           stream=stream, kv_dtype=dt)
    elif k == "ragged":
        ctx.decode_ragged(p(s.q), p(s.k), p(s.v), p(s.offs), p(s.lens), p(s.out), c["n_seq"], NH, NKV, HD, c["max_len"],
                          total_rows=s.total, stream=stream, kv_dtype=dt)
    elif k == "paged":
        ctx.decode_paged(p(s.q), p(s.k), p(s.v), s.n_pages, p(s.table), s.max_pages, p(s.lens), p(s.out), c["n_seq"], NH,
                         NKV, HD, c["max_len"], total_rows=s.total, stream=stream, kv_dtype=dt)
    else:
        ctx.layer_attention_paged(p(s.q), p(s.kn), p(s.vn), p(s.k), p(s.v), s.n_pages, p(s.table), s.max_pages, p(s.pos),
                                  p(s.out), c["n_seq"], NH, NKV, HD, c["max_len"], BASE, stream=stream, kv_dtype=dt)
        return {"out": s.out, "k": s.k, "v": s.v}
    return s.out


# ---------------------------------------------------------------- the same in 64 bits

def _dequant(w, qt, rows, cols):
    """float64 [rows][cols] of quantized blocks (GGML Q5_0, Q8_0, Q4_K, Q6_K)."""
    half = lambda a: w[:, a:a + 2].contiguous().view(torch.float16).double()  # noqa: E731
    byte = lambda a, b: w[:, a:b].to(torch.int64)  # noqa: E731
    if qt == "q8_0":
        v = w[:, 2:34].contiguous().view(torch.int8).double() * half(0)
    elif qt == "q5_0":
        qh = sum(byte(2 + i, 3 + i) << (8 * i) for i in range(4))
        bit = torch.arange(32, device=w.device)
        q = torch.cat([byte(6, 22) & 15, byte(6, 22) >> 4], 1) | (((qh >> bit) & 1) << 4)
        v = (q - 16).double() * half(0)
    elif qt == "q4_k":
        s = byte(4, 16)
        lo, hi = s[:, :4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)
        mlo, mhi = s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)
        sc, mn = torch.cat([lo, hi], 1).double(), torch.cat([mlo, mhi], 1).double()
        qs = byte(16, 144).view(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
        v = half(0)[:, :, None] * sc[:, :, None] * q - half(2)[:, :, None] * mn[:, :, None]
    else:
        ql, qh = byte(0, 128).view(-1, 2, 2, 32), byte(128, 192).view(-1, 2, 1, 32)
        nib = torch.cat([ql & 15, ql >> 4], 2)
        sh = torch.tensor([0, 2, 4, 6], device=w.device).view(1, 1, 4, 1)
        q = ((nib | (((qh >> sh) & 3) << 4)) - 32).double().reshape(-1, 16, 16)
        sc = w[:, 192:208].contiguous().view(torch.int8).double().view(-1, 16, 1)
        v = half(208)[:, :, None] * sc * q
    return v.reshape(rows, cols)


def _gemv64(w, qt, rows, cols, x):
    out, nb = [], cols // QBLOCK[qt][0]
    for i in range(0, rows, 4096):
        n = min(4096, rows - i)
        out.append(_dequant(w[i * nb:(i + n) * nb], qt, n, cols) @ x.double())
    return torch.cat(out)


def _rope64(x, pos):
    """Adjacent-pair RoPE of [..., heads, 64] at `pos` (a number, or one for each leading row): the angle is the
    fp32 product pos * (1 / base^(d/64)) that defines the position, its sine and cosine taken in 64 bits."""
    theta = torch.tensor([np.float32(1) / np.float32(math.pow(BASE, d / HD)) for d in range(0, HD, 2)],
                         dtype=torch.float32, device=x.device)
    a = (torch.as_tensor(pos, device=x.device).float()[..., None] * theta).double()[..., None, :]
    c, s = torch.cos(a), torch.sin(a)
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack([x0 * c - x1 * s, x0 * s + x1 * c], -1).flatten(-2)


def _attend64(q, k, v):
    """q [nh][hd], k / v [rows][nkv][hd] in float64 -> [nh * hd]."""
    (nh, hd), nkv = q.shape, k.shape[1]
    s = torch.matmul(q.view(nkv, nh // nkv, hd), k.permute(1, 2, 0).contiguous()) / math.sqrt(hd)
    return torch.matmul(torch.softmax(s, -1), v.transpose(0, 1).contiguous()).reshape(-1)


def exact(case, seed):
    k = case["kind"]
    s = prepare(case, seed)
    if k in ("ops", "step"):
        layers, pos = (1, case["past_len"]) if k == "ops" else (LAYERS, case["pos"])
        proj = k == "ops" or case["proj"]
        kc, vc = s.kc.double(), s.vc.double()
        q, kn, vn = (t.double() for t in (s.q, s.kn, s.vn))
        if proj:
            q, kn, vn = (torch.stack([_dequant(w.view(layers, -1, w.shape[1])[i], qt, r, QD) @ s.x[i].double() + b[i].double()
                                      for i in range(layers)])
                         for w, qt, r, b in ((s.wq, "q5_0", QD, s.bq), (s.wk, "q5_0", KVD, s.bk),
                                             (s.wv, "q8_0", KVD, s.bv)))
        qr = _rope64(q.view(layers, NH, HD), pos)
        kc[:, pos] = _rope64(kn.view(layers, NKV, HD), pos).reshape(layers, KVD)
        vc[:, pos] = vn
        out = torch.stack([_attend64(qr[i], kc[i, :pos + 1].view(-1, NKV, HD), vc[i, :pos + 1].view(-1, NKV, HD))
                           for i in range(layers)])
        res = {"out": out, "k": kc, "v": vc}
        if proj:
            o = [_dequant(s.wo.view(layers, -1, 22)[i], "q5_0", QD, QD) @ out[i] for i in range(layers)]
            res["h"] = o[0] if k == "ops" else s.h0.double() + torch.stack(o).sum(0)
            if k == "step":
                res["q"] = q
        return res
    if k == "gemv":
        return _gemv64(s.w, case["qtype"], case["rows"], case["cols"], s.x)
    if k == "any":
        nh, nkv, hd, n = case["nh"], case["nkv"], case["hd"], case["n_pos"]
        return torch.stack([_attend64(s.q[i].double().view(nh, hd), s.k[i * n:(i + 1) * n].double().view(n, nkv, hd),
                                      s.v[i * n:(i + 1) * n].double().view(n, nkv, hd)) for i in range(case["n_seq"])])
    name = case["cache"]
    per = 1 if name != "q8" else NKV  # stored rows of the cache tensor per cache row

    def rows_of(t, idx):
        if per > 1:
            idx = (idx[:, None] * per + torch.arange(per, device=idx.device)).reshape(-1)
        return _values(t[idx], name)

    def row_index(i, n, base):
        r = torch.arange(n, device="cuda")
        return base + r if not hasattr(s, "table") else s.table[i][r // 16].long() * 16 + r % 16

    if k in ("prefill", "prompt"):
        # The path's operands are q, k and v rounded to bf16, its sums and weights fp32.
        n, n_q, prefix = case["n_seq"], case["n_q"], case["prefix"]
        rows = prefix + n_q
        out = torch.empty(n, n_q, NH, HD, device="cuda", dtype=torch.float64)
        for i in range(n):
            idx = row_index(i, rows, i * rows)
            kk, vv = (rows_of(t, idx).float().to(torch.bfloat16).double() for t in (s.k, s.v))
            qq = s.q[i].to(torch.bfloat16).double().view(n_q, NH, HD)
            hidden = torch.arange(rows, device="cuda")[None, :] > (prefix + torch.arange(n_q, device="cuda"))[:, None]
            for h in range(NH):
                a = torch.matmul(qq[:, h].contiguous(), kk[:, h // G].t().contiguous()) / math.sqrt(HD)
                a = torch.softmax(a.masked_fill_(hidden, -math.inf), -1)
                out[i, :, h] = torch.matmul(a, vv[:, h // G].contiguous())
        return out.view(n, n_q, QD)
    n = case["n_seq"]
    lens = np.full(n, case["n_pos"]) if k == "decode" else _lens(case)
    base = np.concatenate([[0], np.cumsum(lens[:-1].astype(np.int64))])
    out = torch.empty(n, QD, device="cuda", dtype=torch.float64)
    q = s.q.double().view(n, NH, HD)
    if k != "serve":
        for i in range(n):
            idx = row_index(i, int(lens[i]), int(base[i]))
            out[i] = _attend64(q[i], rows_of(s.k, idx), rows_of(s.v, idx))
        return out
    # The layer step: q and the new k rotated at the last row, the new row in the cache's own type.
    q = _rope64(q, s.pos)
    kn = _rope64(s.kn.double().view(n, NKV, HD), s.pos)
    vn = s.vn.double().view(n, NKV, HD)
    at = torch.stack([row_index(i, int(lens[i]), 0)[-1] for i in range(n)])
    if name == "q8":  # stored bytes are not computed numbers; attend what the reference's rule stores
        new_k, new_v = _quantized(kn), _quantized(vn)
        res = {"out": out, "k": None, "v": None}
    else:
        new_k, new_v = (t.to(s.k.dtype).double() if name != "f32" else t for t in (kn, vn))
        full = [t.double() for t in (s.k, s.v)]
        full[0][at], full[1][at] = new_k.reshape(n, KVD), new_v.reshape(n, KVD)
        res = {"out": out, "k": full[0], "v": full[1]}
    for i in range(n):
        idx = row_index(i, int(lens[i]), 0)
        kk, vv = rows_of(s.k, idx), rows_of(s.v, idx)
        kk[-1], vv[-1] = new_k[i], new_v[i]
        out[i] = _attend64(q[i], kk, vv)
    return res


def _quantized(x):
    """Blocks of 32 as a Q8_0 cache holds them: d = max|x| / 127 in fp16 (truncated), q rounded half to even."""
    y = x.float().reshape(-1, 32)
    d = y.abs().amax(-1, keepdim=True) / 127
    q = torch.round(y / d)
    bits = d.view(torch.int32)
    dh = ((((bits >> 23) & 0xFF) - 112) << 10) | ((bits & 0x7FFFFF) >> 13)
    return (q.double() * dh.to(torch.int16).view(torch.float16).double()).view(x.shape)


def tolerance(case):
    # About four times the largest error against `exact` that was seen for the kind: 32-bit sums 3.4e-7 (long
    # contexts add rows), 16-bit and quantized caches 2.4e-6 (queries and weights in 16-bit parts), prefill 4.8e-6
    # (weights in two bf16 parts).
    k = case["kind"]
    if k in ("prefill", "prompt"):
        return {"rel": 2e-5, "max": 1e-3}
    if case.get("cache", "f32") != "f32":
        if k == "serve":  # a rotated value on a rounding edge of the cache's type may fall either way
            return {"rel": 1e-4, "max": 1e-2}
        return {"rel": 1e-5, "max": 5e-4}
    return {"rel": 2e-6, "max": 1e-4}
