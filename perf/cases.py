"""Timed cases of the Qwen2 attention library: what a TTS or ASR program has it do.

Every case is a call sequence of the C ABI (include/vva.h) over the shapes of
the 0.5B, 1.5B and 7B language models, with the tensor descriptors built once,
as a C++ caller holds them.  The five kinds:

  step   one new token per sequence over `layers` layers: vva_decode_step
  prefill  a run of tokens: vva_rope_append, vva_attn
  block  the attention half of a layer, normed input to residual sum:
         projections + RoPE + append, attention, output projection
  proj   its two linear layers alone, at their prefill sizes
  flash  vva_flash_attn_ext on strided K and V with an explicit mask

listed() gives the fixed cases, draw() others of the same ranges, prepare()
the state a program holds before the call, run() one pass, work() the bytes and
operations of a pass, tolerance() how far two correct results may differ, and
exact() the result in 64 bits.
"""
import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

THETA = 1.0e6
# hidden size, query heads, kv heads, head dim
MODELS = {"0.5b": (896, 14, 2, 64), "1.5b": (1536, 12, 2, 128), "7b": (3584, 28, 4, 128)}
TYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def _vva():
    """The binding of the tree that is the working folder."""
    if "vva" not in sys.modules:
        path = os.path.join(os.getcwd(), "vibevoice.cpp_amd", "vva.py")
        spec = importlib.util.spec_from_file_location("vva", path)
        mod = importlib.util.module_from_spec(spec)
        sys.modules["vva"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["vva"]


def _case(kind, model, cache, tokens, past, batch=1, layers=1, ragged=False, weights="f16", io="f32", flash=True,
          mask="f16"):
    return {"kind": kind, "model": model, "cache": cache, "tokens": tokens, "past": past, "batch": batch,
            "layers": layers, "ragged": ragged, "weights": weights, "io": io, "flash": flash, "mask": mask}


def listed():
    cases = [
        # The classifier-free-guidance step of the realtime TTS: two streams, one token each, through the 24 layers
        # of the 0.5B model on a 1k F16 cache.  Latency and launches are all of it.
        ("step_tts_0p5b_f16_1k", _case("step", "0.5b", "f16", 1, 1024, batch=2, layers=24)),
        # The transcript decode of long-form ASR: Q8_0 caches of 32768 positions, two streams.  Eight layers' caches
        # in rotation (570 MB), so they come from HBM as the 28 layers' do.
        ("step_asr_7b_q8_32k", _case("step", "7b", "q8_0", 1, 32768, batch=2, layers=8)),
        # The same decode of one stream on the F16 cache that a caller keeps when memory allows, 20k positions in.
        ("step_asr_7b_f16_20k", _case("step", "7b", "f16", 1, 20011, layers=8)),
        # The guidance step of the 1.5B TTS behind its 4k voice prompt on the F32 cache, the type the reference itself
        # keeps: two streams, the second shorter.
        ("step_tts_1p5b_f32_4k", _case("step", "1.5b", "f32", 1, 4096, batch=2, layers=8, ragged=True)),
        # The attention half of a 7B decode layer with Q8_0 weights and cache: two streams of different lengths,
        # eight layers' weights in rotation.
        ("block_step_7b_q8", _case("block", "7b", "q8_0", 1, 2048, batch=2, layers=8, ragged=True, weights="q8_0")),
        # One five-token text window of the realtime TTS behind its voice prompt, four layers.
        ("block_window_0p5b_f16", _case("block", "0.5b", "f16", 5, 611, layers=4, weights="q8_0")),
        # The 0.5B prompt (257 tokens, none a multiple of a tile) on the reference's own F32 cache.
        ("block_prompt_0p5b_f32", _case("block", "0.5b", "f32", 257, 0, layers=4)),
        # The 1.5B voice-cloning prompt: 4096 tokens, BF16 tensors and cache.
        ("prefill_voice_1p5b_bf16_4k", _case("prefill", "1.5b", "bf16", 4096, 0, io="bf16")),
        # Long-form ASR in one prefill: 32768 tokens, BF16 tensors, F16 cache.  The largest case.
        ("prefill_asr_7b_f16_32k", _case("prefill", "7b", "f16", 32768, 0, io="bf16")),
        # One of the 512-token chunks that the ASR program really prefills in, half-way through an hour, Q8_0 cache.
        ("prefill_chunk_7b_q8_16k", _case("prefill", "7b", "q8_0", 512, 15872, io="bf16")),
        # The linear layers of a 4096-token prefill, F16 weights.
        ("proj_7b_f16_4k", _case("proj", "7b", "f16", 4096, 0, weights="f16")),
        # The linear layers of a 512-token chunk with the Q8_0 weights that GGUF files ship.
        ("proj_chunk_7b_q8", _case("proj", "7b", "f16", 512, 512, weights="q8_0")),
    ]
    return [dict(name=n, **c) for n, c in cases]


def draw(rng):
    """Another case of these ranges: sizes spread over their logarithm, odd ones among them."""
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["step", "step", "prefill", "prefill", "block", "block", "proj", "flash"])
    model = rng.choice(list(MODELS))
    cache = rng.choice(["f16", "f16", "q8_0", "bf16", "f32"])
    io = rng.choice(["f32", "f32", "bf16", "f16"])
    weights = rng.choice(["f16", "q8_0"])
    ragged = rng.random() < 0.5
    if kind == "step":
        return _case(kind, model, cache, 1, size(32, 32768), batch=rng.choice([1, 1, 2, 2, 2, 4]), layers=4,
                     ragged=ragged, io=io)
    if kind == "prefill":
        flash = cache != "f32" or rng.random() < 0.6
        # the fp32 eager branch is the reference's comparator at prompt sizes
        return _case(kind, model, cache, size(9, 8192) if flash else size(9, 600), rng.choice([0, size(64, 16384)]) if
                     flash else 0, batch=rng.choice([1, 1, 1, 2]), ragged=ragged, io=io, flash=flash)
    if kind == "block":
        step = rng.random() < 0.4
        return _case(kind, model, cache, 1 if step else size(2, 2048), size(32, 8192), batch=rng.choice([1, 2, 2, 4]) if
                     step else 1, layers=4, ragged=ragged, weights=weights, io=io)
    if kind == "proj":
        return _case(kind, model, cache if cache != "f32" else "f16", size(16, 4096), size(1, 2048), weights=weights,
                     io=io)
    # the drop-in ggml call: permuted Q, strided K and V, the caller's own mask over a window of any length
    return _case(kind, model, cache if cache != "f32" else "f16", size(9, 1024), size(1, 8192), io=io,
                 mask=rng.choice(["f16", "f32"]))


# ------------------------------------------------------------------ inputs

def _pasts(c):
    """Valid rows of each sequence before the call: with `ragged`, later streams hold fewer."""
    return [c["past"] - (c["past"] * b // (2 * c["batch"]) if c["ragged"] else 0) for b in range(c["batch"])]


def _row_bytes(cache, d):
    return d // 32 * 34 if cache == "q8_0" else d * (4 if cache == "f32" else 2)


def _q8_pack(x):
    """F32 [..., n] -> GGUF Q8_0 blocks as bytes [..., n / 32 * 34]."""
    b = x.float().unflatten(-1, (-1, 32))
    d = b.abs().amax(-1, keepdim=True) / 127.0
    inv = torch.where(d > 0, 1.0 / d, torch.zeros_like(d))
    y = b * inv
    codes = (torch.sign(y) * torch.floor(y.abs() + 0.5)).to(torch.int8)
    return torch.cat([d.half().view(torch.uint8), codes.view(torch.uint8)], -1).flatten(-2)


def _q8_unpack(raw):
    """Q8_0 bytes [..., n / 32 * 34] -> F64 [..., n]."""
    b = raw.unflatten(-1, (-1, 34))
    d = b[..., :2].contiguous().view(torch.float16).double()
    return (b[..., 2:].contiguous().view(torch.int8).double() * d).flatten(-2)


def _inputs(c, seed):
    """Every tensor of a case, from the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    hidden, hq, hkv, d = MODELS[c["model"]]
    T, B, n = c["tokens"], c["batch"], c["layers"]
    io = TYPES[c["io"]]

    def normal(*shape, dtype=torch.float32, scale=1.0):
        return (torch.randn(shape, generator=gen, device="cuda") * scale).to(dtype)

    s = {"io": io}
    if c["kind"] == "flash":
        L = c["past"] + T
        s["q"] = normal(1, hq, T, d, dtype=io)
        raw = normal(2, L, hkv, d)
        s["kv"] = _q8_pack(raw) if c["cache"] == "q8_0" else raw.to(TYPES[c["cache"]])
        # the mask a caller builds: 0 up to the query's own position, -inf past it, the rows padded
        pad = (L + 31) // 32 * 32
        j = torch.arange(pad, device="cuda")
        i = torch.arange(T, device="cuda")[:, None] + c["past"]
        s["mask"] = torch.where(j <= i, 0.0, float("-inf")).to(TYPES[c["mask"]])[None].contiguous()
        return s
    # the cache rows each sequence already holds: [layers][seq] of [2, past, hkv, row]
    s["past"] = []
    for _ in range(n):
        rows = []
        for p in _pasts(c):
            raw = normal(2, p, hkv, d)
            rows.append(_q8_pack(raw) if c["cache"] == "q8_0" else raw.to(TYPES[c["cache"]]))
        s["past"].append(rows)
    s["pos"] = torch.stack([torch.arange(p, p + T, dtype=torch.int32, device="cuda") for p in _pasts(c)])
    if c["kind"] in ("step", "prefill"):
        s["q"] = normal(n, B, T, hq, d, dtype=io)
        s["k"] = normal(n, B, T, hkv, d, dtype=io)
        s["v"] = normal(n, B, T, hkv, d, dtype=io)
    else:
        def weight(m, k):
            w = normal(n, m, k, scale=k ** -0.5)
            return _q8_pack(w) if c["weights"] == "q8_0" else w.half()
        s["xn"] = normal(n, B, T, hidden, dtype=io)
        s["x"] = normal(n, B, T, hidden)
        s["w"] = {"q": weight(hq * d, hidden), "k": weight(hkv * d, hidden), "v": weight(hkv * d, hidden),
                  "o": weight(hidden, hq * d)}
        s["b"] = {"q": normal(n, hq * d, scale=0.1), "k": normal(n, hkv * d, scale=0.1),
                  "v": normal(n, hkv * d, scale=0.1)}
        if c["kind"] == "proj":
            s["o"] = normal(n, B, T, hq * d, scale=0.2)
    return s


# ---------------------------------------------------------------- the state

class _DeviceArray:
    """Device memory of a library object, for torch.as_tensor.  The tensor's storage holds this object, and so the
    owner: the memory outlives every view of it."""

    def __init__(self, owner, ptr, shape, strides, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "strides": strides,
                                         "typestr": typestr, "version": 2}


def _cache_tensor(kv, cache, hkv, d):
    """The resident cache as a torch tensor [layer][seq][K, V][row][head * d] (Q8_0: the blocks' bytes)."""
    def ptr(layer, seq, which):
        return int(kv.views(layer, seq)[which].data)
    base = ptr(0, 0, 0)
    pair = ptr(0, 0, 1) - base
    seq = ptr(0, 1, 0) - base if kv.n_seq > 1 else 2 * pair
    lay = ptr(1, 0, 0) - base if kv.n_layers > 1 else seq * kv.n_seq
    row = hkv * _row_bytes(cache, d)
    kind, es = {"f32": ("<f4", 4), "f16": ("<f2", 2), "bf16": ("<i2", 2), "q8_0": ("|u1", 1)}[cache]
    t = torch.as_tensor(_DeviceArray(kv, base, (kv.n_layers, kv.n_seq, 2, kv.max_seq, row // es),
                                     (lay, seq, pair, row, es), kind), device="cuda")
    return t.view(torch.bfloat16) if cache == "bf16" else t


def prepare(case, seed):
    """Context, resident cache with its past rows, weights and descriptors: what a program holds between calls."""
    vva = _vva()
    c = case
    hidden, hq, hkv, d = MODELS[c["model"]]
    T, B, n = c["tokens"], c["batch"], c["layers"]
    s = _inputs(c, seed)
    ctx = vva.Context(0)
    st = {"ctx": ctx, "lib": ctx.lib, "h": ctx.h, "keep": s, "scale": d ** -0.5}
    refs = st["refs"] = []

    def ref(t, **kw):
        v = vva.view(t, **kw)
        refs.append(v)
        return ctypes.byref(v)

    if c["kind"] == "flash":
        L = c["past"] + T
        rb = _row_bytes(c["cache"], d)
        typ = {"f16": vva.F16, "bf16": vva.BF16, "q8_0": vva.Q8_0}[c["cache"]]
        es = 34 if c["cache"] == "q8_0" else 2
        kv_ref = [ref(s["kv"][i], ggml_ne=[d, L, hkv, 1], ggml_nb=[es, hkv * rb, rb, L * hkv * rb], type_=typ)
                  for i in range(2)]
        st["out"] = torch.empty((1, T, hq, d), device="cuda")
        m = s["mask"]
        es = m.element_size()
        mask = ref(m, ggml_ne=[m.shape[2], T, 1, 1], ggml_nb=[es, m.stride(1) * es, m.stride(1) * es * T,
                                                              m.stride(1) * es * T],
                   type_=vva.F32 if es == 4 else vva.F16)
        q, out = ref(s["q"]), ref(st["out"])
        st["calls"] = [(ctx.lib.vva_flash_attn_ext,
                        (ctx.h, q, kv_ref[0], kv_ref[1], mask, st["scale"], 0.0, 0.0, out))]
        st["result"] = {"out": st["out"]}
        return st

    typ = {"f32": vva.F32, "f16": vva.F16, "bf16": vva.BF16, "q8_0": vva.Q8_0}[c["cache"]]
    pasts = _pasts(c)
    kv = vva.KVCache(ctx, n, hkv, d, c["past"] + T, B, typ)
    st["kv"] = kv
    mem = _cache_tensor(kv, c["cache"], hkv, d)
    for layer in range(n):
        for b, p in enumerate(pasts):
            if p:
                mem[layer, b, :, :p] = s["past"][layer][b].flatten(2)
    del s["past"]
    for b, p in enumerate(pasts):
        kv.set_len(b, p)
    if not c["flash"]:
        ctx.set_flash_attn(False)
    # the rows the call appends: results, beside what it returns
    rows = [mem[:, b, :, p:p + T] for b, p in enumerate(pasts)]
    pos = ref(s["pos"])
    h, lib, scale = ctx.h, ctx.lib, st["scale"]
    qr = torch.empty((n, B, T, hq, d), dtype=s["io"], device="cuda")
    out = torch.empty((n, B, T, hq, d), device="cuda")
    calls = st["calls"] = []
    if c["kind"] == "step":
        for i in range(n):
            calls.append((lib.vva_decode_step, (h, kv.h, i, ref(s["q"][i]), ref(s["k"][i]), ref(s["v"][i]), pos, None,
                                                THETA, scale, ref(qr[i]), ref(out[i]))))
        st["result"] = {"out": out, "q": qr, "rows": rows}
        return st
    if c["kind"] == "prefill":
        for i in range(n):
            q = ref(qr[i])
            calls.append((lib.vva_rope_append, (h, kv.h, i, ref(s["q"][i]), ref(s["k"][i]), ref(s["v"][i]), pos, None,
                                                THETA, q)))
            calls.append((lib.vva_attn, (h, kv.h, i, q, None, None, scale, ref(out[i]))))
        st["result"] = {"out": out, "q": qr, "rows": rows}
        return st

    def weight(name, i, m, k):
        w = vva.Weight(s["w"][name][i].reshape(-1).view(torch.uint8), typ_w, k, m)
        refs.append(w)
        return ctypes.byref(w.t)
    typ_w = vva.Q8_0 if c["weights"] == "q8_0" else vva.F16
    hs = torch.empty_like(s["x"])
    m_all = (hq + 2 * hkv) * d
    fused = c["kind"] == "block" and T == 1 and c["cache"] == "q8_0"
    y = torch.empty((n, B, T, m_all), device="cuda") if fused else None
    for i in range(n):
        w = [weight("q", i, hq * d, hidden), weight("k", i, hkv * d, hidden), weight("v", i, hkv * d, hidden),
             weight("o", i, hidden, hq * d)]
        bias = [ref(s["b"][k][i]) for k in "qkv"]
        q, xn = ref(qr[i]), ref(s["xn"][i])
        if fused:
            calls.append((lib.vva_qkv_proj, (h, xn, *w[:3], *bias, ref(y[i]))))
            qkv = [ref(t.unflatten(-1, (-1, d))) for t in
                   y[i].split([hq * d, hkv * d, hkv * d], -1)]
            calls.append((lib.vva_decode_step, (h, kv.h, i, *qkv, pos, None, THETA, scale, q, ref(out[i]))))
        else:
            calls.append((lib.vva_qkv_rope_append, (h, kv.h, i, xn, *w[:3], *bias, pos, None, THETA, q)))
            if c["kind"] == "block":
                calls.append((lib.vva_attn, (h, kv.h, i, q, None, None, scale, ref(out[i]))))
        o = s["o"][i] if c["kind"] == "proj" else out[i].flatten(-2)
        calls.append((lib.vva_out_proj_residual, (h, ref(o), w[3], ref(s["x"][i]), ref(hs[i]))))
    st["result"] = {"h": hs, "q": qr, "rows": rows}
    if c["kind"] == "block":
        st["result"]["out"] = out
    return st


def run(state):
    """One pass: the calls in a layer stack's order, on the context's stream.  The lengths stay where they are, so a
    pass appends the same rows again."""
    check = state["ctx"].check
    for fn, args in state["calls"]:
        check(fn(*args))
    return state["result"]


# ------------------------------------------------------- work and tolerance

def work(case):
    c = case
    hidden, hq, hkv, d = MODELS[c["model"]]
    T, B = c["tokens"], c["batch"]
    io = 4 if c["io"] == "f32" else 2
    row = hkv * _row_bytes(c["cache"], d)
    pasts = _pasts(c)
    seen = sum(p + T for p in pasts)                                    # cache rows attended to
    pairs = sum(T * p + T * (T + 1) // 2 for p in pasts)                # visible (query, key) pairs
    attn_flops = 4.0 * hq * d * pairs
    n_tok = T * B
    if c["kind"] == "flash":
        L = c["past"] + T
        mask = T * L * (4 if c["mask"] == "f32" else 2)
        return {"bytes": 2.0 * L * row + mask + T * hq * d * (io + 4), "flops": attn_flops}
    if c["kind"] in ("step", "prefill"):
        # q, k, v in; the rotated q, the new rows and the output written; the window read
        b = n_tok * ((hq + 2 * hkv) * d * io + hq * d * (io + 4) + 2 * row) + 2 * seen * row
        return {"bytes": float(b) * c["layers"], "flops": attn_flops * c["layers"]}
    wrow = hidden // 32 * 34 if c["weights"] == "q8_0" else 2 * hidden
    orow = hq * d // 32 * 34 if c["weights"] == "q8_0" else 2 * hq * d
    m = (hq + 2 * hkv) * d
    b = m * (wrow + 4) + hidden * orow                                  # the weights and biases
    b += n_tok * (hidden * (io + 8) + hq * d * (io + 4) + 2 * row)      # xn, x, h; the rotated q, o; the new rows
    f = 2.0 * n_tok * (hidden * m + hq * d * hidden)
    if c["kind"] == "block":
        b += 2 * seen * row
        f += attn_flops
    return {"bytes": float(b) * c["layers"], "flops": f * c["layers"]}


def tolerance(case):
    """About four times what the coarsest type on a case's path was seen to put between a result and its 64-bit value
    (2-norm): 1.7e-3 where rows or outputs are BF16; 4.6e-4 where dot products run on dequantized Q8_0 blocks; 2.1e-4
    where rows, outputs or probabilities are F16; 6e-7 where everything is F32."""
    c = case
    q8_weights = c["kind"] in ("block", "proj") and c["weights"] == "q8_0"
    # F32 caches: one token and the eager branch stay in F32; a block's projections read F16 or Q8_0 weights
    f32 = c["cache"] == "f32" and c["io"] == "f32" and c["kind"] in ("step", "prefill") and (
        c["tokens"] == 1 or not c["flash"])
    if c["io"] == "bf16" or c["cache"] == "bf16":
        rel = 7e-3
    elif c["cache"] == "q8_0" or q8_weights:
        rel = 2e-3
    else:
        rel = 2.5e-6 if f32 else 1e-3
    # codes of Q8_0 rows: a value next to a rounding tie lands on either side; more of them do where the value comes
    # out of products of dequantized weights
    return {"rel": rel, "differ": 1e-2 if q8_weights else 1e-3}


# ------------------------------------------------------------ 64-bit results

def _rope64(x, pos, d):
    """NeoX rotation of [B, T, H, d] in 64 bits, by the fp32 angle recurrence that defines the positions' angles."""
    ts = float(np.float32(math.pow(THETA, -2.0 / d)))
    th, steps = pos.float(), []
    for _ in range(d // 2):
        steps.append(th)
        th = th * torch.tensor(ts, dtype=torch.float32, device="cuda")
    ang = torch.stack(steps, -1).double()[:, :, None]
    c, s = torch.cos(ang), torch.sin(ang)
    a, b = x.double().split(d // 2, -1)
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def _as_cache(x, cache):
    """Values as the cache holds them."""
    if cache == "q8_0":
        return _q8_unpack(_q8_pack(x.float()))
    return x.float().to(TYPES[cache]).double()


def _attend64(q, k, v, past, scale, mask=None):
    """q [T, Hq, d], k and v [L, Hkv, d] in 64 bits -> [T, Hq, d]; causal from `past`, or by the mask rows."""
    T, hq, d = q.shape
    L, hkv, _ = k.shape
    g = hq // hkv
    out = torch.empty_like(q)
    step = max(1, int(2.5e8 // (g * L)))
    j = torch.arange(L, device="cuda")
    for hk in range(hkv):
        kt, vh = k[:, hk].t().contiguous(), v[:, hk].contiguous()
        for t0 in range(0, T, step):
            qt = q[t0:t0 + step, hk * g:(hk + 1) * g]
            n = qt.shape[0]
            sc = (qt.reshape(n * g, d) @ kt).view(n, g, L) * scale
            if mask is None:
                hidden = j > (past + torch.arange(t0, t0 + n, device="cuda"))[:, None]
                sc.masked_fill_(hidden[:, None], float("-inf"))
            else:
                sc += mask[t0:t0 + n, None, :L].double()
            out[t0:t0 + n, hk * g:(hk + 1) * g] = (torch.softmax(sc, -1).view(n * g, L) @ vh).view(n, g, d)
    return out


def exact(case, seed):
    """What run() returns, computed in 64 bits.  What the library documents as its operands' roundings (Q to the type
    of K, the input rows to the weights' dot type, the rows to the cache's type) is part of the inputs here."""
    c = case
    hidden, hq, hkv, d = MODELS[c["model"]]
    T, B, n = c["tokens"], c["batch"], c["layers"]
    scale = d ** -0.5
    s = _inputs(c, seed)
    # an F32 cache is read in F16 on the flash branch of a prefill, Q with it
    kt = "f16" if c["cache"] == "f32" and c["flash"] and T > 1 else c["cache"]

    def window(raw):
        return _q8_unpack(raw) if c["cache"] == "q8_0" else raw.double()

    def heads(x):
        return _as_cache(x.to(s["io"]), kt)

    if c["kind"] == "flash":
        k, v = window(s["kv"])
        return {"out": _attend64(heads(s["q"][0]).transpose(0, 1).contiguous(), k, v, 0, scale, s["mask"][0])[None]}

    def layer(i, q, k, v):
        """RoPE, append and attention of a layer: (rotated q, new rows per sequence, output)."""
        qr, kr = _rope64(q, s["pos"], d), _rope64(k, s["pos"], d)
        outs, rows = [], []
        for b, p in enumerate(_pasts(c)):
            rows.append(torch.stack([kr[b], v[b].double()]))
            if c["kind"] != "proj":
                win = torch.cat([window(s["past"][i][b]), _as_cache(rows[-1], c["cache"])], 1)
                if kt != c["cache"]:
                    win = _as_cache(win, kt)
                outs.append(_attend64(heads(qr[b]), win[0], win[1], p, scale))
        return qr, rows, torch.stack(outs) if outs else None

    def linear(x, w):
        x = _q8_unpack(_q8_pack(x.float())) if c["weights"] == "q8_0" else x.half().double()
        w = _q8_unpack(w) if c["weights"] == "q8_0" else w.double()
        return x.flatten(0, 1) @ w.t().contiguous()

    res = {"out": [], "q": [], "h": []}
    rows = [[] for _ in range(B)]
    for i in range(n):
        if c["kind"] in ("step", "prefill"):
            q, k, v = s["q"][i], s["k"][i], s["v"][i]
        else:
            q, k, v = ((linear(s["xn"][i], s["w"][m][i]) + s["b"][m][i].double()).view(B, T, -1, d) for m in "qkv")
        qr, new, out = layer(i, q, k, v)
        res["q"].append(qr)
        res["out"].append(out)
        for b in range(B):
            rows[b].append(new[b].flatten(2))
        if c["kind"] in ("block", "proj"):
            o = out.float().flatten(-2) if c["kind"] == "block" else s["o"][i]
            res["h"].append(s["x"][i].double() + linear(o, s["w"]["o"][i]).view(B, T, hidden))
    got = {"q": torch.stack(res["q"])}
    if c["kind"] != "proj":
        got["out"] = torch.stack(res["out"])
    if res["h"]:
        got["h"] = torch.stack(res["h"])
    # the bytes of Q8_0 rows have no 64-bit value
    got["rows"] = [None if c["cache"] == "q8_0" else torch.stack(r) for r in rows]
    return got
