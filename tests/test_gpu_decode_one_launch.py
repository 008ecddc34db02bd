"""GPU parity of the one-launch single-token attention (decode_step.hip) where
its dispatch and its loops can go wrong: F32, F16 and BF16 caches at the edges
of a wave's keys and of a chunk, several chunks per workgroup, in-launch merge
and merge kernel, ragged streams whose short windows leave splits without a
key, strided K and V, scales of either sign.

Each call is compared with the general row kernel (attn_path 1) on the same
cache and with the fp64 oracle: 2e-3 max-abs / 1e-3 mean-abs for the 16-bit
types, 1e-4 for F32 (the tolerances of these paths everywhere)."""
import numpy as np
import pytest

import vva
from gpu_util import as_f32, assert_close, fill_cache, oracle_attn, to_gpu

pytestmark = pytest.mark.gpu

TOL = {vva.F32: (1e-4, 1e-4), vva.F16: (2e-3, 1e-3), vva.BF16: (2e-3, 1e-3)}

CASES = [
    # d, Hq, Hkv, lens after the step, workgroups planned for (0: automatic)
    (64, 14, 2, [1], 0),
    (64, 8, 1, [16, 17, 32, 33], 0),
    (128, 28, 4, [63, 64, 65], 0),
    (128, 12, 2, [127, 128, 129], 0),
    (128, 28, 4, [3001, 70], 0),          # the second stream has far fewer chunks than there are splits
    (64, 14, 2, [2500, 2049], 8),         # 2 splits per stream and head: many chunks each, in-launch merge
    (128, 12, 2, [4600], 2),              # one split: no merge
    (128, 4, 4, [4097, 1], 160),          # one query head per kv head, 20 splits at most: merge kernel
]


@pytest.mark.parametrize("t", [vva.F32, vva.F16, vva.BF16])
@pytest.mark.parametrize("d,Hq,Hkv,lens,wgs", CASES)
def test_one_launch_step_and_attention(ctx, torch_gpu, d, Hq, Hkv, lens, wgs, t):
    torch = torch_gpu
    B = len(lens)
    print(f"one-launch d={d} Hq={Hq} Hkv={Hkv} type={t} lens={lens} wgs={wgs}", flush=True)
    past = [n - 1 for n in lens]
    a = vva.KVCache(ctx, 1, Hkv, d, max(lens), B, t)
    u = vva.KVCache(ctx, 1, Hkv, d, max(lens), B, t)
    for kv in (a, u):
        fill_cache(kv, past, seed=d + sum(lens))
    rng = np.random.default_rng(11)
    for it in (vva.F32, vva.BF16):
        q, k, v = (to_gpu(torch, rng.standard_normal((B, 1, n, d)), it) for n in (Hq, Hkv, Hkv))
        pos = torch.tensor([[n] for n in past], dtype=torch.int32, device="cuda")
        qa, qu = torch.empty_like(q), torch.empty_like(q)
        oa, ou, of = (torch.full((B, 1, Hq, d), float("nan"), device="cuda") for _ in range(3))
        with ctx.schedule(decode_wgs=wgs):
            ctx.decode_step(a, 0, q, k, v, pos, qa, oa, d ** -0.5)
            splits = ctx.last_decode_splits()
            ctx.rope_append(u, 0, q, k, v, pos, qu)
            ctx.attn(u, 0, qu, of, d ** -0.5)             # the attention alone, same kernel
        ctx.set_attn_path(1)
        try:
            ctx.attn(u, 0, qu, ou, d ** -0.5)             # the row kernel
        finally:
            ctx.set_attn_path(0)
        torch.cuda.synchronize()
        assert torch.equal(qa, qu), "rotated q differs"
        assert torch.equal(oa, of), "the step differs from append + attention"
        for s in range(B):
            for x, y in zip(a.download(0, s, lens[s]), u.download(0, s, lens[s])):
                np.testing.assert_array_equal(x, y)
        assert_close(as_f32(torch, oa), as_f32(torch, ou), *TOL[t], what="vs the row kernel")
        ref = oracle_attn(as_f32(torch, qa), a, 0, range(B), lens, 1, d ** -0.5)
        mx, mn = assert_close(as_f32(torch, oa), ref, *TOL[t], what="vs exact")
        print(f"  q type {it}: {splits} splits, vs exact max {mx:.2e} mean {mn:.2e}")
    # scales of either sign and zero (a uniform mean of V)
    for scale in (-0.2, 0.0):
        ctx.attn(u, 0, qu, of, scale)
        torch.cuda.synchronize()
        ref = oracle_attn(as_f32(torch, qu), u, 0, range(B), lens, 1, scale)
        assert_close(as_f32(torch, of), ref, *TOL[t], what=f"scale {scale}")
    a.free()
    u.free()


@pytest.mark.parametrize("dt", ["float32", "float16", "bfloat16"])
def test_one_token_flash_on_strided_rows(ctx, torch_gpu, dt):
    """vva_flash_attn_ext, one token, K and V of different strides (V inside a
    wider tensor), equal to the same values laid out densely."""
    torch = torch_gpu
    d, Hq, Hkv, L, B = 64, 14, 2, 777, 2
    print(f"flash one token strided {dt}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(3)
    typ = getattr(torch, dt)
    q = torch.randn((B, Hq, 1, d), generator=gen, device="cuda")
    k = torch.randn((B, L, Hkv, d), generator=gen, device="cuda").to(typ).transpose(1, 2)    # [B, Hkv, L, d] view
    wide = torch.randn((B, Hkv, L, 2 * d), generator=gen, device="cuda").to(typ)
    v = wide[..., d:]
    outs = []
    for kk, vv in ((k, v), (k.contiguous(), v.contiguous())):
        out = torch.full((B, 1, Hq, d), float("nan"), device="cuda")
        ctx.flash_attn_ext(q, kk, vv, out, d ** -0.5)
        torch.cuda.synchronize()
        outs.append(out)
    assert torch.equal(outs[0], outs[1])
    g = Hq // Hkv
    qd = q.to(typ).double()                               # Q rounded to K's type
    s = torch.matmul(qd.view(B, Hkv, g, d), k.double().transpose(2, 3).contiguous()) * d ** -0.5
    ref = torch.matmul(torch.softmax(s, -1), v.double().contiguous()).view(B, 1, Hq, d)
    tol = 1e-4 if dt == "float32" else 2e-3
    assert (outs[0].double() - ref).abs().max().item() <= tol


@pytest.mark.parametrize("t", [vva.F16, vva.BF16])
@pytest.mark.parametrize("d,Hkv", [(64, 3), (128, 6)])
def test_other_head_counts_keep_fp32_probabilities(ctx, torch_gpu, d, Hkv, t):
    """kv head counts that do not divide 8, 16-bit caches: one-token attention
    and steps beyond 8192 keys keep the row kernel (fp32 probabilities and V):
    bit for bit, and a BF16 V beyond the f16 range stays finite."""
    torch = torch_gpu
    Hq, L = 2 * Hkv, 8300
    print(f"fp32 one-token d={d} Hkv={Hkv} type={t}", flush=True)
    a = vva.KVCache(ctx, 1, Hkv, d, L, 1, t)
    u = vva.KVCache(ctx, 1, Hkv, d, L, 1, t)
    rng = np.random.default_rng(d)
    k, v = (rng.standard_normal((L, Hkv, d)).astype(np.float32) for _ in range(2))
    if t == vva.BF16:
        v[L // 2] = 1e5                                     # 65504 is the largest finite f16
    for kv in (a, u):
        kv.upload(0, 0, 0, k, v)
    qkv = [to_gpu(torch, rng.standard_normal((1, 1, n, d)), vva.F32) for n in (Hq, Hkv, Hkv)]
    pos = torch.tensor([L - 1], dtype=torch.int32, device="cuda")
    qa, qu = torch.empty_like(qkv[0]), torch.empty_like(qkv[0])
    outs = [torch.full((1, 1, Hq, d), float("nan"), device="cuda") for _ in range(3)]
    for kv in (a, u):
        kv.set_len(0, L - 1)
    ctx.decode_step(a, 0, *qkv, pos, qa, outs[0], d ** -0.5)
    ctx.rope_append(u, 0, *qkv, pos, qu)
    ctx.attn(u, 0, qu, outs[1], d ** -0.5)
    ctx.set_attn_path(1)
    try:
        ctx.attn(u, 0, qu, outs[2], d ** -0.5)
    finally:
        ctx.set_attn_path(0)
    torch.cuda.synchronize()
    assert torch.equal(qa, qu)
    assert torch.isfinite(outs[2]).all()
    assert torch.equal(outs[0], outs[2]) and torch.equal(outs[1], outs[2])
    a.free()
    u.free()


@pytest.mark.parametrize("t,L", [(vva.F16, 1000), (vva.BF16, 130), (vva.F32, 60), (vva.F16, 5000)])
def test_step_output_on_8_byte_boundaries(ctx, torch_gpu, t, L):
    """Output rows 8 bytes off a 16-byte boundary: the one-launch step with the
    bits of the aligned call (the same splits), at most 16 splits otherwise."""
    torch = torch_gpu
    d, Hq, Hkv = 128, 28, 4
    print(f"8-byte output type={t} L={L}", flush=True)
    kv = vva.KVCache(ctx, 1, Hkv, d, L, 1, t)
    fill_cache(kv, [L - 1], seed=L)
    rng = np.random.default_rng(L)
    q, k, v = (to_gpu(torch, rng.standard_normal((1, 1, n, d)), vva.F32) for n in (Hq, Hkv, Hkv))
    pos = torch.tensor([L - 1], dtype=torch.int32, device="cuda")
    qo = torch.empty_like(q)
    wide = torch.full((2 + Hq * (d + 2),), float("nan"), device="cuda")
    outs = [torch.full((1, 1, Hq, d), float("nan"), device="cuda"), wide[2:].view(1, 1, Hq, d + 2)[..., :d]]
    splits = []
    for out in outs:
        ctx.decode_step(kv, 0, q, k, v, pos, qo, out, d ** -0.5)
        splits.append(ctx.last_decode_splits())
    torch.cuda.synchronize()
    if splits[0] <= 16:
        assert torch.equal(outs[0], outs[1]) and splits[0] == splits[1]
    else:
        assert splits[1] <= 16
        assert_close(as_f32(torch, outs[1]), as_f32(torch, outs[0]), *TOL[t], what="fewer splits")
    assert torch.isnan(wide[2:].view(Hq, d + 2)[:, d:]).all() and torch.isnan(wide[:2]).all()
    kv.free()


@pytest.mark.parametrize("L,key", [(500, 3), (3000, 2990)])
def test_infinite_value_on_an_f32_cache(ctx, torch_gpu, L, key):
    """An infinite V element: that dim is infinite and the others as the row
    kernel has them, merged in the launch (8 splits of 16 slots) and by the
    merge kernel (47 splits; the slots past the last one hold nothing)."""
    torch = torch_gpu
    d, Hq, Hkv = 128, 12, 2
    print(f"infinite V element L={L} key={key}", flush=True)
    kv = vva.KVCache(ctx, 1, Hkv, d, L, 1, vva.F32)
    rng = np.random.default_rng(L)
    k, v = (rng.standard_normal((L, Hkv, d)).astype(np.float32) for _ in range(2))
    v[key, :, 7] = np.inf
    kv.upload(0, 0, 0, k, v)
    kv.set_len(0, L - 1)
    q = to_gpu(torch, rng.standard_normal((1, 1, Hq, d)), vva.F32)
    outs = [torch.full((1, 1, Hq, d), float("nan"), device="cuda") for _ in range(2)]
    ctx.attn(kv, 0, q, outs[0], d ** -0.5)
    assert (ctx.last_decode_splits() > 16) == (L == 3000)
    ctx.set_attn_path(1)
    try:
        ctx.attn(kv, 0, q, outs[1], d ** -0.5)
    finally:
        ctx.set_attn_path(0)
    torch.cuda.synchronize()
    a, b = (as_f32(torch, o) for o in outs)
    assert np.isposinf(a[..., 7]).all() and np.isposinf(b[..., 7]).all()
    rest = np.arange(d) != 7
    assert_close(a[..., rest], b[..., rest], *TOL[vva.F32], what="the other dims")
    kv.free()


@pytest.mark.parametrize("t,past", [(vva.F32, 900), (vva.F16, 8300)])
def test_step_output_over_its_projections(ctx, torch_gpu, t, past):
    """The output written densely over the [q | k | v] records that the step
    reads: the values of a step whose output lies elsewhere."""
    torch = torch_gpu
    d, Hq, Hkv, B = 64, 14, 2, 2
    print(f"output over the projections type={t} past={past}", flush=True)
    rng = np.random.default_rng(past)
    y0 = to_gpu(torch, rng.standard_normal((B, 1, (Hq + 2 * Hkv) * d)), vva.F32)
    pos = torch.full((1,), past, dtype=torch.int32, device="cuda")
    outs = []
    for over in (False, True):
        y = y0.clone()
        q, k, v = (x.view(B, 1, -1, d) for x in (y[..., :Hq * d], y[..., Hq * d:-Hkv * d], y[..., -Hkv * d:]))
        kv = vva.KVCache(ctx, 1, Hkv, d, past + 1, B, t)
        fill_cache(kv, [past] * B, seed=3)
        out = y.view(-1)[:B * Hq * d].view(B, 1, Hq, d) if over else torch.empty((B, 1, Hq, d), device="cuda")
        ctx.decode_step(kv, 0, q, k, v, pos, torch.empty((B, 1, Hq, d), device="cuda"), out, d ** -0.5)
        torch.cuda.synchronize()
        outs.append((as_f32(torch, out), [kv.download(0, s, past + 1) for s in range(B)]))
        kv.free()
    assert_close(outs[1][0], outs[0][0], *TOL[t], what="over the records")
    for a, b in zip(outs[0][1], outs[1][1]):
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
