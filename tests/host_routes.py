"""Routes of the C ABI on the CPU (a child program of test_host_routes.py, not
a test module): libvva.so over a stand-in of the HIP runtime
(tests/cpp/fake_hip.cpp) that records kernel launches and allocations instead
of making them.  `python host_routes.py NAME` runs the scenario NAME; its
assertions set the exit status.  Device pointers are made up: the host code
never reads them."""
import ctypes
import os
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(os.path.dirname(HERE), "vibevoice.cpp_amd"))
FAKE = ctypes.CDLL(os.path.join(HERE, "cpp", "bin", "libfakehip.so"), mode=ctypes.RTLD_GLOBAL)
FAKE.fake_take_log.restype = ctypes.c_char_p
FAKE.fake_set.argtypes = [ctypes.c_int, ctypes.c_size_t]

import vva  # noqa: E402 — after the stand-in

LIB = vva.load_library()
ES = {vva.F32: 4, vva.F16: 2, vva.BF16: 2, vva.I32: 4, vva.Q8_0: 34}
NO_LIMIT = 1 << 40
ref = ctypes.byref


def row_bytes(t, n):
    return n // 32 * 34 if t == vva.Q8_0 else n * ES[t]


class Host:
    """A fresh context over the stand-in; tensors at made-up addresses."""

    def __init__(self):
        self.h = ctypes.c_void_p()
        FAKE.fake_set(0, NO_LIMIT)
        assert LIB.vva_create(0, None, ref(self.h)) == vva.OK
        self.next = 1 << 45
        FAKE.fake_take_log()

    def kv(self, Hkv, d, max_seq, n_seq, t, lens):
        h = ctypes.c_void_p()
        assert LIB.vva_kv_create(self.h, ref(vva.KVDesc(1, Hkv, d, max_seq, n_seq, t)), ref(h)) == vva.OK
        for s, n in enumerate(lens):
            assert LIB.vva_kv_set_len(h, s, n) == vva.OK
        FAKE.fake_take_log()
        return h

    def tensor(self, t, ne, nb=None, data=None, off=0):
        """ne as ggml's; dense unless nb; at a fresh 4 KiB boundary + off unless data."""
        ne = list(ne) + [1] * (4 - len(ne))
        if nb is None:
            nb = [ES[t], row_bytes(t, ne[0])]
            nb += [nb[1] * ne[1], nb[1] * ne[1] * ne[2]]
        if data is None:
            data = self.next
            self.next += (sum(n * b for n, b in zip(ne[1:], nb[1:])) + 8191) // 4096 * 4096
        x = vva.Tensor()
        x.data, x.type = data + off, t
        for i in range(4):
            x.ne[i], x.nb[i] = ne[i], nb[i]
        return x

    def call(self, fn, *args, capturing=False, malloc_max=NO_LIMIT):
        """Status, names of the kernels launched, allocations made."""
        FAKE.fake_set(int(capturing), malloc_max)
        st = getattr(LIB, fn)(self.h, *args)
        FAKE.fake_set(0, NO_LIMIT)
        log = FAKE.fake_take_log().decode().splitlines()
        self.grids = [ln.split(" grid ")[1] for ln in log if ln.startswith("kernel ")]
        return (st, [ln.split(" grid ")[0][len("kernel "):] for ln in log if ln.startswith("kernel ")],
                [int(ln.split()[1]) for ln in log if ln.startswith("malloc ")])

    def err(self):
        return LIB.vva_last_error(self.h).decode()


def bf16_v_window():
    """A BF16 V window whose f16 copy [L][Hkv][d] would leave the prefill
    kernel's 32-bit range (2^30 bytes) although the caller's head-major rows,
    2 d bytes apart, do not: the kernel then converts as it reads."""
    d, T = 128, 2000
    for Hkv, L, converts in ((4, 4000, True), (64, 65536 - 65, True), (64, 65536 - 64, False), (64, 262145, False)):
        c = Host()
        nb = [2, 2 * d, 2 * d * L, 2 * d * L * Hkv]                   # ne = [d, L, Hkv, 1]
        k, v = c.tensor(vva.BF16, [d, L, Hkv], nb), c.tensor(vva.BF16, [d, L, Hkv], nb)
        q = c.tensor(vva.F32, [d, T, Hkv])
        out = c.tensor(vva.F32, [d, Hkv, T])
        st, kernels, _ = c.call("vva_flash_attn_ext", ref(q), ref(k), ref(v), None, d ** -0.5, 0.0, 0.0, ref(out))
        assert st == vva.OK, c.err()
        print(Hkv, L, kernels)
        assert ("window_bf16_v_kernel" in kernels) == converts
        want = f"prefill_kernel<{d}, {vva.BF16}, {vva.F16 if converts else vva.BF16}, false>"
        assert want in kernels, want


def one_token_call(t, Hkv, Hq, d, L, q_off=0, out_off=0, B=1):
    """vva_attn of one token over L keys: the kernels it takes."""
    c = Host()
    kv = c.kv(Hkv, d, L, B, t, [L - 1] * B)
    q, out = c.tensor(vva.F32, [d, Hq, 1, B], off=q_off), c.tensor(vva.F32, [d, Hq, 1, B], off=out_off)
    st, kernels, _ = c.call("vva_attn", kv, 0, ref(q), None, None, d ** -0.5, ref(out))
    assert st == vva.OK, c.err()
    return kernels


def step_call(t, Hkv, Hq, d, L, qo_off=0, out_off=0, B=1, q_out=None, out=None, host=None, **kw):
    """vva_decode_step to L keys: status and the kernels it takes.  q_out and
    out: functions of (host, q, k, v) giving other tensors."""
    c = host or Host()
    kv = c.kv(Hkv, d, L, B, t, [L - 1] * B)
    q, k, v = (c.tensor(vva.F32, [d, h, 1, B]) for h in (Hq, Hkv, Hkv))
    pos = c.tensor(vva.I32, [1])
    qo = q_out(c, q, k, v) if q_out else c.tensor(vva.F32, [d, Hq, 1, B], off=qo_off)
    o = out(c, q, k, v, qo) if out else c.tensor(vva.F32, [d, Hq, 1, B], off=out_off)
    st, kernels, mallocs = c.call("vva_decode_step", kv, 0, ref(q), ref(k), ref(v), ref(pos), None, 1e6, d ** -0.5,
                                  ref(qo), ref(o), **kw)
    return st, kernels, mallocs


def one_token_precision():
    """One-token attention over 16-bit caches: f16 probabilities (and f16 V for
    BF16 caches) only for the calls that decode_kernel has always taken with
    them; other head counts and unaligned rows keep the fp32 row kernel, in
    vva_attn and in steps beyond 8192 keys.  F32 caches are fp32 throughout."""
    def name(kernels):
        assert len(kernels) == 1 or kernels[1].startswith("decode_merge_kernel"), kernels
        return kernels[0].split("<")[0]
    for d in (64, 128):
        for t in (vva.F16, vva.BF16, vva.F32):
            for Hkv, G in ((1, 8), (2, 7), (3, 2), (4, 1), (5, 1), (6, 4), (7, 1), (8, 2), (12, 2), (16, 1)):
                fp16 = t != vva.F32 and 8 % Hkv == 0
                want = "decode_step_kernel" if fp16 or t == vva.F32 else "attn_rows_kernel"
                got = name(one_token_call(t, Hkv, Hkv * G, d, 300))
                assert got == want, (d, t, Hkv, G, got)
                for L in (300, 8192):                             # short steps: every head count, as ever
                    st, kernels, _ = step_call(t, Hkv, Hkv * G, d, L)
                    assert st == vva.OK and name(kernels) == "decode_step_kernel", (d, t, Hkv, G, L, kernels)
                st, kernels, _ = step_call(t, Hkv, Hkv * G, d, 8193)
                assert st == vva.OK
                if want == "decode_step_kernel":
                    assert name(kernels) == want, (d, t, Hkv, G, kernels)
                else:
                    assert [k.split("<")[0] for k in kernels] == ["rope_append_vec_kernel", want], (d, t, Hkv, kernels)
            if t == vva.F32:
                continue
            # rows of q or out that are not 16-byte aligned
            for off in ((4, 0), (8, 0), (0, 4)):
                assert name(one_token_call(t, 2, 14, d, 300, *off)) == "attn_rows_kernel", (d, t, off)
            st, kernels, _ = step_call(t, 2, 14, d, 9000, qo_off=8)
            assert st == vva.OK and kernels[1].split("<")[0] == "attn_rows_kernel", kernels


def proj_call(mode, wt, heads, N, T=None, xt=vva.F32, cache=vva.F16, host=None, stride=0, **kw):
    """vva_qkv_rope_append ("qkv") or vva_out_proj_residual ("out") of N token
    rows: status, kernels, allocations.  stride: bytes of a weight row, if not dense."""
    c = host or Host()
    d, Hq, Hkv, hidden = heads
    T = T or N
    B = N // T
    def weight(M, K):
        return c.tensor(wt, [K, M], [ES[wt], stride, stride * M, stride * M] if stride else None)
    if mode == "out":
        o, x, h = c.tensor(xt, [Hq * d, T, B]), c.tensor(vva.F32, [hidden, T, B]), c.tensor(vva.F32, [hidden, T, B])
        return c.call("vva_out_proj_residual", ref(o), ref(weight(hidden, Hq * d)), ref(x), ref(h), **kw)
    kv = c.kv(Hkv, d, T, B, cache, [0] * B)
    x, q = c.tensor(xt, [hidden, T, B]), c.tensor(vva.F32, [d, Hq, T, B])
    pos = c.tensor(vva.I32, [T])
    return c.call("vva_qkv_rope_append", kv, 0, ref(x), *(ref(weight(n * d, hidden)) for n in (Hq, Hkv, Hkv)), None,
                  None, None, ref(pos), None, 1e6, ref(q), **kw)


H05, H15, H7 = (64, 14, 2, 896), (128, 12, 2, 1536), (128, 28, 4, 3584)      # d, Hq, Hkv, hidden


def workspace_one_can_do_without():
    """Calls that use the workspace only to be faster run without it where it
    cannot grow: under capture on a fresh context, or on a full device."""
    for kw in ({"capturing": True}, {"malloc_max": 1 << 19}):
        # a BF16 prefill converts V as it reads
        c = Host()
        kv = c.kv(4, 128, 16384, 1, vva.BF16, [0])
        q, out = c.tensor(vva.BF16, [128, 28, 16384]), c.tensor(vva.F32, [128, 28, 16384])
        args = (kv, 0, ref(q), None, None, 0.1, ref(out))
        st, kernels, mallocs = c.call("vva_attn", *args, **kw)
        assert st == vva.OK and not mallocs, c.err()
        assert kernels == [f"prefill_kernel<128, {vva.BF16}, {vva.BF16}, false>"], kernels
        st, kernels, mallocs = c.call("vva_attn", *args)
        assert st == vva.OK and kernels[0] == "window_bf16_v_kernel" and mallocs, kernels
        # 4 to 8 rows of F16 weights: the GEMV instead of the GEMM (the q/k/v
        # call's GEMV itself needs the first megabyte)
        for mode in ("qkv", "out"):
            for N in (4, 8):
                c = Host()
                if mode == "qkv":
                    assert proj_call(mode, vva.F16, H7, 3, host=c)[2] == [1 << 20]
                st, kernels, mallocs = proj_call(mode, vva.F16, H7, N, host=c, **kw)
                assert st == vva.OK and not mallocs and kernels[0].startswith("proj_gemv_"), (kernels, mallocs, c.err())
                st, kernels, _ = proj_call(mode, vva.F16, H7, N, host=c)
                assert st == vva.OK and kernels[-1].startswith("proj_gemm_kernel"), kernels
    # what cannot do without says so, and the next call is none the worse
    c = Host()
    kv = c.kv(4, 128, 2048, 1, vva.F16, [2047])
    q, out = c.tensor(vva.F32, [128, 28]), c.tensor(vva.F32, [128, 28])
    for kw, want in (({"malloc_max": 1 << 19}, vva.ERR_OOM), ({"capturing": True}, vva.ERR_INVALID_ARG), ({}, vva.OK)):
        st, kernels, _ = c.call("vva_attn", kv, 0, ref(q), None, None, 0.1, ref(out), **kw)
        assert st == want and bool(kernels) == (want == vva.OK), (st, want, c.err())


def f32_step_without_workspace():
    """One-token calls on an F32 cache are accepted wherever their split
    partials cannot be held, with fewer splits; a 16-bit cache's are refused
    there, as they always were."""
    d, Hq, Hkv, B = 128, 28, 4, 2
    per_split = B * Hq * (d + 2) * 4
    for kw, refusal in (({"capturing": True}, vva.ERR_INVALID_ARG), ({"malloc_max": 1 << 21}, vva.ERR_OOM)):
        for warm in (0, 300):                                     # keys of an earlier call: 0, none
            for L in (64, 65, 4097, 32768):
                c = Host()
                if warm:
                    assert step_call(vva.F32, Hkv, Hq, d, warm, B=B, host=c)[2] == [1 << 20]
                st, kernels, mallocs = step_call(vva.F32, Hkv, Hq, d, L, B=B, host=c, **kw)
                assert st == vva.OK, (kw, L, c.err())
                n = LIB.vva_last_decode_splits(c.h)
                assert kernels[0].startswith("decode_step_kernel") and c.grids[0] == f"{n},{Hkv},{B}"
                have = max([1 << 20 if warm else 0] + mallocs)
                chunks, most = -(-L // 64), 512 // (Hkv * B)      # 64 keys a chunk, 512 workgroups
                want = -(-chunks // -(-chunks // most))
                assert n == max(1, min(want, have // per_split)), (n, want, have)
                # vva_attn alone, the same workspace
                c = Host()
                if warm:
                    step_call(vva.F32, Hkv, Hq, d, warm, B=B, host=c)
                kv = c.kv(Hkv, d, L, B, vva.F32, [L - 1] * B)
                q, out = c.tensor(vva.F32, [d, Hq, 1, B]), c.tensor(vva.F32, [d, Hq, 1, B])
                assert c.call("vva_attn", kv, 0, ref(q), None, None, 0.1, ref(out), **kw)[0] == vva.OK, c.err()
                assert LIB.vva_last_decode_splits(c.h) == n
        assert step_call(vva.F16, Hkv, Hq, d, 8192, B=B, **kw)[0] == (refusal if "capturing" in kw else vva.OK)
    # the static scratch: splits forced beyond it
    for t, want in ((vva.F32, vva.OK), (vva.F16, vva.ERR_INVALID_ARG)):
        c = Host()
        assert LIB.vva_set_schedule(c.h, 1 << 20, 0, 0) == vva.OK
        kv = c.kv(Hkv, d, 65536, 16, t, [65535] * 16)
        q, out = c.tensor(vva.F32, [d, Hq, 1, 16]), c.tensor(vva.F32, [d, Hq, 1, 16])
        st, kernels, _ = c.call("vva_attn_noalloc", kv, 0, ref(q), None, None, 0.1, ref(out))
        assert st == want and bool(kernels) == (want == vva.OK), (t, st, c.err())
        if want == vva.OK:
            n = LIB.vva_last_decode_splits(c.h)
            assert n * 16 * Hq * (d + 2) * 4 <= 36 << 20 < (n + 1) * 16 * Hq * (d + 2) * 4


def step_output_alignment():
    """Output rows on 8-byte boundaries stay in the one-launch step, merged in
    the launch (decode_merge_kernel writes 16-byte aligned rows); 4-byte ones
    take the two calls."""
    for t in (vva.F32, vva.F16, vva.BF16):
        for L, off, one in ((1000, 8, True), (8192, 8, True), (1000, 4, False)):
            st, kernels, _ = step_call(t, 4, 28, 128, L, out_off=off)
            assert st == vva.OK and ("decode_step_kernel" in kernels[0]) == one and (len(kernels) == 1) == one, kernels
    st, kernels, _ = step_call(vva.F16, 4, 28, 128, 8192)
    assert kernels[1].startswith("decode_merge_kernel")


def output_over_inputs():
    """A step's output rows laid over its inputs: q itself in one launch, any
    other overlap as the two calls (whose attention starts when the inputs have
    been read); rows of several sequences side by side do not overlap."""
    d, Hq, Hkv, B = 64, 14, 2, 2
    row = (Hq + 2 * Hkv) * d * 4                                   # [q | k | v] of a sequence
    for t in (vva.F32, vva.F16):
        for L in (300, 9000):
            def step(out, q_out=None):
                st, kernels, _ = step_call(t, Hkv, Hq, d, L, B=B, q_out=q_out, out=out)
                assert st == vva.OK
                return kernels[0].split("<")[0]
            at = lambda c, x, off=0, nb=None: c.tensor(vva.F32, [d, Hq, 1, B], nb, data=x.data + off)    # noqa: E731
            one, two = "decode_step_kernel", "rope_append_vec_kernel"
            assert step(lambda c, q, k, v, qo: at(c, q)) == one
            assert step(lambda c, q, k, v, qo: at(c, qo)) == two
            assert step(lambda c, q, k, v, qo: at(c, k)) == two
            assert step(lambda c, q, k, v, qo: at(c, v, -d * 4)) == two
            assert step(lambda c, q, k, v, qo: at(c, q, d * 4)) == two
            assert step(lambda c, q, k, v, qo: at(c, q, 0, [4, d * 4, d * Hq * 4, row])) == two
            # q_out and out side by side in each sequence's record
            nb = [4, d * 4, 2 * d * Hq * 4, 2 * d * Hq * 4]
            assert step(lambda c, q, k, v, qo: at(c, qo, d * Hq * 4, nb),
                        lambda c, q, k, v: c.tensor(vva.F32, [d, Hq, 1, B], nb)) == one
            # vva_attn: out over a [q | k | v] record's q, dense and at the record's stride
            c = Host()
            kv = c.kv(Hkv, d, L, B, t, [L - 1] * B)
            q = c.tensor(vva.F32, [d, Hq, 1, B], [4, d * 4, row, row])
            for nb, want in (([4, d * 4, row, row], "decode_step_kernel"),
                             (None, "decode_kernel" if t == vva.F16 else "attn_gqa_f32_kernel")):
                out = c.tensor(vva.F32, [d, Hq, 1, B], nb, data=q.data)
                st, kernels, _ = c.call("vva_attn", kv, 0, ref(q), None, None, 0.1, ref(out))
                assert st == vva.OK and kernels[0].split("<")[0] == want, kernels


def rope_of_few_rows():
    """Fewer than 80 rows of 64-dim heads into a Q8_0 cache take the scalar
    kernel, other calls of aligned rows the vector one."""
    for d, Hq, Hkv in ((64, 14, 2), (128, 28, 4)):
        for t in (vva.F32, vva.F16, vva.BF16, vva.Q8_0):
            for T, B in ((1, 1), (79, 1), (39, 2), (80, 1), (40, 2), (1100, 1)):
                c = Host()
                kv = c.kv(Hkv, d, T, B, t, [0] * B)
                q, k, v = (c.tensor(vva.F32, [d, h, T, B]) for h in (Hq, Hkv, Hkv))
                qo, pos = c.tensor(vva.F32, [d, Hq, T, B]), c.tensor(vva.I32, [T])
                st, kernels, _ = c.call("vva_rope_append", kv, 0, ref(q), ref(k), ref(v), ref(pos), None, 1e6, ref(qo))
                scalar = d == 64 and t == vva.Q8_0 and T * B < 80
                assert st == vva.OK and kernels[0].split("<")[0] == ("rope_append_kernel" if scalar else
                                                                     "rope_append_vec_kernel"), (d, t, T, B, kernels)


def gemm_of(kernels, grids):
    """(kernel, tile rows, tile columns, workgroups, dequantized weights)"""
    i = next(i for i, k in enumerate(kernels) if "gemm" in k)
    k, wgs = kernels[i], int(grids[i].split(",")[0])
    name = k.split("<")[0][len("proj_gemm_"):]
    a = k.split("<")[1].rstrip(">").split(", ")
    tm, tn = (int(a[2]), int(a[3])) if name == "kernel" else (256, 128) if name.startswith("wide") else (256, 256)
    return name.split("_")[0], tm, tn, wgs, "vva::proj_dequant_q8_kernel" in kernels


def projection_plans():
    """The GEMM's plan over shapes: the tiles cover the rows, a tile of
    proj_gemm_kernel lies in one matrix, its pieces are resident at once and
    within the tickets, dequantized weights meet an F16 kernel of whole 256
    rows; and matrices past the reach of the wide and the big kernel's offsets
    stay with the small tiles."""
    for heads in (H05, H15, H7, (128, 8, 8, 1024), (64, 2, 2, 64)):
        d, Hq, Hkv, hidden = heads
        for wt in (vva.F16, vva.Q8_0):
            for mode, rows, K in (("qkv", [Hq * d, Hkv * d], hidden), ("out", [hidden], Hq * d)):
                if any(r % 128 for r in rows):
                    continue
                M = sum(rows) + (rows[1] if mode == "qkv" else 0)
                for N in [*range(9, 1100, 13), *range(1100, 9000, 171)]:
                    c = Host()
                    st, kernels, _ = proj_call(mode, wt, heads, N, host=c)
                    assert st == vva.OK, c.err()
                    name, tm, tn, wgs, dq = gemm_of(kernels, c.grids)
                    tiles = -(-M // tm) * -(-N // tn)
                    if name == "kernel":
                        ks = wgs // tiles
                        assert all(r % tm == 0 for r in rows) and wgs == tiles * ks and not dq
                        assert 1 <= ks <= 4 and (ks == 1 or (wgs <= 512 and tiles <= 1024 and K // 64 >= 4 * ks))
                    else:
                        assert wgs == tiles if name == "wide" else wgs >= tiles
                        assert (wt == vva.Q8_0) == dq and (not dq or N >= 1024)
    # 900 rows of the 7B q/k/v: one round of wide tiles, not 288 of 128 x 128
    c = Host()
    assert gemm_of(proj_call("qkv", vva.F16, H7, 900, host=c)[1], c.grids)[0] == "wide"
    # weight rows 8 MiB apart: more than 1 GiB of a matrix, 2 GiB of 256 rows
    for wt in (vva.F16, vva.Q8_0):
        for N in (1000, 3000):
            c = Host()
            st, kernels, _ = proj_call("qkv", wt, H7, N, host=c, stride=1 << 23)
            name, tm, *_ = gemm_of(kernels, c.grids)
            assert st == vva.OK and (tm < 256 or (wt == vva.Q8_0 and N >= 1024)), (wt, N, kernels)


def whole_row_windows():
    """vva_attn of one token over 16-bit caches: the register-streamed kernel
    for one query head per kv head over many long windows and for 8 heads of 64
    dims from HBM, the one-launch kernel for the rest (every model's heads)."""
    for d, Hkv, G, B, L, whole in ((64, 8, 1, 4, 1023, False), (64, 8, 1, 4, 1024, True), (64, 2, 1, 15, 4000, False),
                                   (128, 2, 1, 16, 4000, True), (128, 2, 1, 1, 32768, False), (64, 8, 4, 16, 4000, True),
                                   (64, 8, 4, 4, 8000, False), (64, 8, 8, 16, 4000, False), (64, 8, 8, 16, 8192, True),
                                   (128, 8, 8, 16, 16000, False), (64, 2, 7, 16, 32768, False),
                                   (128, 2, 6, 16, 32768, False), (128, 4, 7, 16, 32768, False)):
        for t in (vva.F16, vva.BF16, vva.F32):
            kernel = one_token_call(t, Hkv, Hkv * G, d, L, B=B)[0].split("<")[0]
            want = "decode_kernel" if whole and t != vva.F32 else "decode_step_kernel"
            assert kernel == want, (d, Hkv, G, B, L, t, kernel)


SCENARIOS = [bf16_v_window, one_token_precision, workspace_one_can_do_without, f32_step_without_workspace,
             step_output_alignment, output_over_inputs, rope_of_few_rows,
             projection_plans, whole_row_windows]

if __name__ == "__main__":
    {f.__name__: f for f in SCENARIOS}[sys.argv[1]]()
