// decode_step.hip — single-token attention over F32 / F16 / BF16 caches in one
// launch per layer (and a merge launch for long windows): the whole decode
// step (RoPE of q and k, the K/V append at len(seq_b), the attention over the
// len + 1 keys; src/qwen2.cpp:282-335 with one new token per sequence, the TTS
// CFG loop, src/vibevoice_tts.cpp:862-880, and the transcript loop,
// src/vibevoice_asr.cpp:760-800), or the attention alone for q already rotated
// (STEP = false).  Short windows (0.5B: 1 MB per layer, L2 / MALL resident)
// are a chain of latencies, long ones a stream of K and V from HBM; the layout
// serves both: every load of a chunk is in flight before any is used, and the
// chain from the arguments to the merge is short.
//
// Grid (n_splits, Hkv, B); 4 waves.  A chunk is 128 keys (F32: 64) of a
// sequence's window, 32 (16) per wave; workgroup (s, h, b) takes chunks s,
// s + n_splits, ... for the G <= 8 query heads of kv head h.  Its K and V bytes
// in flight, 64 KB at d = 128, and three workgroups per CU keep the memory
// busy without a ring: the next chunk's K goes out as soon as the scores have
// consumed this one's registers, V as soon as it is in LDS.
//   0. every kernel argument is read in one batch (each scalar-cache miss is
//      a round trip, and that cache starts cold at every launch), then every
//      global load is issued before any is used: q and the new k / v rows as
//      raw 32-bit words, the wave's K rows as MFMA operands, its V rows;
//   1. the angle table of the token's position (the fp32 theta recurrence of
//      rope_append.hip) while the loads fly; RoPE(q), rounded to the cache
//      type (ggml's flash attention casts Q to K's type; F32 stays F32);
//      split 0 writes q_out;
//   2. the split holding key len(seq_b) rotates k and writes the new K and V
//      rows to the cache and, in place of the loaded ones, into its operands;
//   3. per wave and chunk: S^T = K Q^T (16 keys x 16 columns per MFMA, the G
//      heads as columns; K straight from memory, 64 contiguous bytes of a row
//      per four lanes), online softmax per head (fp32, exp2 domain), O^T +=
//      V^T P^T.  16-bit types: v_mfma_f32_16x16x32, P^T converted in place
//      from S^T as f16, V^T read from the wave's LDS V tile with the
//      transposing load.  F32: v_mfma_f32_16x16x4f32, products and sums in
//      fp32, V straight from memory;
//   4. the waves' (max, sum, O) are combined in LDS; with one split that is
//      the output, otherwise the workgroup writes (max, sum, acc).  Up to
//      kInLaunchMerge splits: agent-scope stores (coherent across XCDs without
//      an L2 write-back), a ticket, and the last workgroup of (b, h) merges
//      the splits with one batch of agent-scope loads per 16 and resets the
//      ticket for the next call.  More splits: plain stores, and
//      decode_merge_kernel (one CU would read the partials serially).
// Bound by the chain of latencies up to ~2k keys, by the stream beyond (a
// chunk's opening, ~3.5 us, and the merge, 4 us with its launch, are the
// rest).  Measured per step and layer (us; before: one 32 x 32-tile chunk per
// workgroup for 16-bit windows up to 8192 keys, three launches beyond, and
// rope_append + one workgroup per token and kv head for F32 caches):
//   0.5B, 2 x 1025 keys, F16        7.1 ->  6.8
//   7B, 1001 keys, F16             10.6 ->  9.6
//   7B, 20012 keys, F16            29.6 -> 15.1   (41 MB: 2.7 TB/s)
//   1.5B, 4097 + 3073 keys, F32     228 -> 10.9   (14.7 MB)
#include "vva_internal.hpp"

namespace vva {

namespace {

#include "wave_ops.hpp"
#include "mfma_ops.hpp"

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kStepWaves = 4;
constexpr int kMaxG = 8;                 // query heads per kv head
// Splits merged by the last workgroup: 9 splits (0.5B, 1k keys) take 7.1 us
// that way against 8.0 with the merge kernel, 24 (7B, 2 x 3k keys) 14.4
// against 10.7, 16 (7B, 2k) 9.9 against 10.2.
constexpr int kInLaunchMerge = 16;
constexpr int kStepWgsPerCu = 3;         // workgroups resident per CU (LDS and registers)
// Workgroups per CU that a long window is split for: each split adds partials
// for the merge to read (7B, 20k F16 keys: 16.9 us at 3, 15.1 at 2, 15.6 at 1;
// 4 x 32k: 55.7, 55.3, 54.1; 16k F32: 19.1, 19.1, 18.7).
constexpr int kPlanWgsPerCu = 2;

// Barrier for LDS hand-offs only: unlike __syncthreads it does not wait for
// the wave's outstanding global loads and stores.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");
}

// Element i of a row held as raw 32-bit words (F32, or F16 / BF16 pairs).
__device__ __forceinline__ float raw_elem(const uint32_t* row, int i, int type) {
    if (type == VVA_TYPE_F32) return __uint_as_float(row[i]);
    const uint32_t w = row[i >> 1];
    const uint16_t x = (uint16_t)(i & 1 ? w >> 16 : w);
    return type == VVA_TYPE_F16 ? f16_to_f32(x) : bf16_to_f32(x);
}

// Four floats of an output row on an 8-byte boundary at least.
__device__ __forceinline__ void store_out(char* p, const float4& v) {
    *(float2*)p = make_float2(v.x, v.y);
    *(float2*)(p + 8) = make_float2(v.z, v.w);
}

// The cache types: stored element, value -> stored element, keys per wave and chunk
template <int KT> struct Cell {
    typedef uint16_t elem;
    static constexpr int keys = 32;
    static __device__ __forceinline__ elem cvt(float x) { return KT == VVA_TYPE_F16 ? f32_to_f16(x) : f32_to_bf16(x); }
};
template <> struct Cell<VVA_TYPE_F32> {
    typedef float elem;
    static constexpr int keys = 16;
    static __device__ __forceinline__ elem cvt(float x) { return x; }
};

template <int KT>
__device__ __forceinline__ f32x4 mma16(const u32x4& a, const u32x4& b, const f32x4& c) {
    if constexpr (KT == VVA_TYPE_BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_vec<b8>(a), as_vec<b8>(b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(as_vec<h8>(a), as_vec<h8>(b), c, 0, 0, 0);
}

template <int D, int KT, bool STEP>
__global__ void __launch_bounds__(64 * kStepWaves) __attribute__((amdgpu_waves_per_eu(KT == VVA_TYPE_F32 && D == 128 ? 2 : kStepWgsPerCu)))
decode_step_kernel(StepArgs a) {
    using C = Cell<KT>;
    using E = typename C::elem;
    constexpr bool F32 = KT == VVA_TYPE_F32;
    constexpr int P = D / 2;
    constexpr int KW = C::keys, KC = KW * kStepWaves;    // keys per wave / workgroup and chunk
    constexpr int RB = D * (int)sizeof(E);               // bytes of a head row
    constexpr int NK = RB / 64;                          // 16-byte K loads per lane and 16 keys
    constexpr int KTL = KW / 16;                         // 16-key score tiles
    constexpr int CPR = RB / 16;                         // 16-byte chunks per V head row
    constexpr int NV = KW * CPR / 64;                    // V loads per lane
    constexpr int OT = D / 16;                           // 16-dim output tiles
    constexpr int VP = RB + 32;                          // V tile row pitch: the 8 rows of two lane groups on distinct banks
    constexpr int NQW = kMaxG * D / 256;                 // q words per thread at most (F32 q)
    constexpr int VT_BYTES = F32 ? 0 : kStepWaves * KW * VP;
    constexpr int WO_BYTES = kStepWaves * kMaxG * D * 4;
    __shared__ float cs[P], sn[P];
    __shared__ uint32_t qraw[kMaxG * D], kraw[D], vraw[D];                 // raw input words
    __shared__ __attribute__((aligned(16))) E qh[kMaxG][D];                // RoPE(q), cache type
    __shared__ __attribute__((aligned(16))) E knew[D], vnew[D];            // the new rows
    // the waves' V tiles, then (after the last chunk) their outputs
    __shared__ __attribute__((aligned(16))) char tiles[VT_BYTES > WO_BYTES ? VT_BYTES : WO_BYTES];
    __shared__ float wm[kStepWaves][kMaxG], wl[kStepWaves][kMaxG];
    __shared__ int ticket;

    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c = lane & 15, g = lane >> 4;
    const int split = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
    const int n_splits = gridDim.x;

    // ---- 0. kernel arguments (one scalar round trip for all of them)
    prefetch_kernargs<sizeof(StepArgs)>();
    const int past = a.past[b], G = a.G, Hq = a.Hq;
    const int q_type = a.q_type, k_type = a.k_type, v_type = a.v_type, qo_type = a.q_out_type;
    const int64_t k_rb = a.k_nb_tok, v_rb = a.v_nb_tok, q_nb_h = a.q_nb_h, qo_nb_h = a.qo_nb_h, o_nb_h = a.o_nb_h;
    const char* const kch = a.kc[b] + h * a.k_nb_head;             // row 0 of head h
    const char* const vch = a.vc[b] + h * a.v_nb_head;
    const char* const qb = a.q + b * a.q_nb_b + (int64_t)h * G * q_nb_h;
    const char* const kn = a.k + b * a.k_nb_b + h * a.k_nb_h;
    const char* const vn = a.v + b * a.v_nb_b + h * a.v_nb_h;
    const int32_t* const posp = a.pos + b * a.pos_stride_b;
    const bool has_qo = a.q_out != nullptr;
    char* const qob = a.q_out + b * a.qo_nb_b + (int64_t)h * G * qo_nb_h;     // used only when has_qo
    char* const ob = (char*)a.out + b * a.o_nb_b + (int64_t)h * G * o_nb_h;
    float* const ws = a.ws;
    unsigned* const tk = a.tickets + b * a.Hkv + h;
    const float theta_scale = a.theta_scale, scale = a.scale;
    const size_t ml_off = (size_t)a.B * Hq * n_splits * D;       // (max, sum) pairs after the accumulators
    const int pos_i = STEP ? *posp : 0;

    const int L = past + 1;
    const int n_chunks = (L + KC - 1) / KC;
    const bool owns_new = STEP && split == (n_chunks - 1) % n_splits;
    // q: G head rows of raw words
    const int qwpr_sh = __builtin_ctz(D) - (q_type == VVA_TYPE_F32 ? 0 : 1);   // log2(words per row)
    const int nqw = G << qwpr_sh;
    uint32_t qw[NQW];
#pragma unroll
    for (int u = 0; u < NQW; ++u) {
        const int idx = tid + 256 * u;
        const int r = idx >> qwpr_sh, i = idx - (r << qwpr_sh);
        const bool ok = idx < nqw;
        qw[u] = ((const uint32_t*)(qb + (ok ? r : 0) * q_nb_h))[ok ? i : 0];
    }
    // the new k row (waves 0, 1) and v row (waves 2, 3): a wave-uniform choice
    const bool is_k = __builtin_amdgcn_readfirstlane(w) < 2;
    const int nwi = is_k ? tid : tid - 128;
    const bool nw_ok = nwi < (D >> ((is_k ? k_type : v_type) == VVA_TYPE_F32 ? 0 : 1));
    uint32_t nw = 0;
    if (owns_new) {
        if (is_k) nw = ((const uint32_t*)kn)[nw_ok ? nwi : 0];
        else      nw = ((const uint32_t*)vn)[nw_ok ? nwi : 0];
    }
    // K of a chunk: tile kt, lane (c, g) holds key kb + 16 kt + c, bytes 64 j +
    // 16 g .. + 15 of its row in load j (keys past the window read row 0 and
    // are masked).  V: 16-bit types as whole rows, chunk i = lane + 64 u being
    // row i / CPR, bytes 16 (i % CPR); F32: load (s, j) is row kb + 4 g + s,
    // bytes 256 j + 16 c.
    u32x4 kf[KTL][NK], vf[NV];
    auto load_k = [&](int kb) {
#pragma unroll
        for (int kt = 0; kt < KTL; ++kt) {
            const int key = kb + 16 * kt + c;
            const char* kr = kch + (int64_t)(key < L ? key : 0) * k_rb + g * 16;
#pragma unroll
            for (int j = 0; j < NK; ++j) kf[kt][j] = *(const u32x4*)(kr + j * 64);
        }
    };
    auto load_v = [&](int kb) {
#pragma unroll
        for (int u = 0; u < NV; ++u) {
            const int row = F32 ? 4 * g + u / (D / 64) : (lane + 64 * u) / CPR;
            const int off = F32 ? 256 * (u % (D / 64)) + 16 * c : (lane + 64 * u) % CPR * 16;
            const int key = kb + row;
            vf[u] = *(const u32x4*)(vch + (int64_t)(key < L ? key : 0) * v_rb + off);
        }
    };
    int kb = split * KC + KW * w;                                  // the wave's first key
    load_k(kb);
    load_v(kb);

    // ---- 1. angle table; the raw q / k / v words to LDS
    if (STEP && tid < P) {
        const float th = rope_theta((float)pos_i, theta_scale, tid, P);
        cs[tid] = cosf(th);
        sn[tid] = sinf(th);
    }
#pragma unroll
    for (int u = 0; u < NQW; ++u)
        if (tid + 256 * u < nqw) qraw[tid + 256 * u] = qw[u];
    if (owns_new && nw_ok) (is_k ? kraw : vraw)[nwi] = nw;
    lds_barrier();
    // RoPE(q), rounded to the cache type for the scores
    for (int t = tid; t < G * P; t += 256) {
        const int r = t / P, i = t - r * P;
        const uint32_t* qrow = qraw + (r << qwpr_sh);
        const float x0 = raw_elem(qrow, i, q_type), x1 = raw_elem(qrow, i + P, q_type);
        if constexpr (STEP) {
            const float y0 = fmaf(x0, cs[i], -(x1 * sn[i])), y1 = fmaf(x0, sn[i], x1 * cs[i]);
            // the scores read what q_out holds: rounded to its type first
            qh[r][i] = C::cvt(round_to_type(y0, qo_type));
            qh[r][i + P] = C::cvt(round_to_type(y1, qo_type));
            if (split == 0 && has_qo) {
                const int64_t eo = type_elem_bytes(qo_type);
                char* dst = qob + r * qo_nb_h;
                store_elem(dst + i * eo, qo_type, y0);
                store_elem(dst + (i + P) * eo, qo_type, y1);
            }
        } else {
            qh[r][i] = C::cvt(x0);
            qh[r][i + P] = C::cvt(x1);
        }
    }
    // ---- 2. the new K / V row (the split holding key L - 1): to the cache,
    // and to knew / vnew (substituted into the operands)
    if (owns_new && tid < P) {
        const int i = tid;
        const float x0 = raw_elem(kraw, i, k_type), x1 = raw_elem(kraw, i + P, k_type);
        const float y0 = fmaf(x0, cs[i], -(x1 * sn[i])), y1 = fmaf(x0, sn[i], x1 * cs[i]);
        const E k0 = C::cvt(y0), k1 = C::cvt(y1);
        const E v0 = C::cvt(raw_elem(vraw, i, v_type)), v1 = C::cvt(raw_elem(vraw, i + P, v_type));
        knew[i] = k0;
        knew[i + P] = k1;
        vnew[i] = v0;
        vnew[i + P] = v1;
        E* krow = (E*)(kch + (int64_t)past * k_rb);
        E* vrow = (E*)(vch + (int64_t)past * v_rb);
        krow[i] = k0;
        krow[i + P] = k1;
        vrow[i] = v0;
        vrow[i + P] = v1;
    }
    lds_barrier();

    // ---- 3. the chunks.  Q^T as the B operand: lane (c, g) holds head c (0
    // past G), the bytes of each load j of K
    u32x4 qf[NK];
#pragma unroll
    for (int j = 0; j < NK; ++j) {
        const u32x4 u = *(const u32x4*)((const char*)qh[c < G ? c : 0] + j * 64 + g * 16);
        qf[j] = c < G ? u : u32x4{0u, 0u, 0u, 0u};
    }
    const float sl2 = scale * kLog2e;
    float m = -INFINITY, l = 0.0f;                 // head c: running max (log2 units) and sum of this lane's keys
    f32x4 o[OT];
#pragma unroll
    for (int t = 0; t < OT; ++t) o[t] = f32x4{};
    char* const vt = tiles + w * KW * VP;
    for (int ci = split; ci < n_chunks; ci += n_splits) {
        const bool more = ci + n_splits < n_chunks;
        const int kn_b = kb + n_splits * KC;       // the wave's first key of its next chunk
        if constexpr (!F32) {
            // V rows into the wave's tile: zeros past the window (their p is 0,
            // and 0 * inf would not be)
#pragma unroll
            for (int u = 0; u < NV; ++u) {
                const int i = lane + 64 * u, row = i / CPR, off = i % CPR * 16, key = kb + row;
                u32x4 x = key < L ? vf[u] : u32x4{0u, 0u, 0u, 0u};
                if (STEP && key == past) x = *(const u32x4*)((const char*)vnew + off);
                *(u32x4*)(vt + row * VP + off) = x;
            }
            wave_lds_sync();
            if (more) load_v(kn_b);
        }
        f32x4 st[KTL];
#pragma unroll
        for (int kt = 0; kt < KTL; ++kt) {
            if (STEP && kb + 16 * kt + c == past) {
#pragma unroll
                for (int j = 0; j < NK; ++j) kf[kt][j] = *(const u32x4*)((const char*)knew + j * 64 + g * 16);
            }
            st[kt] = f32x4{};
#pragma unroll
            for (int j = 0; j < NK; ++j) {
                if constexpr (F32) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        st[kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(kf[kt][j][e]),
                                                                      __uint_as_float(qf[j][e]), st[kt], 0, 0, 0);
                } else {
                    st[kt] = mma16<KT>(kf[kt][j], qf[j], st[kt]);
                }
            }
        }
        if (more) load_k(kn_b);
        // softmax: st[kt][r] is head c, key kb + 16 kt + 4 g + r
        float mr = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < KTL; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                mr = fmaxf(mr, kb + 16 * kt + 4 * g + r < L ? st[kt][r] * sl2 : -INFINITY);
        const float mn = fmaxf(m, max_swap32(max_swap16(mr)));
        const float nb = mn == -INFINITY ? 0.0f : -mn;
        const float alpha = __builtin_amdgcn_exp2f(m + nb);           // 0 while m = -inf
        m = mn;
        l *= alpha;
#pragma unroll
        for (int t = 0; t < OT; ++t) o[t] *= alpha;
        auto prob = [&](int kt, int r) {
            return kb + 16 * kt + 4 * g + r < L ? __builtin_amdgcn_exp2f(fmaf(st[kt][r], sl2, nb)) : 0.0f;
        };
        if constexpr (F32) {
            float p[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                p[r] = prob(0, r);
                l += p[r];
            }
            // step s: lane group g supplies key kb + 4 g + s; tile (j, e) row c is dim 64 j + 4 c + e
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int key = kb + 4 * g + s;
#pragma unroll
                for (int j = 0; j < D / 64; ++j) {
                    u32x4 x = key < L ? vf[s * (D / 64) + j] : u32x4{0u, 0u, 0u, 0u};
                    if (STEP && key == past) x = *(const u32x4*)((const char*)vnew + 256 * j + 16 * c);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        o[4 * j + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(x[e]), p[s], o[4 * j + e],
                                                                            0, 0, 0);
                }
            }
            if (more) load_v(kn_b);
        } else {
            h8 pf;
#pragma unroll
            for (int i = 0; i < 8; i += 2) {
                const float p0 = prob(i >> 2, i & 3), p1 = prob(i >> 2, (i & 3) + 1);
                const h2 pp = {(_Float16)p0, (_Float16)p1};
                pf[i] = pp.x;
                pf[i + 1] = pp.y;
                l = __builtin_amdgcn_fdot2(pp, h2{(_Float16)1.0f, (_Float16)1.0f}, l, false);
            }
            // P^T's 8 keys of lane group g: kb + 4 g + 0..3 and kb + 16 + 4 g + 0..3.  V^T: in
            // each 16-lane group, lane i points at row 4 g + i / 4, dims 4 (i % 4) ..;
            // the transposing read gives it the 4 keys of dim i
            const lds_char* va = (const lds_char*)vt + (4 * g + (c >> 2)) * VP + (c & 3) * 8;
#pragma unroll
            for (int t = 0; t < OT; ++t) {
                const h8 vv = v_frag<KT>(va + t * 32, va + t * 32 + 16 * VP);
                o[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vv, pf, o[t], 0, 0, 0);
            }
            wave_lds_sync();                       // the next chunk rewrites the tile
        }
        kb = kn_b;
    }
    l = add_swap32(add_swap16(l));

    // ---- 4. the waves' (max, sum, O) combined in LDS.  o[t][r] is head c, dim
    // 16 t + 4 g + r; F32: dim 64 (t / 4) + 16 g + 4 r + t % 4
    float (*const wo)[kMaxG][D] = (float (*)[kMaxG][D])tiles;
    if constexpr (!F32) lds_barrier();                             // every wave is done with its V tile
    if (c < G) {
        if (g == 0) {
            wm[w][c] = m;
            wl[w][c] = l;
        }
        if constexpr (F32) {
#pragma unroll
            for (int j = 0; j < D / 64; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    *(float4*)&wo[w][c][64 * j + 16 * g + 4 * r] =
                        make_float4(o[4 * j][r], o[4 * j + 1][r], o[4 * j + 2][r], o[4 * j + 3][r]);
        } else {
#pragma unroll
            for (int t = 0; t < OT; ++t)
                *(float4*)&wo[w][c][16 * t + 4 * g] = make_float4(o[t][0], o[t][1], o[t][2], o[t][3]);
        }
    }
    lds_barrier();
    // thread t: head t / (D / 4), dims 4 (t % (D / 4)) .. + 3
    const bool in_launch = n_splits <= kInLaunchMerge;
    if (tid < G * (D / 4)) {
        const int r = tid / (D / 4), d0 = 4 * (tid - r * (D / 4));
        float M = -INFINITY;
#pragma unroll
        for (int v = 0; v < kStepWaves; ++v) M = fmaxf(M, wm[v][r]);
        const float Mb = M == -INFINITY ? 0.0f : M;
        float lt = 0.0f;
        float4 ot = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
        for (int v = 0; v < kStepWaves; ++v) {
            const float f = __builtin_amdgcn_exp2f(wm[v][r] - Mb);      // 0 for a wave with no key
            const float4 ov = *(const float4*)&wo[v][r][d0];
            lt = fmaf(wl[v][r], f, lt);
            ot.x = fmaf(ov.x, f, ot.x);
            ot.y = fmaf(ov.y, f, ot.y);
            ot.z = fmaf(ov.z, f, ot.z);
            ot.w = fmaf(ov.w, f, ot.w);
        }
        const size_t rowi = ((size_t)b * Hq + h * G + r) * n_splits + split;
        if (n_splits == 1) {
            const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
            store_out(ob + r * o_nb_h + d0 * 4, make_float4(ot.x * inv, ot.y * inv, ot.z * inv, ot.w * inv));
        } else if (in_launch) {
            store_coherent2(ws + rowi * D + d0, ot.x, ot.y);
            store_coherent2(ws + rowi * D + d0 + 2, ot.z, ot.w);
            if (d0 == 0) store_coherent2(ws + ml_off + rowi * 2, M, lt);
        } else {
            *(float4*)(ws + rowi * D + d0) = ot;
            if (d0 == 0) *(float2*)(ws + ml_off + rowi * 2) = make_float2(M, lt);
        }
    }
    if (n_splits == 1 || !in_launch) return;
    // every partial store of this workgroup has completed before its ticket
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) ticket = (int)__hip_atomic_fetch_add(tk, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    lds_barrier();
    if (ticket != n_splits - 1) return;
    // ---- the last workgroup of (b, h): log-sum-exp over the splits, every
    // split's (max, sum) and accumulators loaded in one batch; thread t takes
    // head t / (D / 4), dims 4 (t % (D / 4)) .. + 3, so G D / 4 <= 256 threads
    // do it in one pass (in two passes of pairs the second pass's loads cost
    // another round trip: 10.6 against 9.6 us per step at 7B heads, 1k keys)
    if (tid < G * (D / 4)) {
        const int r = tid / (D / 4), d0 = 4 * (tid - r * (D / 4));
        const size_t row0 = ((size_t)b * Hq + h * G + r) * n_splits;
        float2 ml[kInLaunchMerge], a0[kInLaunchMerge], a1[kInLaunchMerge];
#pragma unroll
        for (int e = 0; e < kInLaunchMerge; ++e) {
            const bool in = e < n_splits;
            const size_t ri = row0 + (in ? e : 0);
            ml[e] = load_coherent2(ws + ml_off + ri * 2);
            a0[e] = load_coherent2(ws + ri * D + d0);
            a1[e] = load_coherent2(ws + ri * D + d0 + 2);
            if (!in) ml[e] = make_float2(-INFINITY, 0.0f);
        }
        float M = -INFINITY;
#pragma unroll
        for (int e = 0; e < kInLaunchMerge; ++e) M = fmaxf(M, ml[e].x);
        const float base = M == -INFINITY ? 0.0f : M;
        float n0 = 0.0f, n1 = 0.0f, n2 = 0.0f, n3 = 0.0f, den = 0.0f;
#pragma unroll
        for (int e = 0; e < kInLaunchMerge; ++e) {
            const float f = __builtin_amdgcn_exp2f(ml[e].x - base);
            n0 = fmaf(a0[e].x, f, n0);
            n1 = fmaf(a0[e].y, f, n1);
            n2 = fmaf(a1[e].x, f, n2);
            n3 = fmaf(a1[e].y, f, n3);
            den = fmaf(ml[e].y, f, den);
        }
        // The weight 0 of a slot past the last split does not silence an infinite
        // sum: F32 caches, whose infinite V elements give infinity, then sum once
        // more over the splits alone.  (Selects on the 16 slots cost 0.16 us of
        // every step, branches among their loads 1.3, this 0.08.)
        if constexpr (F32) {
            if (__builtin_expect(__builtin_isnan((n0 + n1) + (n2 + n3)), 0)) {
                n0 = n1 = n2 = n3 = 0.0f;
                for (int e = 0; e < n_splits; ++e) {
                    const float f = __builtin_amdgcn_exp2f(load_coherent2(ws + ml_off + (row0 + e) * 2).x - base);
                    const float2 x = load_coherent2(ws + (row0 + e) * D + d0);
                    const float2 y = load_coherent2(ws + (row0 + e) * D + d0 + 2);
                    n0 = fmaf(x.x, f, n0);
                    n1 = fmaf(x.y, f, n1);
                    n2 = fmaf(y.x, f, n2);
                    n3 = fmaf(y.y, f, n3);
                }
            }
        }
        const float inv = den > 0.0f ? 1.0f / den : 0.0f;
        store_out(ob + r * o_nb_h + d0 * 4, make_float4(n0 * inv, n1 * inv, n2 * inv, n3 * inv));
    }
    if (tid == 0) __hip_atomic_store(tk, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace

bool decode_step_supported(const StepArgs& a) {
    if (a.cache_type != VVA_TYPE_F16 && a.cache_type != VVA_TYPE_BF16 && a.cache_type != VVA_TYPE_F32) return false;
    if (a.d != 64 && a.d != 128) return false;
    if (a.Hq % a.Hkv || a.Hq / a.Hkv > kMaxG) return false;
    if (a.B * a.Hkv > kMaxStepTickets) return false;
    // q, k and v are read as 32-bit words
    for (const int64_t x : {(int64_t)(uintptr_t)a.q, a.q_nb_h, a.q_nb_b, (int64_t)(uintptr_t)a.k, a.k_nb_h, a.k_nb_b,
                            (int64_t)(uintptr_t)a.v, a.v_nb_h, a.v_nb_b})
        if (x % 4) return false;
    // cache rows as 16-byte vectors
    for (int b = 0; b < a.B; ++b)
        if ((uintptr_t)a.kc[b] % 16 || (uintptr_t)a.vc[b] % 16) return false;
    if (a.k_nb_tok % 16 || a.k_nb_head % 16 || a.v_nb_tok % 16 || a.v_nb_head % 16) return false;
    // the output as 16- or 8-byte vectors
    return (uintptr_t)a.out % 8 == 0 && a.o_nb_h % 8 == 0 && a.o_nb_b % 8 == 0;
}

// One chunk per workgroup up to kPlanWgsPerCu workgroups per CU (every byte
// of the window in flight), equal shares of the chunks beyond that.
int decode_step_splits(const StepArgs& a, int n_cu, int wgs) {
    const int kc = (a.cache_type == VVA_TYPE_F32 ? Cell<VVA_TYPE_F32>::keys : Cell<VVA_TYPE_F16>::keys) * kStepWaves;
    int Lmax = 1;
    for (int b = 0; b < a.B; ++b) Lmax = max(Lmax, a.past[b] + 1);
    const int chunks = (Lmax + kc - 1) / kc;
    int most = max(1, (wgs > 0 ? wgs : n_cu * kPlanWgsPerCu) / (a.B * a.Hkv));
    // decode_merge_kernel writes 16-byte aligned rows only
    if ((uintptr_t)a.out % 16 || a.o_nb_h % 16 || a.o_nb_b % 16) most = min(most, kInLaunchMerge);
    const int per = (chunks + most - 1) / most;
    return (chunks + per - 1) / per;
}
size_t decode_step_ws_bytes(const StepArgs& a, int n_splits) {
    return n_splits > 1 ? (size_t)n_splits * a.B * a.Hq * (a.d + 2) * sizeof(float) : 0;
}

namespace {

template <bool STEP>
hipError_t launch_step(const StepArgs& a, int n_splits, hipStream_t s) {
    const dim3 grid(n_splits, a.Hkv, a.B), block(64 * kStepWaves);
#define VVA_STEP(D, KT) hipLaunchKernelGGL((decode_step_kernel<D, KT, STEP>), grid, block, 0, s, a)
    switch (a.cache_type) {
        case VVA_TYPE_F32:
            if (a.d == 64) VVA_STEP(64, VVA_TYPE_F32); else VVA_STEP(128, VVA_TYPE_F32);
            break;
        case VVA_TYPE_BF16:
            if (a.d == 64) VVA_STEP(64, VVA_TYPE_BF16); else VVA_STEP(128, VVA_TYPE_BF16);
            break;
        default:
            if (a.d == 64) VVA_STEP(64, VVA_TYPE_F16); else VVA_STEP(128, VVA_TYPE_F16);
    }
#undef VVA_STEP
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || n_splits <= kInLaunchMerge) return e;
    AttnArgs m{};
    m.out = a.out; m.o_nb_h = a.o_nb_h; m.o_nb_b = a.o_nb_b;
    m.d = a.d; m.Hq = a.Hq; m.Hkv = a.Hkv; m.T = 1; m.B = a.B;
    return launch_decode_merge(m, a.ws, n_splits, s, a.cache_type == VVA_TYPE_F32);
}

}  // namespace

hipError_t launch_decode_step(const StepArgs& a, int n_splits, hipStream_t s) {
    return launch_step<true>(a, n_splits, s);
}
hipError_t launch_decode_attn(const StepArgs& a, int n_splits, hipStream_t s) {
    return launch_step<false>(a, n_splits, s);
}

}  // namespace vva
