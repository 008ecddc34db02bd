// rope_append.hip — fused NeoX RoPE of Q and K plus the KV-cache append.
//
// Replaces, in one launch, the four ggml ops the reference builds per layer
// (src/qwen2.cpp:282-306): ggml_rope_ext on q, ggml_rope_ext on k (NeoX,
// src/rope.hpp:14-15), and the two ggml_cpy's of k and v into the resident
// cache views at row past_len.  The cache may be F32 / F16 / BF16 / Q8_0; the
// rotated Q is written in the attention's input type.
//
// rope_append_vec_kernel takes head dims 64 and 128 with aligned rows, every
// cache type; rope_append_kernel the rest, and few rows of 64-dim heads into a
// Q8_0 cache.
//
// rope_append_kernel: one workgroup per (token t, batch b), 256 threads.
// Threads 0..d/2-1 first build the angle table of the token in LDS with the
// fp32 recurrence ggml's CPU rope cache uses (theta_0 = pos, theta_{i+1} =
// theta_i * base^(-2/d)); then every thread takes rotation pairs
// (x[i], x[i+d/2]) of the Hq q heads, the Hkv k heads and the Hkv v heads
// ("slots").  With d/2 a multiple of 32, each aligned group of 32 threads
// holds exactly two Q8_0 blocks of one head (elements i and i + d/2), so the
// block amax is a 32-lane butterfly and the codes are written without LDS.
//
// Memory: HBM-bound elementwise pass; per token it reads Hq+2*Hkv source rows
// and writes Hq rows of Q plus one K and one V cache row.
#include "vva_internal.hpp"

namespace vva {

namespace {

#include "wave_ops.hpp"

__global__ void __launch_bounds__(256) rope_append_kernel(RopeAppendArgs a, int items_per_block) {
    prefetch_kernargs<sizeof(RopeAppendArgs)>();
    const int t = blockIdx.x, b = blockIdx.y;
    const int P = a.d >> 1;
    __shared__ float cs[128], sn[128];
    const float p = (float)a.pos[b * a.pos_stride_b + t];
    for (int i = threadIdx.x; i < P; i += blockDim.x) {
        const float th = rope_theta(p, a.theta_scale, i, P);
        cs[i] = cosf(th);
        sn[i] = sinf(th);
    }
    __syncthreads();

    const int nq = a.do_q ? a.Hq : 0;
    const int nslots = nq + (a.do_kv ? 2 * a.Hkv : 0);
    // blockIdx.z takes a multiple-of-256 slice of the token's items, so few-token
    // calls (decode) still spread over many workgroups
    const int w_begin = blockIdx.z * items_per_block;
    const int total = min(nslots * P, w_begin + items_per_block);
    for (int w = w_begin + threadIdx.x; w < total; w += blockDim.x) {
        const int slot = w / P;
        const int i = w - slot * P;
        const float c = cs[i], s = sn[i];
        if (slot < nq) {
            const int64_t es = type_elem_bytes(a.q_type);
            const char* src = a.q + b * a.q_nb_b + t * a.q_nb_t + slot * a.q_nb_h;
            const float x0 = load_elem(src + i * es, a.q_type);
            const float x1 = load_elem(src + (i + P) * es, a.q_type);
            const float y0 = fmaf(x0, c, -(x1 * s));
            const float y1 = fmaf(x0, s, x1 * c);
            const int64_t eo = type_elem_bytes(a.q_out_type);
            char* dst = a.q_out + b * a.qo_nb_b + t * a.qo_nb_t + slot * a.qo_nb_h;
            store_elem(dst + i * eo, a.q_out_type, y0);
            store_elem(dst + (i + P) * eo, a.q_out_type, y1);
        } else {
            const int hs = slot - nq;
            const bool is_k = hs < a.Hkv;
            const int h = is_k ? hs : hs - a.Hkv;
            const int typ = is_k ? a.k_type : a.v_type;
            const int64_t es = type_elem_bytes(typ);
            const char* src = is_k ? a.k + b * a.k_nb_b + t * a.k_nb_t + h * a.k_nb_h
                                   : a.v + b * a.v_nb_b + t * a.v_nb_t + h * a.v_nb_h;
            const float x0 = load_elem(src + i * es, typ);
            const float x1 = load_elem(src + (i + P) * es, typ);
            float y0 = x0, y1 = x1;
            if (is_k) {
                y0 = fmaf(x0, c, -(x1 * s));
                y1 = fmaf(x0, s, x1 * c);
            }
            char* row = (is_k ? a.k_dst[b] : a.v_dst[b]) + t * a.cache_row_bytes + h * a.cache_head_bytes;
            if (a.cache_type == VVA_TYPE_Q8_0) {
                store_q8_pair(row, i, P, y0, y1);
            } else {
                const int64_t ec = type_elem_bytes(a.cache_type);
                store_elem(row + i * ec, a.cache_type, y0);
                store_elem(row + (i + P) * ec, a.cache_type, y1);
            }
        }
    }
}

// 8 consecutive elements (16-byte aligned): as loaded, as fp32, and stored.
struct Raw8 {
    uint4 a, b;                                       // b: F32 only
};
__device__ __forceinline__ Raw8 load_raw8(const char* p, int type) {
    Raw8 r;
    r.a = *(const uint4*)p;
    if (type == VVA_TYPE_F32) r.b = ((const uint4*)p)[1];
    return r;
}
__device__ __forceinline__ void raw8_to_f32(const Raw8& r, int type, float (&x)[8]) {
    const uint32_t w[8] = {r.a.x, r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w};
    if (type == VVA_TYPE_F32) {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = __uint_as_float(w[e]);
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint16_t lo = (uint16_t)(w[e] & 0xffffu), hi = (uint16_t)(w[e] >> 16);
        x[2 * e] = type == VVA_TYPE_F16 ? f16_to_f32(lo) : bf16_to_f32(lo);
        x[2 * e + 1] = type == VVA_TYPE_F16 ? f16_to_f32(hi) : bf16_to_f32(hi);
    }
}
__device__ __forceinline__ void store8(char* p, int type, const float (&y)[8]) {
    if (type == VVA_TYPE_F32) {
        ((float4*)p)[0] = make_float4(y[0], y[1], y[2], y[3]);
        ((float4*)p)[1] = make_float4(y[4], y[5], y[6], y[7]);
        return;
    }
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint16_t lo = type == VVA_TYPE_F16 ? f32_to_f16(y[2 * e]) : f32_to_bf16(y[2 * e]);
        const uint16_t hi = type == VVA_TYPE_F16 ? f32_to_f16(y[2 * e + 1]) : f32_to_bf16(y[2 * e + 1]);
        w[e] = (uint32_t)lo | ((uint32_t)hi << 16);
    }
    *(uint4*)p = make_uint4(w[0], w[1], w[2], w[3]);
}
// Elements i .. i + 7 of a Q8_0 row (i a multiple of 8): the 4 lanes of an
// aligned group hold a block, whose max they share by DPP; the arithmetic is
// store_q8_pair's, so the bytes are too.
__device__ __forceinline__ void store8_q8(char* row, int i, const float (&y)[8]) {
    float am = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) am = fmaxf(am, fabsf(y[e]));
    am = fmaxf(am, dpp<kDppXor1>(am));
    am = fmaxf(am, dpp<kDppXor2>(am));
    const float d = am / 127.0f;
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    char* blk = row + (i / kQK8) * kQ8Bytes;
    const int j = i & (kQK8 - 1);
    if (j == 0) *(uint16_t*)blk = f32_to_f16(d);
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        const uint8_t lo = (uint8_t)(int8_t)roundf(y[e] * id), hi = (uint8_t)(int8_t)roundf(y[e + 1] * id);
        *(uint16_t*)(blk + 2 + j + e) = (uint16_t)(lo | ((uint16_t)hi << 8));
    }
}

// The same pass for 16-byte aligned rows (Q8_0 caches: rows of whole 2-byte
// units), every cache type: a workgroup takes TOK tokens (blockIdx.z: a slice
// of their items), a lane 8 rotation pairs of a head row (16-byte loads and
// stores of elements i .. i + 7 and i + P .. i + P + 7).  HBM-bound for long
// calls, bound by its chain of latencies for short ones, so the first items'
// loads go out before the angles are computed, and each later item's loads
// before the one in hand is stored.  The angles: one lane per token runs the
// fp32 recurrence once, P products, into LDS (a chain per angle, all lanes
// selecting theirs, was P times that), then a thread per angle takes its sine
// or cosine.  Results are the scalar kernel's bit for bit.
// Measured, us per call, before (8 tokens per workgroup, a chain per angle;
// Q8_0 caches and calls under 64 rows on the scalar kernel) and now: 512
// tokens at 7B heads into Q8_0 13.6 -> 5.9, into F16 14.6 -> 6.1; 4096 tokens
// at 1.5B heads, BF16, 23.0 -> 11.0 (33 MB: 3.0 TB/s); 32768 at 7B heads into
// F16 144 -> 135 (604 MB: 4.5 TB/s); 4096 at 7B heads into Q8_0 39.7 -> 24.1.
// BF16 results then rounded in one instruction (f32_to_bf16; 8 layers' calls, 2
// of 32768, in a captured graph): 4096 at 1.5B heads 11.9 -> 11.0, 32768 at 7B
// heads, BF16 in and F16 cache, 131 -> 116 (604 MB: 5.2 TB/s), 4096 at 7B heads
// into Q8_0 25.2 -> 22.8, 2000 at 0.5B heads 6.8 -> 6.2.
template <int P, int TOK>
__global__ void __launch_bounds__(256) rope_append_vec_kernel(RopeAppendArgs a, int items_per_block) {
    prefetch_kernargs<sizeof(RopeAppendArgs)>();
    constexpr int C = P / 8;                          // 8-pair chunks per row
    const int t0 = blockIdx.x * TOK, b = blockIdx.y;
    const int nt = min(TOK, a.T - t0);
    __shared__ float th[TOK][P + 1];
    __shared__ __attribute__((aligned(16))) float cs[TOK][P], sn[TOK][P];

    const int nq = a.do_q ? a.Hq : 0;
    const int per_tok = (nq + (a.do_kv ? 2 * a.Hkv : 0)) * C;
    const int w_end = min(nt * per_tok, (int)(blockIdx.z + 1) * items_per_block);
    struct Item {
        Raw8 x0, x1;
        int tl, slot, i0, type;
    };
    auto fetch = [&](int w) {
        Item it;
        it.tl = w / per_tok;
        const int r = w - it.tl * per_tok;
        it.slot = r / C;
        it.i0 = (r - it.slot * C) * 8;
        const int t = t0 + it.tl, hs = it.slot - nq;
        const char* src;
        if (hs < 0) {
            it.type = a.q_type;
            src = a.q + b * a.q_nb_b + t * a.q_nb_t + it.slot * a.q_nb_h;
        } else if (hs < a.Hkv) {
            it.type = a.k_type;
            src = a.k + b * a.k_nb_b + t * a.k_nb_t + hs * a.k_nb_h;
        } else {
            it.type = a.v_type;
            src = a.v + b * a.v_nb_b + t * a.v_nb_t + (hs - a.Hkv) * a.v_nb_h;
        }
        const int es = it.type == VVA_TYPE_F32 ? 4 : 2;
        it.x0 = load_raw8(src + it.i0 * es, it.type);
        it.x1 = load_raw8(src + (it.i0 + P) * es, it.type);
        return it;
    };
    int w = blockIdx.z * items_per_block + threadIdx.x;
    Item cur{};
    if (w < w_end) cur = fetch(w);

    if (threadIdx.x < nt) {
        float x = (float)a.pos[b * a.pos_stride_b + t0 + threadIdx.x];
        for (int i = 0; i < P; ++i) {
            th[threadIdx.x][i] = x;
            x *= a.theta_scale;
        }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < nt * 2 * P; k += blockDim.x) {
        const int tl = k / (2 * P), i = k % P;
        const float x = th[tl][i];
        if (k % (2 * P) < P) cs[tl][i] = cosf(x);     // (whole waves at P = 64)
        else                 sn[tl][i] = sinf(x);
    }
    __syncthreads();

    for (; w < w_end; w += blockDim.x) {
        const Item it = cur;
        if (w + (int)blockDim.x < w_end) cur = fetch(w + blockDim.x);
        float x0[8], x1[8], y0[8], y1[8];
        raw8_to_f32(it.x0, it.type, x0);
        raw8_to_f32(it.x1, it.type, x1);
        const bool rot = it.slot < nq + a.Hkv;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float c = cs[it.tl][it.i0 + e], sv = sn[it.tl][it.i0 + e];
            y0[e] = rot ? fmaf(x0[e], c, -(x1[e] * sv)) : x0[e];
            y1[e] = rot ? fmaf(x0[e], sv, x1[e] * c) : x1[e];
        }
        const int t = t0 + it.tl, hs = it.slot - nq;
        char* dst;
        int type;
        if (hs < 0) {
            dst = a.q_out + b * a.qo_nb_b + t * a.qo_nb_t + it.slot * a.qo_nb_h;
            type = a.q_out_type;
        } else {
            dst = (hs < a.Hkv ? a.k_dst[b] : a.v_dst[b]) + t * a.cache_row_bytes +
                  (hs < a.Hkv ? hs : hs - a.Hkv) * a.cache_head_bytes;
            type = a.cache_type;
        }
        if (type == VVA_TYPE_Q8_0) {
            store8_q8(dst, it.i0, y0);
            store8_q8(dst, it.i0 + P, y1);
        } else {
            const int eo = type == VVA_TYPE_F32 ? 4 : 2;
            store8(dst + it.i0 * eo, type, y0);
            store8(dst + (it.i0 + P) * eo, type, y1);
        }
    }
}

bool rope_vec_ok(const RopeAppendArgs& a) {
    if (a.d != 64 && a.d != 128) return false;
    auto al = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
    auto al64 = [](int64_t x) { return (x & 15) == 0; };
    if (a.do_q && (!al(a.q) || !al(a.q_out) || !al64(a.q_nb_h) || !al64(a.q_nb_t) || !al64(a.q_nb_b) ||
                   !al64(a.qo_nb_h) || !al64(a.qo_nb_t) || !al64(a.qo_nb_b)))
        return false;
    if (a.do_kv) {
        if (!al(a.k) || !al(a.v) || !al64(a.k_nb_h) || !al64(a.k_nb_t) || !al64(a.k_nb_b) || !al64(a.v_nb_h) ||
            !al64(a.v_nb_t) || !al64(a.v_nb_b))
            return false;
        // Q8_0 rows are written in 2-byte units (every block is 34 bytes)
        if (a.cache_type != VVA_TYPE_Q8_0) {
            if (!al64(a.cache_row_bytes) || !al64(a.cache_head_bytes)) return false;
            for (int b = 0; b < a.B; ++b)
                if (!al(a.k_dst[b]) || !al(a.v_dst[b])) return false;
        }
    }
    return true;
}

}  // namespace

hipError_t launch_rope_append(const RopeAppendArgs& a, hipStream_t s) {
    if (a.T <= 0 || a.B <= 0) return hipSuccess;
    const int items = ((a.do_q ? a.Hq : 0) + (a.do_kv ? 2 * a.Hkv : 0)) * (a.d / 2);
    if (items <= 0) return hipSuccess;
    const int64_t n = (int64_t)a.T * a.B;
    // Few rows of 64-dim heads into a Q8_0 cache: the scalar kernel's workgroups
    // (3 a token at 0.5B heads) fit the CUs and its lanes have one pair each to
    // quantize (us per call, 9 rows 4.00 against 4.16 of the vector kernel, 64
    // rows 4.11 against 4.25 (BF16 input 4.37); 100 rows 4.32 against 4.25; 128-dim
    // heads, 9 rows 4.72 against 3.96).
    const bool few_q8 = a.d == 64 && n < 80 && a.do_kv && a.cache_type == VVA_TYPE_Q8_0;
    if (!few_q8 && rope_vec_ok(a)) {
        const int per_tok = items / 8;
        // Tokens per workgroup: short calls need the workgroups (512 tokens at
        // 7B heads, BF16 in, Q8_0 cache: 5.9 us at 1 in slices of 256 items,
        // 6.5 unsliced, 8.6 at 2), long ones pay less per token for the angles
        // (32768 tokens: 155 us at 1, 135 at 2, 135 at 4, 137 at 8; 4096 tokens
        // at 1.5B heads: 13.5, 11.0, 11.1, 12.9; 2000 at 0.5B: 7.3, 5.8, 6.8, 7.6).
        const int tok = n < 1024 ? 1 : 2;
        const int slices = tok == 1 ? (per_tok + 255) / 256 : 1;
        const int per_block = ((tok * per_tok + slices - 1) / slices + 255) / 256 * 256;
        const dim3 grid((a.T + tok - 1) / tok, a.B, slices);
#define VVA_ROPE(TOK)                                                                                               \
        case TOK:                                                                                                   \
            if (a.d == 64) hipLaunchKernelGGL((rope_append_vec_kernel<32, TOK>), grid, dim3(256), 0, s, a, per_block); \
            else           hipLaunchKernelGGL((rope_append_vec_kernel<64, TOK>), grid, dim3(256), 0, s, a, per_block); \
            break;
        switch (tok) {
            VVA_ROPE(1) VVA_ROPE(2)
        }
#undef VVA_ROPE
        return hipGetLastError();
    }
    int split = 1;
    if ((int64_t)a.T * a.B < 512) split = (items + 255) / 256;       // one item per thread
    const int per_block = ((items + split - 1) / split + 255) / 256 * 256;
    split = (items + per_block - 1) / per_block;
    dim3 grid(a.T, a.B, split);
    hipLaunchKernelGGL(rope_append_kernel, grid, dim3(256), 0, s, a, per_block);
    return hipGetLastError();
}

}  // namespace vva
