// Prompt (prefill) stages of the Llama-style decoder: n tokens at once.
//
// candy has no attention on the CPU; a candy model composes it from MatMul / FastSoftmax / MatMul
// (backend.go:78,147) per token. For a prompt of n tokens at positions pos0 .. pos0+n-1 that is,
// per head, softmax over the cached positions 0 .. pos0+i of q_i . K^T * scale, times V:
// the same arithmetic as n successive decode steps, evaluated tile by tile here.
//   k_prefill_rope_kv   Rope (reduce.go:3987-4006: pairs (j, j + d/2)) on q in place and on k, and the
//                       new k / v rows written into the f32 cache [kv_head][position][head_dim]
//   k_kv_parts          cache rows of earlier positions as the sums of 16-bit parts the matrix cores contract
//   k_attn_prefill_mfma causal attention of 64 or 128 queries of one head against the cache on the matrix cores
//   k_attn_prefill      the same on the vector ALU: where there is no memory for the parts (and in comparison runs)
#include <cstdlib>

#include "attention_tiles.h"
#include "blocks.h"
#include "internal.h"

namespace candy {

// Four consecutive cache values as f32; KV is float (candy's cache) or _Float16 (the optional half-size cache).
template <class KV>
__device__ __forceinline__ float4 kv_load4(const KV *p);
template <>
__device__ __forceinline__ float4 kv_load4<float>(const float *p) { return *(const float4 *)p; }
template <>
__device__ __forceinline__ float4 kv_load4<_Float16>(const _Float16 *p) {
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    const h4 v = *(const h4 *)p;
    return make_float4((float)v[0], (float)v[1], (float)v[2], (float)v[3]);
}

template <class KV>
__global__ __launch_bounds__(256) void k_prefill_rope_kv(float *__restrict__ q, const float *__restrict__ k,
                                                         const float *__restrict__ v,
                                                         const float *__restrict__ cos_t,
                                                         const float *__restrict__ sin_t, KV *__restrict__ k_cache,
                                                         KV *__restrict__ v_cache, int n, int pos0, int n_heads,
                                                         int n_kv_heads, int head_dim, int64_t cache_stride) {
    const int half = head_dim >> 1;
    const int slots = n_heads + 2 * n_kv_heads;  // q heads, then k heads, then v heads
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t total = (int64_t)n * slots * half;
    if (idx >= total) return;
    const int j = (int)(idx % half);
    const int slot = (int)((idx / half) % slots);
    const int i = (int)(idx / ((int64_t)half * slots));
    const int pos = pos0 + i;
    const float c = cos_t[(size_t)pos * half + j], s = sin_t[(size_t)pos * half + j];
    if (slot < n_heads) {
        float *p = q + ((size_t)i * n_heads + slot) * head_dim + j;
        const float a = p[0], b = p[half];
        p[0] = a * c - b * s;
        p[half] = a * s + b * c;
    } else if (slot < n_heads + n_kv_heads) {
        const int h = slot - n_heads;
        const float *p = k + ((size_t)i * n_kv_heads + h) * head_dim + j;
        KV *dst = k_cache + (size_t)h * cache_stride + (size_t)pos * head_dim + j;
        const float a = p[0], b = p[half];
        dst[0] = (KV)(a * c - b * s);
        dst[half] = (KV)(a * s + b * c);
    } else {
        const int h = slot - n_heads - n_kv_heads;
        const float *p = v + ((size_t)i * n_kv_heads + h) * head_dim + j;
        KV *dst = v_cache + (size_t)h * cache_stride + (size_t)pos * head_dim + j;
        dst[0] = (KV)p[0];
        dst[half] = (KV)p[half];
    }
}

// The first P parts of four values, part_stride apart: each the rounding of what the parts before it leave.
template <class T, int P>
__device__ __forceinline__ void store_parts(T *dst, int64_t part_stride, float4 x) {
    typedef T t4 __attribute__((ext_vector_type(4)));
    float rest[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
    for (int p = 0; p < P; ++p) {
        t4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            o[e] = (T)rest[e];
            rest[e] -= (float)o[e];
        }
        *(t4 *)(dst + (size_t)p * part_stride) = o;
    }
}

// The first `count` cache rows of every kv head -> the parts k_attn_prefill_mfma reads, in rows like the cache's.
template <class T, int P>
__global__ __launch_bounds__(256) void k_kv_parts(const float *__restrict__ k_cache, const float *__restrict__ v_cache, int64_t cache_stride,
                                                  T *__restrict__ kparts, T *__restrict__ vparts, int64_t part_stride, int count, int c4) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;  // (row, four values)
    if (idx >= (int64_t)count * c4) return;
    const size_t at = (size_t)blockIdx.y * cache_stride + (size_t)idx * 4;
    store_parts<T, P>((blockIdx.z ? vparts : kparts) + at, part_stride, *(const float4 *)((blockIdx.z ? v_cache : k_cache) + at));
}

// The same four pairs per thread, for q, k and v rows that lie end to end in `src` ([n][q heads], [n][kv heads] twice),
// optionally still as the n_split partial copies of a contraction split along K, `stride` floats apart, summed here in
// the order of the separate split sum.  q is written to `q` (which may be `src`), k and v go to the cache and, with an
// f32 cache (P > 0), as parts to the rows the attention kernel reads: a launch and a pass less than k_kv_parts behind it.  The
// positions in front, whose parts may be another layer's, are workgroups of the same launch (`early_blocks` for each kv head of K, then
// of V): us a layer of 20 tokens, 8B shape, behind 16 / 64 / 2000 positions, with a launch of their own 160 / 162 / 253, now 157 / 159 / 249.
template <class KV, class T, int P>
__global__ __launch_bounds__(256) void k_prefill_rope_kv4(float *q, const float *src, int n_split, size_t stride,
                                                          const float *__restrict__ cos_t,
                                                          const float *__restrict__ sin_t, KV *__restrict__ k_cache,
                                                          KV *__restrict__ v_cache, int n, int pos0, int n_heads,
                                                          int n_kv_heads, int head_dim, int64_t cache_stride,
                                                          T *__restrict__ kparts, T *__restrict__ vparts, int64_t part_stride,
                                                          unsigned early_blocks) {
    const int half = head_dim >> 1, hq = half >> 2;
    const int slots = n_heads + 2 * n_kv_heads;  // q heads, then k heads, then v heads
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t total = (int64_t)n * slots * hq;
    if constexpr (P > 0) {
        const unsigned blocks = (unsigned)((total + 255) >> 8);
        if (blockIdx.x >= blocks) {
            const unsigned b = blockIdx.x - blocks, h = b / early_blocks;
            const int64_t e = (int64_t)(b - h * early_blocks) * 256 + threadIdx.x;
            if (e >= (int64_t)pos0 * (head_dim >> 2)) return;
            const bool is_v = h >= (unsigned)n_kv_heads;
            const size_t at = (size_t)(is_v ? h - n_kv_heads : h) * cache_stride + (size_t)e * 4;
            store_parts<T, P>((is_v ? vparts : kparts) + at, part_stride, *(const float4 *)((is_v ? v_cache : k_cache) + at));
            return;
        }
    }
    if (idx >= total) return;
    const int j = (int)(idx % hq) * 4;
    const int slot = (int)((idx / hq) % slots);
    const int i = (int)(idx / ((int64_t)hq * slots));
    const int pos = pos0 + i;
    auto load = [&](size_t off) {
        float4 t = *(const float4 *)(src + off);
        for (int k = 1; k < n_split; ++k) {
            const float4 u = *(const float4 *)(src + (size_t)k * stride + off);
            t.x += u.x; t.y += u.y; t.z += u.z; t.w += u.w;
        }
        return t;
    };
    auto store = [&](KV *dst, float4 t) {  // 4-element aligned: head_dim % 8 == 0
        typedef KV kv4 __attribute__((ext_vector_type(4)));
        kv4 o;
        o[0] = (KV)t.x; o[1] = (KV)t.y; o[2] = (KV)t.z; o[3] = (KV)t.w;
        *(kv4 *)dst = o;
    };
    const size_t k_base = (size_t)n * n_heads * head_dim, v_base = k_base + (size_t)n * n_kv_heads * head_dim;
    if (slot >= n_heads + n_kv_heads) {
        const int h = slot - n_heads - n_kv_heads;
        const size_t off = v_base + ((size_t)i * n_kv_heads + h) * head_dim + j;
        const size_t at = (size_t)h * cache_stride + (size_t)pos * head_dim + j;
        const float4 x = load(off), y = load(off + half);
        store(v_cache + at, x);
        store(v_cache + at + half, y);
        store_parts<T, P>(vparts + at, part_stride, x);
        store_parts<T, P>(vparts + at + half, part_stride, y);
        return;
    }
    const float4 c = *(const float4 *)(cos_t + (size_t)pos * half + j), s = *(const float4 *)(sin_t + (size_t)pos * half + j);
    const bool is_q = slot < n_heads;
    const int h = is_q ? slot : slot - n_heads;
    const size_t off = is_q ? ((size_t)i * n_heads + h) * head_dim + j : k_base + ((size_t)i * n_kv_heads + h) * head_dim + j;
    const float4 a = load(off), b = load(off + half);
    const float4 lo = make_float4(a.x * c.x - b.x * s.x, a.y * c.y - b.y * s.y, a.z * c.z - b.z * s.z, a.w * c.w - b.w * s.w);
    const float4 hi = make_float4(a.x * s.x + b.x * c.x, a.y * s.y + b.y * c.y, a.z * s.z + b.z * c.z, a.w * s.w + b.w * c.w);
    if (is_q) {
        *(float4 *)(q + off) = lo;
        *(float4 *)(q + off + half) = hi;
    } else {
        const size_t at = (size_t)h * cache_stride + (size_t)pos * head_dim + j;
        store(k_cache + at, lo);
        store(k_cache + at + half, hi);
        store_parts<T, P>(kparts + at, part_stride, lo);
        store_parts<T, P>(kparts + at + half, part_stride, hi);
    }
}

// grid (n_heads, ceil(n / 32)), 256 threads. Thread t serves query row t/8 throughout: in the score
// phase it owns keys {t%8 + 8r}, in the output phase columns {4*(t%8) + 32r .. +3}; the 8 threads of
// a row sit in adjacent lanes, so the row maximum and sum are three xor-shuffles.
template <int HD, class KV>
__global__ __launch_bounds__(256) void k_attn_prefill(const float *__restrict__ q, const KV *__restrict__ k_cache,
                                                      const KV *__restrict__ v_cache, float *__restrict__ out,
                                                      int n, int pos0, int n_heads, int n_kv_heads,
                                                      int64_t cache_stride, float scale) {
    constexpr int QT = 32, KT = 32, PITCH = HD + 4;  // pitch = 4 mod 64 banks: the 8 rows of a read never collide
    __shared__ __align__(16) float s_q[QT * PITCH];
    __shared__ __align__(16) float s_k[KT * PITCH];
    __shared__ __align__(16) float s_v[KT * HD];
    __shared__ __align__(16) float s_p[QT * KT];
    const int tid = threadIdx.x, qi = tid >> 3, sub = tid & 7;
    const int head = blockIdx.x, i0 = blockIdx.y * QT;
    const int kvh = head / (n_heads / n_kv_heads);
    const KV *kh = k_cache + (size_t)kvh * cache_stride, *vh = v_cache + (size_t)kvh * cache_stride;
    const int rows = min(QT, n - i0);
    const int n_keys = pos0 + i0 + rows;    // the tile's last query sees this many positions
    const int my_last = pos0 + i0 + qi;     // last position query row qi may attend
    constexpr int F4 = HD / 4;

    for (int e = tid; e < QT * F4; e += 256) {
        const int r = e / F4, c4 = e % F4;
        const int i = min(i0 + r, n - 1);
        *(float4 *)&s_q[r * PITCH + 4 * c4] = *(const float4 *)(q + ((size_t)i * n_heads + head) * HD + 4 * c4);
    }
    float m_run = -INFINITY, l_run = 0.0f;
    float4 o[HD / 32];
#pragma unroll
    for (int r = 0; r < HD / 32; ++r) o[r] = make_float4(0.f, 0.f, 0.f, 0.f);

    for (int p0 = 0; p0 < n_keys; p0 += KT) {
        __syncthreads();  // previous tile fully consumed (and s_q written, first time round)
        for (int e = tid; e < KT * F4; e += 256) {
            const int r = e / F4, c4 = e % F4;
            const size_t p = (size_t)min(p0 + r, n_keys - 1);
            *(float4 *)&s_k[r * PITCH + 4 * c4] = kv_load4(kh + p * HD + 4 * c4);
            *(float4 *)&s_v[r * HD + 4 * c4] = kv_load4(vh + p * HD + 4 * c4);
        }
        __syncthreads();
        // scores of (row qi, keys sub + 8r)
        float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
        for (int d = 0; d < HD; d += 4) {
            const float4 qv = *(const float4 *)&s_q[qi * PITCH + d];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float4 kv = *(const float4 *)&s_k[(sub + 8 * r) * PITCH + d];
                s[r] += qv.x * kv.x + qv.y * kv.y + qv.z * kv.z + qv.w * kv.w;
            }
        }
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const bool ok = p0 + sub + 8 * r <= my_last;
            s[r] = ok ? s[r] * scale : -INFINITY;
            mx = fmaxf(mx, s[r]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 1));
        mx = fmaxf(mx, __shfl_xor(mx, 2));
        mx = fmaxf(mx, __shfl_xor(mx, 4));
        const float m_new = fmaxf(m_run, mx);  // position 0 is visible to every row, so m_new is finite
        const float corr = expf(m_run - m_new);
        float ps = 0.0f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float pw = expf(s[r] - m_new);  // exp(-inf) = 0 for masked keys
            s_p[qi * KT + sub + 8 * r] = pw;
            ps += pw;
        }
        ps += __shfl_xor(ps, 1);
        ps += __shfl_xor(ps, 2);
        ps += __shfl_xor(ps, 4);
        l_run = l_run * corr + ps;
        m_run = m_new;
#pragma unroll
        for (int r = 0; r < HD / 32; ++r) {
            o[r].x *= corr; o[r].y *= corr; o[r].z *= corr; o[r].w *= corr;
        }
        __syncthreads();  // probabilities of the whole tile are in LDS
#pragma unroll 4
        for (int kk = 0; kk < KT; ++kk) {
            const float pw = s_p[qi * KT + kk];
#pragma unroll
            for (int r = 0; r < HD / 32; ++r) {
                const float4 vv = *(const float4 *)&s_v[kk * HD + 4 * sub + 32 * r];
                o[r].x += pw * vv.x; o[r].y += pw * vv.y; o[r].z += pw * vv.z; o[r].w += pw * vv.w;
            }
        }
    }
    if (qi < rows) {
        const float inv = 1.0f / l_run;
        float *dst = out + ((size_t)(i0 + qi) * n_heads + head) * HD;
#pragma unroll
        for (int r = 0; r < HD / 32; ++r)
            *(float4 *)(dst + 4 * sub + 32 * r) = make_float4(o[r].x * inv, o[r].y * inv, o[r].z * inv, o[r].w * inv);
    }
}

// ------------------------------------------------------------------ causal attention on the matrix cores
// An f32 operand meets the matrix cores as a sum of parts, each part the rounding of what the parts before it leave:
//   head_dim 128, f32 cache   two fp16 parts of q, K, V and the weights (22 bits), three products
//   head_dim 64, f32 cache    three bfloat16 parts (24 bits and f32's range: what the vector ALU had), six products
//   fp16 cache                K and V are their own single part; q and the weights in two fp16 parts, for head_dim 64 in three
//                             (24 bits and f32's range: a query's row scaled to 2^13 .. 2^14, the weights by 2^15, so that what
//                             falls below the last part's 2^-24 is 2^-38 of the row's largest value or the largest weight)
// K and V parts lie in memory as rows like the cache's (k_kv_parts; a fp16 cache is read as it is), so that a tile goes
// to LDS by direct loads and no workgroup converts what the others of its head convert as well.
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4h __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));

template <class T> struct PartVec;
template <> struct PartVec<_Float16> { typedef half8 v8; typedef half4h v4; };
template <> struct PartVec<__bf16> { typedef __bf16 v8 __attribute__((ext_vector_type(8))); typedef __bf16 v4 __attribute__((ext_vector_type(4))); };

__device__ __forceinline__ float4v mfma16(half8 a, half8 b, float4v c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ float4v mfma16(PartVec<__bf16>::v8 a, PartVec<__bf16>::v8 b, float4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// One query's attention by a wavefront on the vector ALU in f32, 64 keys at a time: lane d returns result d of 64.  For results
// of the matrix cores that are no numbers: an infinity, or a value that rounds to one, becomes inf - inf in parts, where in
// one piece it may only have been a weight of 0 or an infinite result.
template <class KV>
__device__ float attn_row_valu(const float *__restrict__ q, const KV *__restrict__ k, const KV *__restrict__ v, int n_keys, float scale, int lane) {
    float m = -INFINITY, l = 0.0f, o = 0.0f;
    for (int p0 = 0; p0 < n_keys; p0 += 64) {
        const KV *row = k + (size_t)min(p0 + lane, n_keys - 1) * 64;
        float s = 0.0f;
        for (int d = 0; d < 64; d += 4) {
            const float4 a = *(const float4 *)(q + d), b = kv_load4(row + d);
            s += a.x * b.x + a.y * b.y + a.z * b.z + a.w * b.w;
        }
        s = p0 + lane < n_keys ? s * scale : -INFINITY;
        const float m_new = fmaxf(m, wave_max(s));
        const float m_at = m_new == -INFINITY ? 0.0f : m_new, corr = expf(m - m_at), w = expf(s - m_at);
        m = m_new;
        l = l * corr + wave_sum(w);
        o *= corr;
        for (int i = 0; i < min(64, n_keys - p0); ++i)
            o += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w), i)) * (float)v[(size_t)(p0 + i) * 64 + lane];
    }
    return o * (1.0f / l);
}

template <int HD, class T, int KVP, int QP, int PP, int QH, int KG>
__global__ __launch_bounds__(64 * QH * KG, KVP * KG * HD * 256 > 81920 && QH * KG == 4 ? 1 : 2) void k_attn_prefill_mfma(const float *__restrict__ q, const T *__restrict__ kparts, const T *__restrict__ vparts,
                                                              int64_t part_stride, int64_t head_stride, float *__restrict__ out, int n, int pos0,
                                                              int n_heads, int group, int q_tiles, float scale,
                                                              _Float16 *__restrict__ xh_out, const float *k_cache, const float *v_cache) {
    typedef typename PartVec<T>::v8 v8;
    typedef typename PartVec<T>::v4 v4;
    constexpr int THREADS = 64 * QH * KG, QT = 32 * QH, R = 32 * KG, C = HD / 8, KS = HD / 32, DT = HD / 16;
    constexpr int ARR = R * C, STEP = 2 * KVP * ARR;  // 16-byte pieces of one part of K or V, and of everything a step stages
    constexpr int IT = ARR / THREADS;
    static_assert(ARR % THREADS == 0 && (HD == 64 || HD == 128), "whole pieces per thread");
    constexpr int MERGE = KG == 1 ? 0 : (2 + 4 * DT) * 32 * QH;  // half of either key group's state at the end
    __shared__ __align__(16) uint4 s_all[2 * STEP > MERGE ? 2 * STEP : MERGE];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int qh = wave % QH, kg = wave / QH;
    int head, qt0;
    attn_tile(blockIdx.x, n_heads, q_tiles, head, qt0);
    const int i0 = qt0 * QT;
    const T *kh = kparts + (size_t)(head / group) * head_stride, *vh = vparts + (size_t)(head / group) * head_stride;
    const int n_keys = pos0 + min(i0 + QT, n);  // positions the tile's last query may see
    const int wq0 = pos0 + i0 + 32 * qh;         // first position of this wavefront's 32 queries

    // q as the B operand (column = query, 8 consecutive d per lane), scaled for a softmax on powers of two
    constexpr bool WIDE = KVP == 1 && QP == 3;  // fp16 parts that stand for 32 bits
    v8 qf[2][KS][QP];
    float q_up[2], q_down[2];  // WIDE: a power of two on the query's row, and its inverse
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const float *qr = q + ((size_t)min(i0 + 32 * qh + 16 * t + r16, n - 1) * n_heads + head) * HD;
        if (WIDE) {
            float amax = 0.0f;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const float4 a = *(const float4 *)(qr + ks * 32 + g * 8), b = *(const float4 *)(qr + ks * 32 + g * 8 + 4);
                amax = fmaxf(amax, fmaxf(fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))),
                                         fmaxf(fmaxf(fabsf(b.x), fabsf(b.y)), fmaxf(fabsf(b.z), fabsf(b.w)))));
            }
            const int up = min(14 - __builtin_amdgcn_frexp_expf(quad16_max(amax) * (scale * 1.44269504088896341f)), 120);
            q_up[t] = ldexpf(1.0f, up);
            q_down[t] = ldexpf(1.0f, -up);
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const float4 a = *(const float4 *)(qr + ks * 32 + g * 8), b = *(const float4 *)(qr + ks * 32 + g * 8 + 4);
            const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float rest = v[e] * (scale * 1.44269504088896341f);
                if (WIDE) rest *= q_up[t];
#pragma unroll
                for (int p = 0; p < QP; ++p) {
                    qf[t][ks][p][e] = (T)rest;
                    rest -= (float)qf[t][ks][p][e];
                }
            }
        }
    }
    float m_run[2] = {-INFINITY, -INFINITY}, l_run[2] = {0.0f, 0.0f};  // the sum is over this lane's keys until the end
    float4v o[2][DT];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int d = 0; d < DT; ++d) o[t][d] = float4v{0.f, 0.f, 0.f, 0.f};

    auto turn = [](int r) { return v_turn(C, r); };  // K and V alike
    auto stage = [&](int p0, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int a = 0; a < 2 * KVP; ++a) {
            const T *src = (a < KVP ? kh : vh) + (size_t)(a < KVP ? a : a - KVP) * part_stride;
#pragma unroll
            for (int it = 0; it < IT; ++it) {
                const int e = it * THREADS + tid, row = e / C, c = (e % C) ^ turn(row);
                const T *from = src + (size_t)min(p0 + row, n_keys - 1) * HD + c * 8;
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)from,
                                                 (__attribute__((address_space(3))) void *)&s_all[buf * STEP + a * ARR + it * THREADS + wave * 64], 16, 0, 0);
            }
        }
    };
    const int k_at = turn(r16), v_row = 4 * g + (r16 >> 2), v_at = turn(v_row), v_half = (r16 & 3) >> 1;
    const int n_steps = (n_keys + R - 1) / R;
    stage(0, 0);
    for (int step = 0; step < n_steps; ++step) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();  // the tile has landed for every wavefront, and the other buffer is consumed
        if (step + 1 < n_steps) stage((step + 1) * R, (step + 1) & 1);
        const int p0 = step * R + 32 * kg;  // this wavefront's 32 keys
        if (p0 > wq0 + 31 || p0 >= n_keys) continue;
        const uint4 *base = s_all + (step & 1) * STEP + 32 * kg * C;
        // ---- scores, transposed: rows are keys, a lane holds those of query r16, keys 16 kt + 4 g + j
        float4v s[2][2];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) s[t][kt] = float4v{0.f, 0.f, 0.f, 0.f};
        constexpr int TOP = QP > KVP ? QP : KVP;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
            v8 kf[KS][KVP];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int p = 0; p < KVP; ++p) kf[ks][p] = __builtin_bit_cast(v8, base[p * ARR + (kt * 16 + r16) * C + ((ks * 4 + g) ^ k_at)]);
#pragma unroll
            for (int sum = TOP - 1; sum >= 0; --sum)  // the smallest products first
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                    for (int p = 0; p < KVP; ++p)
                        if (sum - p >= 0 && sum - p < QP) {
#pragma unroll
                            for (int t = 0; t < 2; ++t) s[t][kt] = mfma16(kf[ks][p], qf[t][ks][sum - p], s[t][kt]);
                        }
        }
        // ---- online softmax: every score of a query is in the four lanes 16 apart
        v8 pf[2][PP];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int qpos = wq0 + 16 * t + r16;
            if (p0 + 31 > wq0 + 16 * t) {
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                    for (int j = 0; j < 4; ++j) s[t][kt][j] = p0 + kt * 16 + 4 * g + j <= qpos ? s[t][kt][j] : -INFINITY;
            }
            float mx = fmaxf(fmaxf(fmaxf(s[t][0][0], s[t][0][1]), fmaxf(s[t][0][2], s[t][0][3])),
                             fmaxf(fmaxf(s[t][1][0], s[t][1][1]), fmaxf(s[t][1][2], s[t][1][3])));
            // WIDE: a maximum rounded up to a whole power of two, so that the weights' scale costs them no bit
            const float m_new = fmaxf(m_run[t], WIDE ? ceilf(quad16_max(mx) * q_down[t]) : quad16_max(mx));
            const float m_at = m_new == -INFINITY ? 0.0f : m_new;  // nothing visible yet: all weights are 2^-inf = 0
            const float corr = __builtin_amdgcn_exp2f(m_run[t] - m_at);
            m_run[t] = m_new;
            float sum = 0.0f;
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float w = __builtin_amdgcn_exp2f(WIDE ? __builtin_fmaf(s[t][kt][j], q_down[t], 15.0f - m_at) : s[t][kt][j] - m_at);
                    sum += w;
#pragma unroll
                    for (int p = 0; p < PP; ++p) {
                        pf[t][p][kt * 4 + j] = (T)w;
                        w -= (float)pf[t][p][kt * 4 + j];
                    }
                }
            l_run[t] = l_run[t] * corr + sum;
            if (__any(corr != 1.0f)) {  // the maxima settle after the first tiles
#pragma unroll
                for (int d = 0; d < DT; ++d) o[t][d] *= corr;
            }
        }
        // ---- outputs, transposed: O^T += V^T P^T; K index 8 g + e stands for key 4 g + e (e < 4) or 16 + 4 g + e - 4
        constexpr int TOPV = PP > KVP ? PP : KVP;
#pragma unroll
        for (int d = 0; d < DT; ++d) {
            v8 vf[KVP];
            const int at = v_row * C + ((2 * d + v_half) ^ v_at);
#pragma unroll
            for (int p = 0; p < KVP; ++p) {
                const T *a = (const T *)(base + (KVP + p) * ARR + at) + (r16 & 1) * 4;
                const v4 lo = lds_columns(a), hi = lds_columns(a + 16 * HD);
                vf[p] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            }
#pragma unroll
            for (int sum = TOPV - 1; sum >= 0; --sum)
#pragma unroll
                for (int p = 0; p < KVP; ++p)
                    if (sum - p >= 0 && sum - p < PP) {
#pragma unroll
                        for (int t = 0; t < 2; ++t) o[t][d] = mfma16(vf[p], pf[t][sum - p], o[t][d]);
                    }
        }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) l_run[t] = quad16_sum(l_run[t]);
    // The two key groups share the end as well: group 0 takes the first 16 queries of each 32, group 1 the others; what the other
    // group needs goes through LDS, value k of thread t of group kg at (2 k + kg) * 64 QH + t.  With one group merging, dividing
    // and quantizing both halves, level by level, what is not the walk along the keys was 17 of 31 us at 512 tokens.  Kernel us, so / now:
    // head_dim 128, 512 tokens 31.5 / 27.4, fp16 cache 24.8 / 19.9, 2000 tokens 129 / 119 (113 to 124 from run to run); head_dim 64, 1500 tokens 78 / 73.
    constexpr int NT = KG == 2 ? 1 : 2;  // 16 queries each
    const int t_own = KG == 2 ? kg : 0;
    if constexpr (KG == 2) {
        constexpr int GROUP = 64 * QH;
        float *st = (float *)s_all;
        const int at = tid & (GROUP - 1);
        auto give = [&](int t) __attribute__((always_inline)) {
            float *to = st + kg * GROUP + at;
            to[0] = m_run[t];
            to[2 * GROUP] = l_run[t];
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int j = 0; j < 4; ++j) to[(4 + 8 * d + 2 * j) * GROUP] = o[t][d][j];
        };
        auto merge = [&](int t) __attribute__((always_inline)) {
            const float *from = st + (1 - kg) * GROUP + at;
            const float m_its = from[0], l_its = from[2 * GROUP];
            const float m = fmaxf(m_run[t], m_its);  // finite: position 0 is in the first group
            const float f_own = __builtin_amdgcn_exp2f(m_run[t] - m), f_its = __builtin_amdgcn_exp2f(m_its - m);
            // the sums in the order of the groups
            const float f0 = t == 0 ? f_own : f_its, f1 = t == 0 ? f_its : f_own;
            l_run[0] = __builtin_fmaf(t == 0 ? l_run[t] : l_its, f0, (t == 0 ? l_its : l_run[t]) * f1);
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float its = from[(4 + 8 * d + 2 * j) * GROUP], own = o[t][d][j];
                    o[0][d][j] = __builtin_fmaf(t == 0 ? own : its, f0, (t == 0 ? its : own) * f1);
                }
        };
        __syncthreads();
        if (kg == 0) give(1);
        else give(0);
        __syncthreads();
        if (kg == 0) merge(0);
        else merge(1);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const float inv = 1.0f / l_run[t];
#pragma unroll
        for (int d = 0; d < DT; ++d) o[t][d] *= inv;
    }
    if constexpr (HD == 64) {
        unsigned long long lost[2] = {0, 0};  // the 16 queries each whose results are no numbers
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            float all = 0.0f;
#pragma unroll
            for (int d = 0; d < DT; ++d) all += (o[t][d][0] + o[t][d][1]) + (o[t][d][2] + o[t][d][3]);
            lost[t] = __ballot(all != all && i0 + 32 * qh + 16 * (t + t_own) + r16 < n);
        }
        if (__builtin_expect((lost[0] | lost[1]) != 0, 0)) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                lost[t] = (lost[t] | lost[t] >> 16 | lost[t] >> 32 | lost[t] >> 48) & 0xFFFF;
                while (lost[t]) {
                    const int r = __builtin_ctzll(lost[t]), row = i0 + 32 * qh + 16 * (t + t_own) + r;
                    lost[t] &= lost[t] - 1;
                    const float *qr = q + ((size_t)row * n_heads + head) * HD;
                    float res;
                    if constexpr (KVP == 1) {
                        res = attn_row_valu(qr, kh, vh, pos0 + row + 1, scale, lane);
                    } else {
                        const size_t at = (size_t)(head / group) * head_stride;
                        res = attn_row_valu(qr, k_cache + at, v_cache + at, pos0 + row + 1, scale, lane);
                    }
#pragma unroll
                    for (int d = 0; d < DT; ++d)
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const float x = __shfl(res, 16 * d + 4 * g + j, 64);
                            if (r16 == r) o[t][d][j] = x;
                        }
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int i = i0 + 32 * qh + 16 * (t + t_own) + r16;
        if (xh_out) {
            // The row leaves as the fp16 image of its Q8_0 quantization (what the o projection's fp16 tiles contract
            // with), the arithmetic of quantize_q8_lane4 + q8_lane4_to_half value by value: a 32-value block is
            // o[2 b] and o[2 b + 1] of the four lanes that share the query.
            const int K = n_heads * HD;
#pragma unroll
            for (int b = 0; b < DT / 2; ++b) {
                float x[8], level[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = o[t][2 * b + (e >> 2)][e & 3];
                float amax = fabsf(x[0]);  // (not 0: a block without a number has no largest value, and stays so)
#pragma unroll
                for (int e = 1; e < 8; ++e) amax = fmaxf(amax, fabsf(x[e]));
                amax = quad16_max(amax);
                const float dq = amax / 127.0f, df = __half2float(__float2half_rn(dq));
                q8_levels8(x, amax, dq, level);
#pragma unroll
                for (int hf = 0; hf < 2; ++hf) {
                    half4h w;
#pragma unroll
                    for (int j = 0; j < 4; ++j) w[j] = (_Float16)(df * level[4 * hf + j]);
                    const int col = head * HD + 32 * b + 16 * hf + 4 * g;
                    if (i < n) *(half4h *)(xh_out + xh_index4(i, col >> 2, K) * 4) = w;
                }
            }
        } else if (i < n) {
            float *dst = out + ((size_t)i * n_heads + head) * HD + 4 * g;
#pragma unroll
            for (int d = 0; d < DT; ++d) *(float4v *)(dst + 16 * d) = o[t][d];
        }
    }
}

// The parts of K and V the matrix-core kernel contracts, for an f32 cache: three bfloat16 or two fp16 ones per value.
size_t attn_prefill_parts_bytes(int n_kv_heads, int head_dim, int max_pos) {
    return (size_t)2 * (head_dim == 64 ? 3 : 2) * n_kv_heads * max_pos * head_dim * 2;
}

static int launch_kv_parts(candy_hip_device *dev, const float *k_cache, const float *v_cache, void *parts, int count, int n_kv_heads,
                           int head_dim, int64_t cache_stride) {
    const int64_t part_stride = (int64_t)n_kv_heads * cache_stride;
    const dim3 grid((unsigned)(((int64_t)count * (head_dim / 4) + 255) / 256), (unsigned)n_kv_heads, 2);
    if (head_dim == 64)
        hipLaunchKernelGGL((k_kv_parts<__bf16, 3>), grid, dim3(256), 0, dev->stream, k_cache, v_cache, cache_stride, (__bf16 *)parts,
                           (__bf16 *)parts + 3 * part_stride, part_stride, count, head_dim / 4);
    else
        hipLaunchKernelGGL((k_kv_parts<_Float16, 2>), grid, dim3(256), 0, dev->stream, k_cache, v_cache, cache_stride, (_Float16 *)parts,
                           (_Float16 *)parts + 2 * part_stride, part_stride, count, head_dim / 4);
    CANDY_LAUNCH_CHECK();
    return CANDY_HIP_OK;
}

int launch_prefill_rope_kv(candy_hip_device *dev, float *q, const float *k, const float *v, const float *cos_t,
                           const float *sin_t, void *k_cache, void *v_cache, bool kv_f16, int n, int pos0, int n_heads,
                           int n_kv_heads, int head_dim, int64_t cache_stride, void *parts, const SplitPending *sp) {
    const int64_t part_stride = (int64_t)n_kv_heads * cache_stride;
    const size_t q_count = (size_t)n * n_heads * head_dim, kv_count = (size_t)n * n_kv_heads * head_dim;
    const bool pending = sp && sp->n_split > 0;
    if (pending) CANDY_REQUIRE(sp->y == q && !sp->res && sp->count == q_count + 2 * kv_count, "internal: pending split sum of another shape");
    if (head_dim % 8 == 0 && k == q + q_count && v == k + kv_count && dev->opt.prefill_fold_split_sums) {
        // q, k and v end to end: four pairs per thread, and the partial copies of a split contraction summed on the way
        const int64_t total4 = (int64_t)n * (n_heads + 2 * n_kv_heads) * (head_dim / 8);
        const int64_t early = parts && !kv_f16 ? ((int64_t)pos0 * (head_dim / 4) + 255) / 256 : 0;
        const int64_t blocks = (total4 + 255) / 256 + 2 * n_kv_heads * early;
        CANDY_REQUIRE(blocks <= 0x7FFFFFFF, "prompt too long for one pass");
        const dim3 grid4((unsigned)blocks);
        const float *src = pending ? sp->part : q;
        const int n_split = pending ? sp->n_split : 1;
        const size_t stride = pending ? sp->stride : 0;
#define CANDY_ROPE4(KV, T, P)                                                                                                            \
    hipLaunchKernelGGL((k_prefill_rope_kv4<KV, T, P>), grid4, dim3(256), 0, dev->stream, q, src, n_split, stride, cos_t, sin_t,          \
                       (KV *)k_cache, (KV *)v_cache, n, pos0, n_heads, n_kv_heads, head_dim, cache_stride, (T *)parts,                   \
                       (T *)parts + P * part_stride, part_stride, (unsigned)early)
        if (kv_f16) CANDY_ROPE4(_Float16, _Float16, 0);
        else if (!parts) CANDY_ROPE4(float, _Float16, 0);
        else if (head_dim == 64) CANDY_ROPE4(float, __bf16, 3);
        else CANDY_ROPE4(float, _Float16, 2);
#undef CANDY_ROPE4
        CANDY_LAUNCH_CHECK();
        return CANDY_HIP_OK;
    }
    if (pending)
        if (int rc = launch_splitk_sum(dev, sp->part, sp->y, nullptr, sp->count, sp->n_split, sp->stride)) return rc;
    const int64_t total = (int64_t)n * (n_heads + 2 * n_kv_heads) * (head_dim / 2);
    const dim3 grid((unsigned)((total + 255) / 256));
    if (kv_f16)
        hipLaunchKernelGGL(k_prefill_rope_kv<_Float16>, grid, dim3(256), 0, dev->stream, q, k, v, cos_t, sin_t,
                           (_Float16 *)k_cache, (_Float16 *)v_cache, n, pos0, n_heads, n_kv_heads, head_dim, cache_stride);
    else
        hipLaunchKernelGGL(k_prefill_rope_kv<float>, grid, dim3(256), 0, dev->stream, q, k, v, cos_t, sin_t,
                           (float *)k_cache, (float *)v_cache, n, pos0, n_heads, n_kv_heads, head_dim, cache_stride);
    CANDY_LAUNCH_CHECK();
    return parts && !kv_f16 ? launch_kv_parts(dev, (const float *)k_cache, (const float *)v_cache, parts, pos0 + n, n_kv_heads, head_dim, cache_stride)
                            : CANDY_HIP_OK;
}

template <int HD, class T, int KVP, int QP, int PP>
static void launch_attn_mfma(candy_hip_device *dev, const float *q, const T *kparts, const T *vparts, int64_t part_stride, float *out, int n,
                             int pos0, int n_heads, int n_kv_heads, int64_t cache_stride, float scale, _Float16 *xh_out,
                             const float *k_cache = nullptr, const float *v_cache = nullptr) {
    // 64 queries per workgroup and two groups of wavefronts on alternate tiles of 32 keys, because a launch lasts as long
    // as its longest walk; 128 queries where the tiles of an f32 cache (96 or 128 KB for two steps) leave a CU room for
    // one workgroup and there are more than two of the small ones per CU.  us, 64 / 128 queries: head_dim 64, f32 cache,
    // 32 heads, 700 tokens 30.6 / 36.5, 1500 95 / 75; head_dim 128 512 tokens 29.4 / 34.3, 1024 60.4 / 61.7, 2048 180 / 133;
    // fp16 cache, head_dim 64, 1500 38.3 / 44.2.  (One group: 1500 91, 2048 147.)
    const int64_t small = (int64_t)n_heads * ((n + 63) / 64);
    const int form = dev->opt.prefill_attention_groups;
#define CANDY_ATTN(QH, KG)                                                                                                            \
    do {                                                                                                                              \
        const int tiles = (n + 32 * QH - 1) / (32 * QH);                                                                              \
        hipLaunchKernelGGL((k_attn_prefill_mfma<HD, T, KVP, QP, PP, QH, KG>), dim3((unsigned)(n_heads * tiles)), dim3(64 * QH * KG),  \
                           0, dev->stream, q, kparts, vparts, part_stride, cache_stride, out, n, pos0, n_heads, n_heads / n_kv_heads, \
                           tiles, scale, xh_out, k_cache, v_cache);                                                                   \
    } while (0)
    if (form == 1) CANDY_ATTN(4, 1);
    else if (form == 2 || KVP == 1 || small <= 2 * (int64_t)dev->num_cus) CANDY_ATTN(2, 2);
    else CANDY_ATTN(4, 2);
#undef CANDY_ATTN
}

// The matrix-core kernel can leave its output as the fp16 image of the quantized rows instead of f32 (no separate
// quantize launch in front of an o projection that runs on the fp16 tiles).
bool attn_prefill_writes_half(const candy_hip_device *dev, bool half_operands) {
    return half_operands && !dev->opt.prefill_attention_valu && dev->opt.prefill_fold_split_sums;
}

int launch_attn_prefill(candy_hip_device *dev, const float *q, const void *k_cache, const void *v_cache, bool kv_f16, void *parts,
                        float *out, int n, int pos0, int n_heads, int n_kv_heads, int head_dim, int64_t cache_stride,
                        float scale, _Float16 *xh_out) {
    CANDY_REQUIRE(head_dim == 64 || head_dim == 128, "head_dim must be 64 or 128");
    CANDY_REQUIRE(n > 0 && pos0 >= 0 && n_heads % n_kv_heads == 0, "invalid attention shape");
    CANDY_REQUIRE(!xh_out || attn_prefill_writes_half(dev, kv_f16 || parts), "internal: this attention kernel writes f32 only");
    const float *kf = (const float *)k_cache, *vf = (const float *)v_cache;
    const _Float16 *kh = (const _Float16 *)k_cache, *vh = (const _Float16 *)v_cache;
    if (dev->opt.prefill_attention_valu || (!kv_f16 && !parts)) {
        const dim3 grid((unsigned)n_heads, (unsigned)((n + 31) / 32));
#define CANDY_VALU(HD, KV, K, V)                                                                                              \
    hipLaunchKernelGGL((k_attn_prefill<HD, KV>), grid, dim3(256), 0, dev->stream, q, K, V, out, n, pos0, n_heads, n_kv_heads, \
                       cache_stride, scale)
        if (head_dim == 64 && kv_f16) CANDY_VALU(64, _Float16, kh, vh);
        else if (head_dim == 64) CANDY_VALU(64, float, kf, vf);
        else if (kv_f16) CANDY_VALU(128, _Float16, kh, vh);
        else CANDY_VALU(128, float, kf, vf);
#undef CANDY_VALU
    } else if (kv_f16) {
        if (head_dim == 64)
            launch_attn_mfma<64, _Float16, 1, 3, 3>(dev, q, kh, vh, 0, out, n, pos0, n_heads, n_kv_heads, cache_stride, scale, xh_out);
        else
            launch_attn_mfma<128, _Float16, 1, 2, 2>(dev, q, kh, vh, 0, out, n, pos0, n_heads, n_kv_heads, cache_stride, scale, xh_out);
    } else {
        const int64_t ps = (int64_t)n_kv_heads * cache_stride;
        const __bf16 *pb = (const __bf16 *)parts;
        const _Float16 *ph = (const _Float16 *)parts;
        if (head_dim == 64)
            launch_attn_mfma<64, __bf16, 3, 3, 3>(dev, q, pb, pb + 3 * ps, ps, out, n, pos0, n_heads, n_kv_heads, cache_stride, scale, xh_out, kf, vf);
        else
            launch_attn_mfma<128, _Float16, 2, 2, 2>(dev, q, ph, ph + 2 * ps, ps, out, n, pos0, n_heads, n_kv_heads, cache_stride, scale, xh_out);
    }
    CANDY_LAUNCH_CHECK();
    return CANDY_HIP_OK;
}

}  // namespace candy
