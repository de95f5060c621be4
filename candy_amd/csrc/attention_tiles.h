// Prompt attention on the matrix cores, what its kernels share: scores S^T = K Q^T and outputs O^T += V^T P^T on 16-bit
// operands, so that a lane holds scores and outputs of one query only (the four lanes 16 apart share the query) and hands
// the weights to the second product from registers; rows of K and V go to LDS as they lie in memory, by direct loads, and
// V is read transposed.
#pragma once

#include "blocks.h"

namespace candy {

typedef float tile_f4 __attribute__((ext_vector_type(4)));

// over the four lanes 16 apart that share a query
__device__ __forceinline__ float quad16_max(float v) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float quad16_sum(float v) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// four rows of a 16-bit matrix in LDS, transposed: lane l of 16 receives column l (lane l points at row l / 4, values
// 4 (l % 4) .. + 3)
template <class T>
__device__ __forceinline__ auto lds_columns(const T *p) {
    typedef short s4 __attribute__((ext_vector_type(4)));
    typedef T t4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(t4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4 *)p));
}

// Rows of a tile lie end to end in LDS, `pieces` of 16 bytes each (a multiple of 8); piece c of row r sits in slot
// c ^ turn(r).  For K a fragment read takes one piece of each of 16 rows, for V a column read two pieces of each of 8 rows:
// either way they are in different banks.
__device__ __forceinline__ constexpr int k_turn(int pieces, int r) { return (pieces & 15) == 0 ? r & 15 : (r >> 1) & 7; }
__device__ __forceinline__ constexpr int v_turn(int pieces, int r) {
    return (pieces & 15) == 0 ? ((r & 7) << 1) | ((r >> 3) & 1) : (((r >> 1) & 3) << 1) | ((r >> 3) & 1);
}

// Workgroup -> head and query tile: the workgroups of neighbouring heads on one XCD (they may share K and V), the longest
// walks first.
__device__ __forceinline__ void attn_tile(int id, int n_heads, int q_tiles, int &head, int &tile) {
    if ((n_heads & 7) == 0) {
        const int per = n_heads >> 3, s = id >> 3;
        head = (id & 7) * per + s % per;
        tile = q_tiles - 1 - s / per;
    } else {
        head = id % n_heads;
        tile = q_tiles - 1 - id / n_heads;
    }
}

// a scale as Bf16Tiles takes it: positive, also where it is 0 (a masked score is -infinity times it)
__device__ __forceinline__ float tile_scale(float s) { return s == 0.0f ? 1.2e-38f : fabsf(s); }

// bfloat16 operands (weights in two parts), 64 queries of one head per workgroup of four wavefronts: two groups of two on
// alternate tiles of 32 keys, 32 queries per wavefront.
template <int DK, int DV>
struct Bf16Tiles {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    typedef __bf16 v4 __attribute__((ext_vector_type(4)));
    static constexpr int QT = 64, R = 64, CK = DK / 8, CV = DV / 8, KS = DK / 32, DT = DV / 16;
    static constexpr int STEP = R * (CK + CV), MERGE = (4 + 2 * 4 * DT) * 32;  // 16-byte pieces
    static constexpr int LDS = 2 * STEP > MERGE ? 2 * STEP : MERGE;
    static_assert(DK % 64 == 0 && DV % 64 == 0, "whole pieces per thread, pieces in eights");
    float m[2], l[2];          // per query: running maximum, sum of weights (of this lane's keys until the end)
    tile_f4 o[2][DT];

    // qf: the wavefront's queries (16 + 16); key(p, c), value(p, c): address of piece c of position p's row; p_first: a multiple of
    // 64; positions up to `last`; wq0: first position of the wavefront's queries; reach: a query sees so many positions back,
    // itself included; the exponent of 2 is mul * raw(z) + add of the product z, with mul > 0, so that the maximum is
    // taken before the one fma that it is subtracted in.  m (finite) and l hold the initial state (second group: none).
    template <class Key, class Value, class Raw>
    __device__ __forceinline__ void run(uint4 *s, int tid, int wq0, int p_first, int last, int reach, const v8 (&qf)[2][KS], Key key, Value value,
                                        Raw raw, float mul, float add) {
        const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4, kg = wave >> 1;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int d = 0; d < DT; ++d) o[t][d] = tile_f4{0.f, 0.f, 0.f, 0.f};
        auto stage = [&](int p0, int buf) __attribute__((always_inline)) {
            auto put = [&](const void *from, int at) __attribute__((always_inline)) {
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)from,
                                                 (__attribute__((address_space(3))) void *)&s[buf * STEP + at + wave * 64], 16, 0, 0);
            };
#pragma unroll
            for (int it = 0; it < R * CK / 256; ++it) {
                const int e = it * 256 + tid, row = e / CK;
                put(key(min(p0 + row, last), (e % CK) ^ k_turn(CK, row)), it * 256);
            }
#pragma unroll
            for (int it = 0; it < R * CV / 256; ++it) {
                const int e = it * 256 + tid, row = e / CV;
                put(value(min(p0 + row, last), (e % CV) ^ v_turn(CV, row)), R * CK + it * 256);
            }
        };
        const int kt_ = k_turn(CK, r16), v_row = 4 * g + (r16 >> 2), vt_ = v_turn(CV, v_row), v_half = (r16 & 3) >> 1;
        const int n_steps = (last - p_first) / R + 1;
        stage(p_first, 0);
        for (int step = 0; step < n_steps; ++step) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();  // the tile has landed for every wavefront, and the other buffer is consumed
            if (step + 1 < n_steps) stage(p_first + (step + 1) * R, (step + 1) & 1);
            const int p0 = p_first + step * R + 32 * kg;  // this wavefront's 32 keys
            if (p0 > wq0 + 31 || p0 > last || p0 + 31 <= wq0 - reach) continue;  // nothing of them is visible to its queries
            const uint4 *kb = s + (step & 1) * STEP + 32 * kg * CK, *vb = s + (step & 1) * STEP + R * CK + 32 * kg * CV;
            tile_f4 z[2][2];
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
                for (int t = 0; t < 2; ++t) z[t][kt] = tile_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    const v8 kf = __builtin_bit_cast(v8, kb[(kt * 16 + r16) * CK + ((ks * 4 + g) ^ kt_)]);
#pragma unroll
                    for (int t = 0; t < 2; ++t) z[t][kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[t][ks], z[t][kt], 0, 0, 0);
                }
            }
            v8 hi[2], lo[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int w0 = wq0 + 16 * t, qpos = w0 + r16;
                const bool whole = p0 + 31 <= w0 && p0 > w0 + 15 - reach;  // every key visible to every query
                float mx = -INFINITY;
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                    for (int j = 0; j < 4; ++j) z[t][kt][j] = raw(z[t][kt][j]);
                auto top = [&]() __attribute__((always_inline)) {
#pragma unroll
                    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                        for (int j = 0; j < 4; ++j) mx = fmaxf(mx, z[t][kt][j]);
                };
                if (whole) {
                    top();
                } else {
                    asm volatile("" ::: "memory");  // keep this a branch: as selects it costs four instructions per score on every tile
#pragma unroll
                    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const int p = p0 + kt * 16 + 4 * g + j;
                            z[t][kt][j] = p <= qpos && p > qpos - reach ? z[t][kt][j] : -INFINITY;
                        }
                    top();
                }
                const float m_new = fmaxf(m[t], __builtin_fmaf(quad16_max(mx), mul, add)), off = add - m_new;
                const float corr = __builtin_amdgcn_exp2f(m[t] - m_new);
                m[t] = m_new;
                float sum = 0.0f;
#pragma unroll
                for (int kt = 0; kt < 2; ++kt) {
                    tile_f4 w;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        w[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(z[t][kt][j], mul, off));
                        sum += w[j];
                    }
                    const v4 h = __builtin_convertvector(w, v4);
                    const v4 r = __builtin_convertvector(w - __builtin_convertvector(h, tile_f4), v4);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        hi[t][kt * 4 + j] = h[j];
                        lo[t][kt * 4 + j] = r[j];
                    }
                }
                l[t] = l[t] * corr + sum;
                if (__any(corr != 1.0f)) {
#pragma unroll
                    for (int d = 0; d < DT; ++d) o[t][d] *= corr;
                }
            }
            // K index 8 g + e of the second product stands for key 4 g + e (e < 4) or 16 + 4 g + e - 4
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                const __bf16 *a = (const __bf16 *)(vb + v_row * CV + ((2 * d + v_half) ^ vt_)) + (r16 & 1) * 4;
                const v8 vf = __builtin_shufflevector(lds_columns(a), lds_columns(a + 16 * DV), 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
                for (int t = 0; t < 2; ++t) o[t][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, lo[t], o[t][d], 0, 0, 0);
#pragma unroll
                for (int t = 0; t < 2; ++t) o[t][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, hi[t], o[t][d], 0, 0, 0);
            }
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) l[t] = quad16_sum(l[t]);
        float *st = (float *)s;  // value k of thread i of the second group at k * 128 + i
        const int at = tid & 127;
        __syncthreads();
        if (kg == 1) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                st[t * 128 + at] = m[t];
                st[(2 + t) * 128 + at] = l[t];
#pragma unroll
                for (int d = 0; d < DT; ++d)
#pragma unroll
                    for (int j = 0; j < 4; ++j) st[(4 + (t * DT + d) * 4 + j) * 128 + at] = o[t][d][j];
            }
        }
        __syncthreads();
        if (kg == 1) return;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const float m1 = st[t * 128 + at], l1 = st[(2 + t) * 128 + at], top = fmaxf(m[t], m1);
            const float f0 = __builtin_amdgcn_exp2f(m[t] - top), f1 = __builtin_amdgcn_exp2f(m1 - top);
            l[t] = l[t] * f0 + l1 * f1;
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int j = 0; j < 4; ++j) o[t][d][j] = o[t][d][j] * f0 + st[(4 + (t * DT + d) * 4 + j) * 128 + at] * f1;
        }
    }
};

}  // namespace candy
