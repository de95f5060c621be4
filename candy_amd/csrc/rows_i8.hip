// 3 to 255 activation rows on the int8 matrix cores, K dealt to wavefronts: y[m, N] = x[m, K] . W^T, exact like the batch-1
// matvec (integer dots of 32 values, scaled in f32; only the order of the f32 sums differs).
//
// The tile kernel of mmq_i8.hip shares activations over the wavefronts of a workgroup, with two barriers a super-block, and on
// most shapes splits K over workgroups whose copies a second launch adds up.  Here nobody waits for anybody: a workgroup owns
// 16 RF weight rows and 16 MT activation rows, each of its WAVES wavefronts takes every WAVES-th super-block of K: the blocks
// of 16 weight rows by direct loads into a slot of its own in LDS, two slots, so that the next 16 rows (or the next
// super-block) arrive while these are contracted; the activations straight into operand registers from an image in operand
// order (rows_i8.h).  The wavefronts' sums meet in LDS at the end, in pairs (reproducible).
//
// Up to eight rows the 16 columns of a product are two groups of eight (PAIRS): one takes the even, the other the odd sub-blocks (Q6_K: the
// first and the second 16 values of each), the other's values being zero in its operand, so that a result register stands for two
// dots and its conversion, product and fma are half as many.  A column's sums meet its twin's at the end.  Vector instructions of a
// super-block and wavefront: Q6_K 250 -> 180, Q4_0 144 -> 112; us of a call, 16 columns / two groups, 6 rows: 4096 x 14336 Q6_K 16.4 / 14.6, Q4_K
// 11.6 / 10.7, Q5_K 12.8 / 12.3, Q8_0 17.5 / 17.0, Q4_0 14.2 / 13.5; 32000 x 4096 Q6_K 26.4 / 23.0, Q4_K 17.7 / 16.2, Q4_0 25.5 / 23.9.
// The distance from 64 bits is smaller than with 16 columns for every format (Q6_K 8.6e-8 -> 8.2e-8, Q4_K 2.2e-7 -> 1.7e-7).
//
// What bounds it: up to 16 rows two launches and their first bytes, then the vector ALU (without any weights or activations fetched
// the Q6_K call of 6 rows took 13.8 of the 16.3 us it took with 16 columns) beside the weights at 3.5 to 4.5 TB/s; from about 48 rows
// the vector ALU alone (a conversion, a product and an fma per result and sub-block).  us of a call, before (int8 tiles, mostly with a
// split of K) -> now:
//   4096 x 14336, 6 rows   Q4_K 18.1 -> 10.6, Q5_K 17.9 -> 12.4, Q6_K 21.0 -> 14.4, Q8_0 24.4 -> 16.8, Q4_0 22.4 -> 13.5
//   11008 x 4096, 32 rows  Q4_K 15.7 -> 14.0, Q5_K 27.7 -> 14.7, Q6_K 31.6 -> 22.0, Q8_0 41.6 -> 18.0, Q4_0 38.1 -> 14.9
//   11008 x 4096, 64 rows  Q5_K 35.0 -> 20.7, Q8_0 44.6 -> 24.2, Q4_0 37.9 -> 23.4
// and prompts of the quantized decoder (four layers and the head): 8B shape 16 / 48 / 160 tokens 603 / 885 / 1861 -> 419 / 617 /
// 1195, 1B shape 435 / 544 / 786 -> 283 / 351 / 517.
//
// The running sums are pinned every few sub-blocks (empty asm statements): left alone the compiler moves the f32 part of a super-block
// behind its last product, into the next basic block, and holds every product's result until then (300 bytes of scratch and more).
#include <algorithm>
#include <type_traits>

#include "blocks.h"
#include "internal.h"
#include "rows_i8.h"

namespace candy {

typedef int int4v __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void rows_lds_fence() {  // orders one wavefront's LDS traffic, which completes in order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The activation side of one super-block: operands of sub-blocks 2p and 2p + 1 (8 values of row lane & 15 each), the row's
// eight scales, and d * sum(q) of sub-blocks 2c and 2c + 1.
template <int MT>
struct RowsX {
    u32x4 q[MT][4];
    float4 d[MT][2];
    float2 m[MT];
};
// The same of up to eight rows, whose 16 columns of a product are two groups of eight: a column belongs to row j & 7 and takes one
// half of what is scaled apart, sub-blocks 2p + (j >> 3), or for Q6_K (halves) 16 values of every sub-block.  What a
// column does not take is zero in its operand.
template <bool HALVES>
struct RowsPairs {
    u32x4 q[HALVES ? 4 : 1];            // Q6_K: as above
    u32x2 even[4], odd[4];              // sub-blocks 2p and 2p + 1
    float d[HALVES ? 8 : 4];
    float2 m[1];
};
__device__ __forceinline__ float rows_d(const float4 (&d)[2], int t) {
    const float4 v = d[t >> 2];
    return (t & 3) == 0 ? v.x : (t & 3) == 1 ? v.y : (t & 3) == 2 ? v.z : v.w;
}
__device__ __forceinline__ long rows_b(const u32x4 (&q)[4], int t) {
    const u32x4 v = q[t >> 1];
    return t & 1 ? (long)(((uint64_t)v.w << 32) | v.z) : (long)(((uint64_t)v.y << 32) | v.x);
}
__device__ __forceinline__ long rows_pack(uint32_t lo, uint32_t hi) { return (long)(((uint64_t)hi << 32) | lo); }

// One policy per format.  A slot holds 16 rows of PIECES 16-byte pieces; lane (row j, chunk c) feeds 8 values of a sub-block.
//   factors()  lane (j, c) unpacks its part of the row's factors into ex[GROUPS][16 rows] for the lanes that own the row in
//              the C layout, and adds the minimum's (or offset's) products to acc
//   operand()  8 values of sub-block t as int8

// Q4_K, Q5_K: d * scale per sub-block, minus dmin * minimum times the activations' sum
template <bool FIVE>
struct RowsQ45K {
    static constexpr int BLOCK = FIVE ? 176 : 144, PIECES = BLOCK / 16, GROUPS = 8;
    static constexpr bool DIRECT = true, HALVES = false;
    struct Row { u32x2 q[4], qh; };
    template <int MT, class X>
    static __device__ __forceinline__ void factors(const uint8_t *wl, int j, int c, float *ex, const X &x, float4v (&acc)[MT]) {
        const u32x4 h = *(const u32x4 *)wl;
        uint32_t sc2, m2;
        q4k_scale_min_pair(h.y, h.z, h.w, c, sc2, m2);
        const float d = half_bits_to_float((uint16_t)(h.x & 0xFFFF)), dmin = half_bits_to_float((uint16_t)(h.x >> 16));
        ex[(2 * c) * 16 + j] = d * (float)(sc2 & 0xFF);
        ex[(2 * c + 1) * 16 + j] = d * (float)(sc2 >> 8);
        const float m_lo = -dmin * (float)(m2 & 0xFF), m_hi = -dmin * (float)(m2 >> 8);
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(m_lo, x.m[t].x, acc[t], 0, 0, 0);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(m_hi, x.m[t].y, acc[t], 0, 0, 0);
        }
    }
    static __device__ __forceinline__ void load(const uint8_t *wl, int c, Row &r) {
        if (FIVE) r.qh = *(const u32x2 *)(wl + 16 + 8 * c);
#pragma unroll
        for (int p = 0; p < 4; ++p) r.q[p] = *(const u32x2 *)(wl + (FIVE ? 48 : 16) + 32 * p + 8 * c);
    }
    static __device__ __forceinline__ long operand(const Row &r, int t, int) {
        const u32x2 q = r.q[t >> 1];
        const int sh = (t & 1) * 4;
        uint32_t lo = (q.x >> sh) & 0x0F0F0F0Fu, hi = (q.y >> sh) & 0x0F0F0F0Fu;
        if (FIVE) {
            lo |= ((r.qh.x >> t) & 0x01010101u) << 4;
            hi |= ((r.qh.y >> t) & 0x01010101u) << 4;
        }
        return rows_pack(lo, hi);
    }
};

// Q8_0: eight 34-byte blocks; the operand is the block's quants as they lie
struct RowsQ8_0 {
    static constexpr int BLOCK = 272, PIECES = 17, GROUPS = 8;
    static constexpr bool DIRECT = true, HALVES = false;
    struct Row { u32x2 q[8]; };
    template <int MT, class X>
    static __device__ __forceinline__ void factors(const uint8_t *wl, int j, int c, float *ex, const X &, float4v (&)[MT]) {
#pragma unroll
        for (int h = 0; h < 2; ++h) ex[(2 * c + h) * 16 + j] = half_bits_to_float(*(const uint16_t *)(wl + 34 * (2 * c + h)));
    }
    static __device__ __forceinline__ void load(const uint8_t *wl, int c, Row &r) {
#pragma unroll
        for (int t = 0; t < 8; ++t) r.q[t] = *(const u32x2_a2 *)(wl + 34 * t + 2 + 8 * c);
    }
    static __device__ __forceinline__ long operand(const Row &r, int t, int) { return rows_pack(r.q[t].x, r.q[t].y); }
};

// Q4_0: eight 18-byte blocks; the operand is 16 (level - 8): the nibble in the upper half of a byte, its top bit flipped
template <bool GGML>
struct RowsQ4_0 {
    static constexpr int BLOCK = 144, PIECES = 9, GROUPS = 8;
    static constexpr bool DIRECT = true, HALVES = false;
    struct Row { u32x2 q[8]; };
    template <int MT, class X>
    static __device__ __forceinline__ void factors(const uint8_t *wl, int j, int c, float *ex, const X &, float4v (&)[MT]) {
#pragma unroll
        for (int h = 0; h < 2; ++h) ex[(2 * c + h) * 16 + j] = 0.0625f * half_bits_to_float(*(const uint16_t *)(wl + 18 * (2 * c + h)));
    }
    static __device__ __forceinline__ void load(const uint8_t *wl, int c, Row &r) {
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            if (GGML) r.q[t] = *(const u32x2_a2 *)(wl + 18 * t + 2 + 8 * (c & 1));
            else r.q[t].x = *(const u32_a2 *)(wl + 18 * t + 2 + 4 * c);
        }
    }
    static __device__ __forceinline__ long operand(const Row &r, int t, int c) {
        const uint32_t M = 0xF0F0F0F0u, TOP = 0x80808080u;
        if (GGML) {
            const int sh = c < 2 ? 4 : 0;
            return rows_pack(((r.q[t].x << sh) & M) ^ TOP, ((r.q[t].y << sh) & M) ^ TOP);
        }
        const uint32_t l = ((r.q[t].x << 4) & M) ^ TOP, h = (r.q[t].x & M) ^ TOP;  // byte i: values 2i and 2i + 1
        return rows_pack(__builtin_amdgcn_perm(h, l, 0x05010400u), __builtin_amdgcn_perm(h, l, 0x07030602u));
    }
};

// Q6_K: blocks of 210 bytes start on any even address, which a direct load does not take: they come through registers, 14
// pieces a row (the last one ends 14 bytes into the next block), 15 from row to row for the banks.  A sub-block's two groups of 16 have a
// scale each: two products whose operand is zero in the other half.
struct RowsQ6K {
    static constexpr int BLOCK = 210, PIECES = 15, GROUPS = 17;
    static constexpr bool DIRECT = false, HALVES = true;
    struct Row { u32x2 ql[4], qh[2]; };
    template <int MT, class X>
    static __device__ __forceinline__ void factors(const uint8_t *wl, int j, int c, float *ex, const X &, float4v (&)[MT]) {
        // the sixteen scales as integers, then d
        const uint32_t sc = *(const uint32_t *)(wl + 192 + 4 * c);
#pragma unroll
        for (int i = 0; i < 4; ++i) ((int *)ex)[(4 * c + i) * 16 + j] = (int)(sc << (24 - 8 * i)) >> 24;
        if (c == 0) ex[16 * 16 + j] = 0.25f * half_bits_to_float(*(const uint16_t *)(wl + 208));
    }
    static __device__ __forceinline__ void load(const uint8_t *wl, int c, Row &r) {
#pragma unroll
        for (int ip = 0; ip < 2; ++ip) {
            r.ql[2 * ip] = *(const u32x2 *)(wl + 64 * ip + 8 * c);
            r.ql[2 * ip + 1] = *(const u32x2 *)(wl + 64 * ip + 32 + 8 * c);
            r.qh[ip] = *(const u32x2 *)(wl + 128 + 32 * ip + 8 * c);
        }
    }
    static __device__ __forceinline__ long operand(const Row &r, int t, int) {
        const u32x2 ql = r.ql[2 * (t >> 2) + (t & 1)], qh = r.qh[t >> 2];
        const int quarter = t & 3;
        uint32_t w2[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            // 4 (level - 32): the level in the upper six bits of a byte, its top bit flipped
            const uint32_t nib = quarter & 2 ? (ql[e] >> 2) & 0x3C3C3C3Cu : (ql[e] << 2) & 0x3C3C3C3Cu;
            w2[e] = (nib | ((qh[e] << (6 - 2 * quarter)) & 0xC0C0C0C0u)) ^ 0x80808080u;
        }
        return rows_pack(w2[0], w2[1]);
    }
};

template <class F, int RF, int MT, int WAVES>
struct RowsLds {
    static constexpr int LOADED = F::DIRECT ? F::PIECES : F::PIECES - 1;  // pieces of a row that are fetched
    static constexpr int IT = (16 * LOADED + 63) / 64;          // loads per slot
    static constexpr int SLOT = 16 * F::PIECES * 16;
    static constexpr int EX = F::GROUPS * 16 * 4;
    static constexpr int WAVE = (F::DIRECT ? 2 : 1) * SLOT + EX;
    static constexpr int SUMS = WAVES * RF * MT * 1024;
    static constexpr int BYTES = WAVES * WAVE > SUMS ? WAVES * WAVE : SUMS;
};

template <class F, int RF, int MT, int WAVES, bool PAIRS>
__global__ __launch_bounds__(WAVES * 64, (WAVES == 16 || MT + F::HALVES <= 2) ? 4 : 2) void k_rows_i8(
    const uint8_t *__restrict__ xfrag, const float *__restrict__ xd, const float *__restrict__ xm, int K, int M, int frag_stride,
    int scale_stride, const RowsJobs jobs) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass knows no buffer descriptors
    static_assert(!PAIRS || MT == 1, "eight rows");
    typedef RowsLds<F, RF, MT, WAVES> L;
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), j = lane & 15, c = lane >> 4;
    uint8_t *const mine = smem + wave * L::WAVE;
    float *const ex = (float *)(mine + (F::DIRECT ? 2 : 1) * L::SLOT);
    const int ji = (int)(blockIdx.x >= (unsigned)jobs.j[0].wg_end) + (int)(blockIdx.x >= (unsigned)jobs.j[1].wg_end);
    const RowsJob job = jobs.j[ji];
    const int wg = blockIdx.x - (ji > 0 ? jobs.j[ji - 1].wg_end : 0);
    const int n0 = wg * (16 * RF), N = job.N, nsb = K >> 8;
    const uint32_t rb = (uint32_t)nsb * F::BLOCK;
    const int count = (nsb - wave + WAVES - 1) / WAVES;  // super-blocks wave, wave + WAVES, ... (may be none)
    xfrag += (size_t)blockIdx.y * MT * frag_stride;
    xd += (size_t)blockIdx.y * MT * scale_stride;
    xm += (size_t)blockIdx.y * MT * scale_stride;

    // a strip past the last row is moved back onto the rows that are there; its rows in front of n0 + 16 r are not stored
    auto strip_row = [&](int r) __attribute__((always_inline)) { return min(n0 + 16 * r, N - 16); };
    uint32_t from[L::IT];  // of a lane's piece, from the strip's first row and super-block
#pragma unroll
    for (int it = 0; it < L::IT; ++it) {
        const int e = min(it * 64 + lane, 16 * L::LOADED - 1);
        from[it] = (uint32_t)(e / L::LOADED) * rb + (uint32_t)(e % L::LOADED) * 16;
    }
    u32x4 held[F::DIRECT ? 1 : L::IT];
    auto request = [&](int sb, int r, int slot) __attribute__((always_inline)) {
        const uint8_t *base = job.W + (size_t)strip_row(r) * rb + (size_t)sb * F::BLOCK;
#pragma unroll
        for (int it = 0; it < L::IT; ++it) {
            if constexpr (!F::DIRECT) {
                held[it] = *(const u32x4_a2 *)(base + from[it]);
            } else if ((it + 1) * 64 <= 16 * F::PIECES || it * 64 + lane < 16 * F::PIECES) {
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(base + from[it]),
                                                 (__attribute__((address_space(3))) void *)(mine + slot * L::SLOT + it * 1024), 16, 0, 0);
            }
        }
    };
    auto park = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int it = 0; it < L::IT; ++it) {
            const int e = min(it * 64 + lane, 16 * L::LOADED - 1);  // lanes past the last piece write it once more
            *(u32x4 *)(mine + (e / L::LOADED) * (F::PIECES * 16) + (e % L::LOADED) * 16) = held[it];
        }
    };
    std::conditional_t<PAIRS, RowsPairs<F::HALVES>, RowsX<MT>> x;
    const int group = j >> 3;  // PAIRS: of columns
    // PAIRS: what a column does not take is asked for past the image's end, and comes as zero
    constexpr uint32_t NOTHING = 0x80000000u;
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)xfrag, 0, frag_stride, 0x00027000);
    const uint32_t mine_at = ((uint32_t)(j & 7) + 16 * c) * 16;
    const uint32_t at_half = c >> 1 == group ? mine_at : NOTHING;
    auto load_x = [&](int sb) __attribute__((always_inline)) {
        if constexpr (PAIRS) {
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                if constexpr (F::HALVES) {
                    x.q[p] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, at_half + p * 1024, sb * 4096, 0));
                } else {
                    const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, mine_at + p * 1024, sb * 4096, 0));
                    x.even[p] = group == 0 ? u32x2{v.x, v.y} : u32x2{0, 0};
                    x.odd[p] = group == 1 ? u32x2{v.z, v.w} : u32x2{0, 0};
                }
            }
            const float *pd = xd + (size_t)sb * 128 + (j & 7) * 8, *pm = xm + (size_t)sb * 128 + (j & 7) * 8 + 2 * c;
            const float4 a = *(const float4 *)pd, b = *(const float4 *)(pd + 4);
            if constexpr (F::HALVES) {
                x.d[0] = a.x; x.d[1] = a.y; x.d[2] = a.z; x.d[3] = a.w; x.d[4] = b.x; x.d[5] = b.y; x.d[6] = b.z; x.d[7] = b.w;
            } else {
                x.d[0] = group ? a.y : a.x; x.d[1] = group ? a.w : a.z; x.d[2] = group ? b.y : b.x; x.d[3] = group ? b.w : b.z;
            }
            const float2 v = *(const float2 *)pm;
            x.m[0] = group == 0 ? float2{v.x, 0.0f} : float2{0.0f, v.y};  // with the products that it is taken off
        } else
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const uint8_t *pf = xfrag + (size_t)t * frag_stride + (size_t)sb * 4096;
            const float *pd = xd + (size_t)t * scale_stride + (size_t)sb * 128, *pm = xm + (size_t)t * scale_stride + (size_t)sb * 128;
#pragma unroll
            for (int p = 0; p < 4; ++p) x.q[t][p] = *(const u32x4 *)(pf + p * 1024 + lane * 16);
            x.d[t][0] = *(const float4 *)(pd + j * 8);
            x.d[t][1] = *(const float4 *)(pd + j * 8 + 4);
            x.m[t] = *(const float2 *)(pm + j * 8 + 2 * c);
        }
    };
    float4v acc[RF][MT];
#pragma unroll
    for (int r = 0; r < RF; ++r)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[r][t] = float4v{0.f, 0.f, 0.f, 0.f};

    if (count > 0) {
        request(wave, 0, 0);
        load_x(wave);
        int slot = 0;
        for (int k = 0; k < count; ++k) {
            const int sb = wave + WAVES * k;
#pragma unroll
            for (int r = 0; r < RF; ++r) {
                if constexpr (F::DIRECT) {
                    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // this slot has landed; the other one's reads are over
                } else {
                    park();
                    rows_lds_fence();
                }
                if (r + 1 < RF) request(sb, r + 1, slot ^ 1);
                else if (k + 1 < count) request(sb + WAVES, 0, slot ^ 1);
                const uint8_t *wl = mine + slot * L::SLOT + j * (F::PIECES * 16);
                F::template factors<MT, decltype(x)>(wl, j, c, ex, x, acc[r]);
                typename F::Row row;
                F::load(wl, c, row);
                rows_lds_fence();
                // Q6_K: the super-block's sum in front of d (PAIRS: of every second sub-block, for a shorter chain of roundings: the
                // columns' sums meet in one rounding more)
                constexpr int PARTS = F::HALVES ? (PAIRS ? 2 : MT) : 1;
                float4v part[PARTS];
                if constexpr (F::HALVES) {
#pragma unroll
                    for (int mt = 0; mt < PARTS; ++mt) part[mt] = float4v{0.f, 0.f, 0.f, 0.f};
                }
                if constexpr (PAIRS && F::HALVES) {
#pragma unroll
                    for (int t = 0; t < 8; ++t) {
                        if (t % 2 == 0) {
                            asm volatile("" : "+v"(part[0]), "+v"(part[PARTS - 1]));
                            __builtin_amdgcn_sched_barrier(0);
                        }
                        const u32x4 v = x.q[t >> 1];
                        const long b = t & 1 ? rows_pack(v.z, v.w) : rows_pack(v.x, v.y);
                        const int4v d = __builtin_amdgcn_mfma_i32_16x16x32_i8(F::operand(row, t, c), b, int4v{0, 0, 0, 0}, 0, 0, 0);
                        const int4v f = *(const int4v *)&ex[(2 * t + group) * 16 + 4 * c];
#pragma unroll
                        for (int i = 0; i < 4; ++i) part[t & 1][i] += x.d[t] * (float)__mul24(d[i], f[i]);
                    }
                } else if constexpr (PAIRS) {
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        if (p % 2 == 0) {
                            asm volatile("" : "+v"(acc[r][0]));
                            __builtin_amdgcn_sched_barrier(0);
                        }
                        int4v d = __builtin_amdgcn_mfma_i32_16x16x32_i8(F::operand(row, 2 * p, c), rows_pack(x.even[p].x, x.even[p].y),
                                                                        int4v{0, 0, 0, 0}, 0, 0, 0);
                        d = __builtin_amdgcn_mfma_i32_16x16x32_i8(F::operand(row, 2 * p + 1, c), rows_pack(x.odd[p].x, x.odd[p].y), d, 0, 0, 0);
                        const float4v f = *(const float4v *)&ex[(2 * p + group) * 16 + 4 * c];
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc[r][0][i] += (f[i] * x.d[p]) * (float)d[i];
                    }
                } else
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    constexpr int TOGETHER = MT == 1 ? (F::HALVES ? 2 : 4) : MT == 2 && !F::HALVES ? 2 : 1;
                    if (t % TOGETHER == 0) {  // the sums so far are made here, not all behind the last product
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt) {
                            if constexpr (F::HALVES) asm volatile("" : "+v"(part[mt]));
                            else asm volatile("" : "+v"(acc[r][mt]));
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    const long a = F::operand(row, t, c);
                    if constexpr (F::HALVES) {
                        const long a_lo = c < 2 ? a : 0, a_hi = c < 2 ? 0 : a;
                        const int4v fl = *(const int4v *)&ex[(2 * t) * 16 + 4 * c], fh = *(const int4v *)&ex[(2 * t + 1) * 16 + 4 * c];
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt) {
                            const long b = rows_b(x.q[mt], t);
                            const int4v dl = __builtin_amdgcn_mfma_i32_16x16x32_i8(a_lo, b, int4v{0, 0, 0, 0}, 0, 0, 0);
                            const int4v dh = __builtin_amdgcn_mfma_i32_16x16x32_i8(a_hi, b, int4v{0, 0, 0, 0}, 0, 0, 0);
                            const float dx = rows_d(x.d[mt], t);
#pragma unroll
                            for (int i = 0; i < 4; ++i)  // |dot| <= 2^18, in fours, |scale| <= 2^7: exact
                                part[mt][i] += dx * (float)(__mul24(dh[i], fh[i]) + __mul24(dl[i], fl[i]));
                        }
                    } else {
                        const float4v f = *(const float4v *)&ex[t * 16 + 4 * c];
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt) {
                            const int4v d = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, rows_b(x.q[mt], t), int4v{0, 0, 0, 0}, 0, 0, 0);
                            const float dx = rows_d(x.d[mt], t);
#pragma unroll
                            for (int i = 0; i < 4; ++i) acc[r][mt][i] += (f[i] * dx) * (float)d[i];  // Q8_0, Q4_0: f * dx is exact
                        }
                    }
                }
                if constexpr (PAIRS && F::HALVES) part[0] += part[PARTS - 1];
                if constexpr (F::HALVES) {
                    const float4v d = *(const float4v *)&ex[16 * 16 + 4 * c];
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) acc[r][mt] += d * part[mt];
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) asm volatile("" : "+v"(acc[r][mt]));
                rows_lds_fence();  // the factors' place is rewritten next
                __builtin_amdgcn_sched_barrier(0);
                if (F::DIRECT) slot ^= 1;
            }
            if (k + 1 < count) load_x(sb + WAVES);
        }
    }
    __syncthreads();  // the slots are consumed
    float4v *const sums = (float4v *)smem;  // [wave][RF][MT][lane]
#pragma unroll
    for (int r = 0; r < RF; ++r)
#pragma unroll
        for (int t = 0; t < MT; ++t) sums[((wave * RF + r) * MT + t) * 64 + lane] = acc[r][t];
    __syncthreads();
    for (int f = wave; f < RF * MT; f += WAVES) {
        const int r = f / MT, t = f - r * MT;
        float4v p[WAVES];
#pragma unroll
        for (int w = 0; w < WAVES; ++w) p[w] = sums[(w * RF * MT + f) * 64 + lane];
#pragma unroll
        for (int d = 1; d < (PAIRS && F::HALVES ? WAVES / 2 : WAVES); d *= 2)  // neighbours first: a shorter chain of roundings
#pragma unroll
            for (int w = 0; w < WAVES; w += 2 * d) p[w] += p[w + d];
        float4v s = p[0];
        // PAIRS: and the same of the row's other column (row_ror:8).  Q6_K: the last two sums and theirs in one rounding, against the
        // rounding more that sums from twice the columns have (the others' chains of a super-block are half as long)
        if constexpr (PAIRS && F::HALVES) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const double v = (double)p[0][i] + (double)p[WAVES / 2][i];
                const uint64_t bits = __builtin_bit_cast(uint64_t, v);
                const uint32_t lo = (uint32_t)dpp_move_i<0x128>((int)(uint32_t)bits), hi = (uint32_t)dpp_move_i<0x128>((int)(uint32_t)(bits >> 32));
                s[i] = (float)(v + __builtin_bit_cast(double, (uint64_t)hi << 32 | lo));
            }
        } else if constexpr (PAIRS) {
#pragma unroll
            for (int i = 0; i < 4; ++i) s[i] += dpp_move<0x128>(s[i]);
        }
        const int m = (blockIdx.y * MT + t) * 16 + j, own = n0 + 16 * r, n = strip_row(r) + 4 * c;  // weight rows n .. n + 3
        if (m >= M) continue;
        float *dst = job.y + (size_t)m * N + n;
        const float *res = job.res ? job.res + (size_t)m * N + n : nullptr;  // may be y: read before the store
        if (n >= own && (N & 3) == 0) {
            if (res) s = *(const float4v *)res + s;
            *(float4v *)dst = s;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (n + i >= own) dst[i] = res ? res[i] + s[i] : s[i];
        }
    }
#endif
}

template <class F, int RF, int MT, int WAVES, bool PAIRS = false>
static int launch_rows_cfg(candy_hip_device *dev, const RowsLaunch &L, int64_t m) {
    typedef RowsLds<F, RF, MT, WAVES> S;
    static_assert(S::BYTES <= 160 * 1024, "LDS");
    RowsJobs jobs{};
    int total = 0;
    for (int i = 0; i < 3; ++i) {
        if (i < L.n) {
            jobs.j[i].W = (const uint8_t *)L.w[i]->data;
            jobs.j[i].y = L.y[i];
            jobs.j[i].res = L.res[i];
            jobs.j[i].N = (int)L.w[i]->rows;
            total += (jobs.j[i].N + 16 * RF - 1) / (16 * RF);
        }
        jobs.j[i].wg_end = total;
    }
    const int K = (int)L.w[0]->cols;
    auto kern = k_rows_i8<F, RF, MT, WAVES, PAIRS>;
    if (S::BYTES > 48 * 1024)
        CANDY_HIP_TRY(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, S::BYTES));
    hipLaunchKernelGGL(kern, dim3((unsigned)total, (unsigned)((m + 16 * MT - 1) / (16 * MT))), dim3(WAVES * 64), S::BYTES, dev->stream,
                       L.x.frag, L.x.d, L.x.m, K, (int)m, (int)L.x.frag_stride, (int)L.x.scale_stride, jobs);
    CANDY_LAUNCH_CHECK();
    return CANDY_HIP_OK;
}

template <class F>
static int launch_rows_fmt(candy_hip_device *dev, const RowsLaunch &L, int64_t m, int rf, int mt, int waves) {
#define CANDY_ROWS(RF, MT, WAVES)                                                                                  \
    if (rf == RF && mt == MT && waves == WAVES) {                                                                  \
        if constexpr (MT == 1)                                                                                     \
            if (m <= 8) return launch_rows_cfg<F, RF, MT, WAVES, true>(dev, L, m);                                 \
        return launch_rows_cfg<F, RF, MT, WAVES>(dev, L, m);                                                       \
    }
    CANDY_ROWS(1, 1, 16) CANDY_ROWS(1, 1, 8)
    if constexpr (std::is_same<F, RowsQ6K>::value) {
        CANDY_ROWS(2, 1, 8)
    } else {
        CANDY_ROWS(4, 1, 8)
    }
    CANDY_ROWS(1, 2, 8) CANDY_ROWS(1, 3, 8) CANDY_ROWS(2, 3, 8)
    if constexpr (std::is_same<F, RowsQ6K>::value) {
        CANDY_ROWS(1, 4, 8) CANDY_ROWS(2, 4, 8)
    } else {
        CANDY_ROWS(1, 2, 16) CANDY_ROWS(2, 2, 16) CANDY_ROWS(2, 2, 8)
    }
#undef CANDY_ROWS
    return fail(CANDY_HIP_ERR_INVALID, "internal: shape of the row contraction");
}

bool rows_i8_covers(const candy_hip_qtensor *w) {
    if (w->cols % 256 != 0 || w->cols > (1 << 20) || w->rows < 16 || w->rows > 0x7FFFFFF || ((uintptr_t)w->data & (w->fmt == CANDY_HIP_Q6_K ? 1 : 15)) != 0)
        return false;
    switch (w->fmt) {
    case CANDY_HIP_Q4_K: case CANDY_HIP_Q5_K: case CANDY_HIP_Q8_0: case CANDY_HIP_Q4_0: case CANDY_HIP_Q4_0_GGML: return true;
    case CANDY_HIP_Q6_K: return w->padded;  // the last piece of a row ends up to 14 bytes behind it
    default: return false;
    }
}

// Super-blocks that a weight row must have for the kernel to be ahead.  With fewer than eight, wavefronts have none and only meet the
// others at the end; past a round or two of workgroups that is most of the time.  Speed of the kernels that were there / this one:
//   Q5_K 16000 x 256, 33 rows 0.57, 32000 x 512, 5 / 17 / 33 rows 0.81, 0.82, 0.55, 32000 x 768 1.00, 1.01, 0.69, 64000 x 1536 1.07, 1.28, 0.91
//   Q6_K 12000 x 512, 5 / 17 rows 2.2, 0.74, 16000 x 1280 1.01, 0.81, 32000 x 1024 0.92, 0.94, 64000 x 1536 0.98, 0.96
//   Q8_0 16000 x 256, 8 / 17 / 33 rows 1.9, 0.84, 0.62, 24000 x 512 2.4, 1.02, 0.85, 32000 x 1024 2.2, 1.61, 1.02 (Q4_0 2.7, 1.5, 0.90)
// Up to eight rows of Q8_0 and Q4_0, and three and four rows at all, the alternative is the looping vector kernel, far behind there.
static int64_t least_blocks(const candy_hip_qtensor *w, int64_t m) {
    const int64_t cus = w->dev->num_cus, strips = (w->rows + 15) / 16;
    const bool q5 = w->fmt == CANDY_HIP_Q5_K, q6 = w->fmt == CANDY_HIP_Q6_K, q8 = w->fmt == CANDY_HIP_Q8_0;
    if (w->fmt == CANDY_HIP_Q4_K) return 1;  // its one-pass kernel is asked first
    if (m <= 4) return !(q5 || q6) || strips <= 10 * cus ? 1 : strips <= 20 * cus ? 3 : 6;
    if (m <= 8 && !q5 && !q6) return 1;
    if (strips <= 2 * cus) return m > 8 ? 2 : 1;
    if (strips <= 4 * cus) return m > 16 ? (q6 ? 7 : q5 ? 3 : 2) : m > 8 || strips > 3 * cus ? 2 : 1;
    if (m <= 16) return q6 && strips > 7 * cus ? 6 : q5 || q6 ? 4 : 3;
    if (m <= 32) return q6 ? 7 : q5 ? 3 : 2;
    const bool far = strips > 7 * cus;
    return q5 || q6 ? (far ? 7 : 4) : q8 ? (far ? 4 : 3) : far ? 6 : 4;
}

// Below 16 activation rows the length of the weight rows is limited by the vector kernels, whichever kernel is ahead: a batch that
// one row more or less would have refused is not taken here either (matvec.hip takes it where its tiles do).
bool rows_i8_takes(const candy_hip_qtensor *w, int64_t m) {
    const Options &o = w->dev->opt;
    if (m < 16 && !matvec_row_fits(w->cols)) return false;
    if (m < o.i8_min_m || o.small_batch_kernel == 0) return false;  // comparison runs that ask for the vector kernels
    if (!o.rows_i8 || o.mmv_max_m == 0 || o.mmq_fp16_only || m < 3 || m > 255 || !rows_i8_covers(w)) return false;
    return o.rows_i8 == 2 || (w->cols >> 8) >= least_blocks(w, m);
}

// Whether launches of four strips of weight rows per workgroup leave a tenth or more of the chip's two slots a CU idle: just past a
// whole round (1025 to 1840 strips, 2049 to 2560).
static bool four_strips_idle(int64_t strips, int64_t cus) {
    const int64_t wgs = (strips + 3) / 4, slots = 2 * cus;
    return strips > 4 * cus && strips <= 10 * cus && 10 * wgs < 9 * slots * ((wgs + slots - 1) / slots);
}

// Quants that are planar already (candy_hip_qmatmul_qact) take a launch more here, which orders them, and none on the vector kernels and
// the tiles.  Speed of those / this one, 3 / 5 rows where there are two: Q8_0 4096 x 4096 0.70, 1.04, 2048 x 4096 0.58, 0.91; Q5_K 11008 x
// 4096 0.85, 1.50, 4096 x 8192 1.27, 1.29, 24576 x 2048 1.26, 2048 x 4096, 5 rows 0.91; Q6_K 4096 x 4096 0.94, 1.21, 16384 x 2048 0.95, 0.98,
// 11008 x 4096 1.10; Q4_K 4096 x 11008 0.90, 1.45, 4096 x 14336 1.38, 1.35, 24576 x 2048 1.37; 10 rows of 1024 x 2048 0.84 (launches only), of
// 24576 x 1024, short rows, 0.82 to 0.87.
static bool planar_behind(const candy_hip_qtensor *w, int64_t m) {
    const int64_t values = w->rows * w->cols, cols = w->cols, cus = w->dev->num_cus;
    const bool q4k = w->fmt == CANDY_HIP_Q4_K, q6k = w->fmt == CANDY_HIP_Q6_K, k_quant = q4k || q6k || w->fmt == CANDY_HIP_Q5_K;
    if (m <= 4) {
        if (!k_quant || (values < 1 << 24 && cols <= 12288)) return true;
        return q6k ? values < 40000000 && cols <= 4096 : values < 100000000 && w->rows < 20000 && cols <= (q4k ? 12288 : 5632);
    }
    if (m <= 16 && k_quant && cols < 2048 && w->rows > (q6k ? 32 : q4k && m <= 8 ? 120 : 48) * cus) return true;
    if (m <= 8) return !q4k && !q6k && values <= 1 << 23 && cols <= 4096 && w->rows <= (k_quant ? 2048 : 4096);
    return m <= 16 && values <= 1 << 22 && cols <= 2560;
}

// Weights of 2 million values and more that are too few rows for the fp16 kernels, which launch a workgroup for 128 weight rows
// (mmq_f16_rows.hip: 16 to 48, from 2048 on) and sum copies of a split of K: this kernel deals K to its wavefronts, strips of 16.  us
// of a call there / here: Q4_K 1024 x 4096, 48 / 96 / 255 rows 14.1 / 7.9, 15.7 / 9.2, 20.8 / 13.0; 2048 x 8192, 48 / 128 rows 19.4 /
// 11.9, 22.1 / 17.4; 4096 x 11008, 64 rows 26.8 / 21.5; 3000 x 2560, 160 / 255 rows 18.8 / 14.5, 22.6 / 19.0; Q6_K 1024 x 4096, 48 /
// 255 rows 15.8 / 8.0, 24.0 / 15.5, 2048 x 8192, 64 rows 21.7 / 16.2; Q8_0 2048 x 4096, 128 rows 22.7 / 13.3.  The vector ALU's work
// per product is what ends it, `work` below, for Q6_K at two thirds (Q4_K 2.1 and 2.7 billion: 2048 x 8192, 128 / 160 rows 22.1 /
// 17.4, 25.5 / 26.2; 2.0 and 2.4: 1536 x 8192, 160 / 192 rows 23.2 / 17.5, 23.9 / 26.0; Q6_K 1.5 and 1.8: 2048 x 5632, 128 / 160 rows
// 23.5 / 19.1, 23.8 / 27.7).  Below 33 rows and with a lower threshold a caller has asked for the fp16 kernels, with a shape or a
// split for theirs.
static bool ahead_of_fp16(const candy_hip_qtensor *w, int64_t m) {
    const Options &o = w->dev->opt;
    const int64_t rows = w->rows, cus = w->dev->num_cus, values = rows * w->cols, work = values * m;
    const bool q4k = w->fmt == CANDY_HIP_Q4_K, q6k = w->fmt == CANDY_HIP_Q6_K;
    if (o.f16_api_min_m < 33 || o.f16_shape || o.f16_split || values < 1 << 21) return false;
    if (rows <= 6 * cus) return work <= (q6k ? 1450000000 : 2200000000);
    // from here mmq_f16_rows.hip has the short rows of small batches
    if (rows <= 8 * cus) return (values >= 1 << 22 || m > 128) && work <= (q6k ? 1450000000 : 2000000000);
    if (rows > 16 * cus) return false;
    if (m > 128) return q6k ? values <= 1 << 22 : work <= 2050000000;
    if (mmq_f16_rows_covers(w, m)) return false;
    return m > 96 ? w->cols <= 4096 : m <= 64 && q4k;
}

// Where the other kernels are ahead or level, us of a call, there / here:
//   Q4_K up to 16 (8192 or fewer weight rows: 32) activation rows of 4096 or fewer values, the one-shot kernel of mmv_i8.hip:
//     4096 x 4096, 16 rows 7.1 / 7.2, 14336 x 4096 11.2 / 12.1, 8192 x 2048, 32 rows 7.7 / 8.0 (but 32000 x 4096 19.6 / 17.8, 14336 x
//     4096, 32 rows 16.4 / 15.1, 4096 x 11008, 16 rows 11.1 / 9.7).  Further on only where this kernel's grid leaves slots idle
//     (16400 x 4096, 3 rows 0.81 of that kernel's speed, 20000 x 2048, 16 rows 0.79, 24576 x 4096 0.95), at seven and eight super-blocks,
//     a step of its wavefronts (64000 x 2048, 3 / 8 / 16 rows 0.93, 0.98, 1.02; 12000 x 2048, 32 rows 0.95), and of 29 to 32
//     super-blocks, two for each of its wavefronts, where a strip a CU is all there is: 2048 x 8192, 3 / 8 / 16 rows 7.7 / 8.3, 7.8 / 8.8,
//     7.8 / 8.2 (but 28 super-blocks level, 33 10.2 / 8.0, 5120 x 8192, 16 rows 11.2 / 10.2).  Planar quants do not go there.
//   three and four rows, the vector kernels: small weights (1024 x 4096, Q5_K 7.2 / 7.2, Q8_0 7.3 / 7.6), and Q8_0 and Q4_0 in two rounds
//     of workgroups whose few super-blocks are soon done (14336 x 4096 15.5 / 18.7 and 12.7 / 15.0, 8208 x 5120 0.89 of the vector
//     kernels' speed, 8208 x 8192 1.01; 4096 x 4096 8.4 / 7.7), where four strips a workgroup leave slots idle (16400 x 4096 0.73 and
//     0.75, 24576 x 8192 0.88 and 0.82, 32000 x 4096 1.01 and 1.05), and Q4_0, three rows of 2304 to 5120 values, in less than one round
//     (5000 x 4096 0.88)
//   the fp16 kernels, whose scales are in the operands, where a call may take them (mmq.f16_api_min_m): Q4_K and Q6_K from 33 rows
//     (11008 x 4096, 48 rows 16.0 / 20.9 and 26.0 / 26.4), the others from 65 (Q8_0 11008 x 4096, 64 rows 44.5 / 24.4, 80 rows 24.7 /
//     35.8); not small weights, where this one is ahead (ahead_of_fp16)
// Weights under a million values are launches and nothing else whatever the kernel.
// Not left to a faster kernel: Q8_0 and Q4_0 whose results come to four million and more (planar quants and prompts of up to 255 rows,
// single calls of up to 64 against 44000 weight rows), which the fp16 tiles of mmq.hip took before (32000 x 4096, 200 rows 119 us
// there, 176 here; 100 rows 109 and 105).  Below the fp16 thresholds every product is exact, and this is the fastest kernel that is.
bool rows_i8_picks(const candy_hip_qtensor *w, int64_t m, bool exact) {
    const Options &o = w->dev->opt;
    const int64_t values = w->rows * w->cols, cus = w->dev->num_cus, strips = (w->rows + 15) / 16, nsb = w->cols >> 8;
    if (!rows_i8_takes(w, m)) return false;
    if (o.rows_i8 == 2) return true;
    if (values < 1 << 20) return false;
    const bool q4k = w->fmt == CANDY_HIP_Q4_K, q6k = w->fmt == CANDY_HIP_Q6_K;
    if (q4k && mmv_covers(w, m)) {
        const bool eight = nsb == 7 || nsb == 8;
        if (nsb <= 16 && w->rows <= (m <= 16 ? 64 * cus : 32 * cus)) return false;
        if (!exact && nsb > 2 && nsb <= 16 && m <= 16 && (four_strips_idle(strips, cus) || (eight && m <= 8))) return false;
        if (!exact && m > 16 && nsb > 4 && nsb <= 8 && w->rows <= 48 * cus) return false;
        if (!exact && nsb > 28 && nsb <= 32 && strips <= cus) return false;
    }
    if (exact && planar_behind(w, m)) return false;
    if (m <= 4 && values <= 1 << 22) return false;
    if (m <= 4 && !q4k && !q6k && w->fmt != CANDY_HIP_Q5_K) {  // Q8_0, Q4_0
        if (nsb <= 24 && strips > 2 * cus && strips <= 4 * cus) return false;
        if (nsb > 5 && four_strips_idle(strips, cus)) return false;
        if (w->fmt != CANDY_HIP_Q8_0 && m == 3 && nsb > 8 && nsb <= 20 && strips > cus && strips < 2 * cus) return false;
    }
    return exact || !mmq_f16_big_covers(w, m, o.f16_api_min_m) || ahead_of_fp16(w, m);
}

// Q6_K, more than 48 rows: the tile whose rounds of workgroups (one a CU at a time: the registers) cost the least.  us of a round against
// rows of 14336 values, and once, for strips x tiles of 2 x 4, 1 x 4, 1 x 3, 1 x 2 and 1 x 1; shorter rows are in proportion.  With two
// strips and four tiles from 65 rows on whatever the grid, half of the CUs idled against 2048 weight rows: us before / so / on the int8
// tiles 2048 x 8192, 100 rows 33.1 / 21.9 / 25.7, 1536 x 14336, 128 rows 54.6 / 33.8 / 33.5, 3072 x 8192, 192 rows 64.1 / 48.2 / 53.5, 5120 x
// 14336, 80 rows 99.9 / 72.6 / 85.0; ten weights x three lengths x ten batches 1.11 times as fast on the geometric mean.
static void rows_q6k_shape(int64_t strips, int64_t m, int64_t cus, int *rf, int *mt) {
    static const struct { int rf, mt; double round, once; } shapes[] = {{2, 4, 48, 6}, {1, 4, 27, 5}, {1, 3, 22, 6}, {1, 2, 17, 5}, {1, 1, 8.7, 7}};
    double best = 1e30;
    for (const auto &s : shapes) {
        const int64_t columns = (m + 16 * s.mt - 1) / (16 * s.mt), wgs = (strips + s.rf - 1) / s.rf * columns;
        const double us = s.once + s.round * (double)((wgs + cus - 1) / cus);
        if (columns * s.mt <= rows_tiles(m) && us < best) { best = us; *rf = s.rf; *mt = s.mt; }
    }
}

// Tile and wavefronts.  One activation tile per workgroup where the strips alone leave half of the CUs idle (weights read
// again come from L2), else the tiles that the registers hold.  Sixteen wavefronts where there is one workgroup per CU, eight (two
// workgroups) otherwise; two or four strips of weight rows per workgroup where a launch would otherwise be more than four
// (17 to 32 rows: three) rounds.  us: Q8_0 2048 x 8192, 32 rows, tiles of 16 / 32 rows 10.6 / 12.1, 4096 x 14336 25.1 / 20.3; 32000 x 4096,
// 16 rows, 1 / 2 / 4 strips 32.7 / 29.5 / 28.0; Q4_K 4096 x 14336, 6 rows, 16 / 8 wavefronts 11.7 / 13.5, 11008 x 4096 12.1 / 9.8.
int launch_rows_i8(candy_hip_device *dev, const RowsLaunch &L, int64_t m) {
    int64_t strips = 0;  // of 16 weight rows
    for (int i = 0; i < L.n; ++i) strips += (L.w[i]->rows + 15) / 16;
    const bool q6k = L.w[0]->fmt == CANDY_HIP_Q6_K;
    const int64_t cus = dev->num_cus, tiles = (m + 15) / 16;
    int rf, mt, waves;
    if (tiles == 1 || (strips <= cus / 2 && strips * tiles <= (q6k && m > 48 ? 1 : 2) * cus)) {
        mt = 1;
        rf = strips <= 4 * cus ? 1 : q6k ? 2 : 4;
        waves = strips * tiles <= cus ? 16 : 8;
    } else if (m <= 32 && q6k) {  // two tiles are 148 registers: eight wavefronts a CU, less than the weights' stream needs past 1024 strips
        mt = strips <= 4 * cus ? 2 : 1;
        rf = strips <= 4 * cus ? 1 : 2;
        waves = 8;
    } else if (m <= 32) {
        mt = 2;
        rf = strips <= 3 * cus ? 1 : 2;
        waves = strips <= cus ? 16 : 8;
    } else if (m <= 48) {
        mt = 3;
        rf = strips <= 4 * cus ? 1 : 2;
        waves = 8;
    } else if (q6k) {
        rows_q6k_shape(strips, m, cus, &rf, &mt);
        waves = 8;
    } else {
        mt = 2;
        rf = 2;
        waves = strips * ((m + 31) / 32) <= 2 * cus ? 16 : 8;
    }
    CANDY_REQUIRE((m + 16 * mt - 1) / (16 * mt) * mt <= rows_tiles(m), "internal: tiles of the row contraction");
    switch (L.w[0]->fmt) {
    case CANDY_HIP_Q4_K: return launch_rows_fmt<RowsQ45K<false>>(dev, L, m, rf, mt, waves);
    case CANDY_HIP_Q5_K: return launch_rows_fmt<RowsQ45K<true>>(dev, L, m, rf, mt, waves);
    case CANDY_HIP_Q6_K: return launch_rows_fmt<RowsQ6K>(dev, L, m, rf, mt, waves);
    case CANDY_HIP_Q8_0: return launch_rows_fmt<RowsQ8_0>(dev, L, m, rf, mt, waves);
    case CANDY_HIP_Q4_0: return launch_rows_fmt<RowsQ4_0<false>>(dev, L, m, rf, mt, waves);
    case CANDY_HIP_Q4_0_GGML: return launch_rows_fmt<RowsQ4_0<true>>(dev, L, m, rf, mt, waves);
    default: return fail(CANDY_HIP_ERR_INVALID, "internal: format of the row contraction");
    }
}

}  // namespace candy

// The rules above, for their tests (no device needed): bit 0 whether a single contraction goes here, bit 1 whether a prompt does.
extern "C" int candy_test_rows_i8(int fmt, int64_t rows, int64_t cols, int64_t m, int num_cus, int exact, int f16_api_min_m, int i8_min_m,
                                  int small_batch_kernel) {
    candy_hip_device dev;
    dev.num_cus = num_cus;
    dev.opt.f16_api_min_m = f16_api_min_m;
    dev.opt.i8_min_m = i8_min_m;
    dev.opt.small_batch_kernel = small_batch_kernel;
    candy_hip_qtensor w;
    w.dev = &dev; w.fmt = fmt; w.rows = rows; w.cols = cols; w.padded = true;
    return (candy::rows_i8_picks(&w, m, exact != 0) ? 1 : 0) | (candy::rows_i8_takes(&w, m) ? 2 : 0);
}
// Tile of a Q6_K launch of more than 48 rows: strips * 100 + tiles.
extern "C" int candy_test_rows_q6k_shape(int64_t weight_rows, int64_t m, int num_cus) {
    int rf = 0, mt = 0;
    candy::rows_q6k_shape((weight_rows + 15) / 16, m, num_cus, &rf, &mt);
    return rf * 100 + mt;
}

// Weights that share a launch, with residuals, for their tests: f32 rows x against n of them.
extern "C" int candy_test_rows_launch(candy_hip_device *dev, int n, const candy_hip_qtensor *const *ws, float *const *ys,
                                      const float *const *res, const float *x, int64_t m) {
    void *ws_p = nullptr;
    if (int rc = candy::use_device(dev)) return rc;
    if (int rc = candy::workspace(dev, candy::rows_image_bytes(m, ws[0]->cols), &ws_p)) return rc;
    candy::RowsLaunch L;
    L.n = n;
    L.x = candy::rows_image(ws_p, m, ws[0]->cols);
    for (int i = 0; i < n; ++i) { L.w[i] = ws[i]; L.y[i] = ys[i]; L.res[i] = res[i]; }
    if (int rc = candy::launch_rows_quantize(dev, x, m, ws[0]->cols, L.x)) return rc;
    return candy::launch_rows_i8(dev, L, m);
}

// The image as the norm (b: its weights) or the SiLU launch (b: up) writes it, and the planar quants of the same launch.
extern "C" int candy_test_rows_image(candy_hip_device *dev, int silu, const float *a, const float *b, int64_t m, int64_t cols, void *image,
                                     int8_t *qs, candy::Q8Scale *scales) {
    if (int rc = candy::use_device(dev)) return rc;
    const candy::RowsImage x = candy::rows_image(image, m, cols);
    for (const candy::RowsImage *to : {&x, (const candy::RowsImage *)nullptr})
        if (int rc = silu ? candy::launch_silu_mul_quant(dev, a, b, m, cols, nullptr, to ? nullptr : qs, to ? nullptr : scales, nullptr, to)
                          : candy::launch_rms_norm_quant(dev, a, b, 1e-5f, m, cols, nullptr, to ? nullptr : qs, to ? nullptr : scales, nullptr, to))
            return rc;
    return CANDY_HIP_OK;
}
