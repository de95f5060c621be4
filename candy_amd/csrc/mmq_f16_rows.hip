// 33 to 128 activation rows of Q4_K and Q6_K, 65 to 128 of Q5_K, Q8_0 and Q4_0, on the fp16 matrix cores, K dealt to wavefronts:
// y[m, N] = x[m, K] . W^T with the operands of mmq_f16.hip.
//
// With so few rows a contraction should last as long as its weights take from memory, but in the role-split tiles of
// mmq_f16.hip a step of K waits for a barrier and for the slower role (at 128 rows 1500 to 2200 cycles for 500 of matrix
// instructions), 128-row tiles are N / 128 x splits workgroups, and the split's copies are added by a launch of its own.
// Here nobody waits for anybody: a workgroup owns 16, 32 or 48 weight rows and all activation rows, and each of its eight
// wavefronts takes every eighth super-block of K: weight blocks by direct loads into its own slice of LDS, dequantized into
// matrix operands in registers, activation fragments straight from their image, each loaded by one wavefront of the
// workgroup.  The wavefronts' sums meet in LDS at the end, in the order of the wavefronts (reproducible).  us of a call, 77
// rows, 11008 x 4096, tiles -> here: Q4_K 28.1 -> 18.7, Q5_K 35.6 -> 19.1, Q6_K 31.4 -> 21.7, Q8_0 40.0 -> 22.7, Q4_0 38.2 -> 18.2; 2048 x
// 1024 Q8_0, the kernels with the split sum 17.1 -> 5.7.
// A step's second half of activations is requested in front of its dequantization, and held there: left alone the compiler
// dequantizes several steps in advance and requests the activations behind that, where nothing hides them.  A wavefront's loads are
// the same in number at every step, with weights to fetch or not (request()).  us of a call, without / with both: 11008 x 4096, 77
// rows Q8_0 24.9 / 22.7, Q4_0 21.9 / 19.7, Q5_K 25.1 / 21.9, Q4_K 20.2 / 17.7; 3000 x 2560 Q5_K 14.9 / 10.9; 8192 x 2048, 100 rows
// Q4_K 16.3 / 13.4 (4096 x 4096, 77 rows Q4_K 14.0 / 14.2).  Fences behind the first half's loads too, or the loads
// three halves ahead: 3 and 7 % slower.  What bounds it: without any weights or activations fetched the Q8_0 call takes 17.6 (a
// launch of the quantizer 2.5, dequantization and products of two wavefronts a SIMD, the sums), the activations, which every CU
// reads (655 KB), add 2 to 3, the weights (48 MB of Q8_0) the rest.
#include <algorithm>
#include <type_traits>

#include "f16_weights.h"
#include "internal.h"

namespace candy {

// 16-byte pieces that hold a super-block wherever it starts (Q6_K: 210 bytes, up to 14 behind the start of a piece)
template <class F>
constexpr int pieces() { return F::BLOCK % 16 == 0 ? F::BLOCK / 16 : (F::BLOCK + 14) / 16; }

// Activation fragments whose sums meet in LDS at a time: half of them where all would be more than its 160 KB
template <int RF, int MF>
constexpr int sums_at_once() { return RF * MF > 20 ? (MF + 1) / 2 : MF; }

template <class F, int RF, int MF>
constexpr size_t lds_bytes() {
    const size_t sums = (size_t)8 * RF * sums_at_once<RF, MF>() * 1024, slices = (size_t)8 * 1024 * ((RF * pieces<F>() + 3) / 4);
    return sums > slices ? sums : slices;
}

template <class F, int RF, int MF>
__global__ __launch_bounds__(512, 2) void k_mmq_f16_rows(const uint8_t *__restrict__ W, const _Float16 *__restrict__ xh, float *y,
                                                         const float *res, int M, int N, int K) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass knows no buffer descriptors
    constexpr bool WHOLE = F::BLOCK % 16 == 0;  // pieces
    extern __shared__ __align__(16) uint8_t smem_raw[];
    // [wave][RF][sums_at_once][lane]; of an odd MF in halves the last slot of the second half is not written, and its activation rows (from
    // 16 MF on) are not there
    float4v *sums = (float4v *)smem_raw;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, c = lane >> 4;
    const int n0 = blockIdx.x * (16 * RF), first = wave;
    const int count = ((K >> 8) - first + 7) >> 3;  // super-blocks first, first + 8, ... of this wavefront (may be none)
    const size_t rb = (size_t)(K >> 8) * F::BLOCK, xrow = (size_t)(K >> 5) * 512;
    const _Float16 *xl = xh + r16 * 32 + (F::RUN16 ? (c >> 1) * 512 + (c & 1) * 16 : c * 8);
    constexpr int HALF = F::RUN16 ? 8 : 512;  // from a step's first chunk of K to its second

    float4v acc[RF][MF];
#pragma unroll
    for (int i = 0; i < RF; ++i)
#pragma unroll
        for (int t = 0; t < MF; ++t) acc[i][t] = float4v{0.f, 0.f, 0.f, 0.f};
    // A super-block of the workgroup's rows comes into the wavefront's own slice of LDS, 16-byte pieces in the order they
    // lie in memory (requests of a lane for its own few bytes of a row cost the cache a line each: Q8_0 9 us per 16 rows of
    // 4096 and CU, against 3 for the bytes themselves); from there to registers, which frees the slice for the next one.
    // A Q6_K block (210 bytes) starts anywhere in its first piece: 14 pieces hold it wherever that is.  us of a call, nine requests of a lane
    // for its own bytes / staged: 4096 x 4096, 64 rows 15.9 / 12.7, 11008 x 4096, 48 rows 25.1 / 17.1, 8192 x 4096, 40 rows 18.8 / 12.8.
    constexpr int PIECES = pieces<F>(), IT = (RF * 16 * PIECES + 63) / 64;
    uint4 *slice = (uint4 *)smem_raw + wave * (IT * 64);
    uint32_t from[IT];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int e = it * 64 + lane, row = min(e / PIECES, RF * 16 - 1);
        from[it] = (uint32_t)(min(n0 + row, N - 1) - n0) * (uint32_t)rb + (uint32_t)(e % PIECES) * 16;
    }
    const uint8_t *w0 = W + (size_t)n0 * rb;
    // any false: the same loads from a matrix of no bytes, so that as many are in flight at every step: behind a branch around them
    // the compiler waits for the activations by the smaller count, which is a wait for the weights too
    auto request = [&](int sb, bool any) __attribute__((always_inline)) {
        const int at = any ? sb * F::BLOCK : 0;  // (a scalar offset past an empty matrix would count as inside)
        // pieces past the last block of a Q6_K matrix: no bytes; its end lies in an aligned word, which counts as a whole
        const int size = WHOLE ? (int)(RF * 16 * rb) : ((int)(min(RF * 16, N - n0) * rb) + 3) & ~3;
        const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void *)w0, 0, any ? size : 0, 0x00027000);
#pragma unroll
        for (int it = 0; it < IT; ++it)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (__attribute__((address_space(3))) void *)(slice + it * 64), 16,
                                                     WHOLE ? from[it] : (from[it] + (uint32_t)at) & ~15u, WHOLE ? at : 0, 0, 0);
    };
    if (count > 0) {
        typename F::Raw raw[RF];
        half8 xf[2][MF];
        auto load_w = [&](int sb) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < RF; ++i) {
                const int row = 16 * i + r16;
                const uint32_t behind = WHOLE ? 0 : ((uint32_t)(min(n0 + row, N - 1) - n0) * (uint32_t)rb + (uint32_t)(sb * F::BLOCK)) & 15;
                F::load((const uint8_t *)slice + row * (16 * PIECES) + behind, c, raw[i]);
            }
        };
        auto load_x = [&](int step, int h) __attribute__((always_inline)) {  // step: in 64s along K
            const _Float16 *p = xl + (size_t)step * 1024 + h * HALF;
#pragma unroll
            for (int t = 0; t < MF; ++t) xf[h][t] = *(const half8 *)(p + t * xrow);
        };
        auto contract = [&](int sb, int sb_next) __attribute__((always_inline)) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                load_x(sb * 4 + g, 1);
                __builtin_amdgcn_sched_barrier(0);  // and the loads are out
                half8 a[RF][2];
#pragma unroll
                for (int i = 0; i < RF; ++i) {
                    int k0, k1;
                    F::dequant(raw[i], g, c, a[i][0], a[i][1], k0, k1);
                }
#pragma unroll
                for (int t = 0; t < MF; ++t)
#pragma unroll
                    for (int i = 0; i < RF; ++i) acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i][0], xf[0][t], acc[i][t], 0, 0, 0);
                load_x(g == 3 ? sb_next * 4 : sb * 4 + g + 1, 0);
#pragma unroll
                for (int t = 0; t < MF; ++t)
#pragma unroll
                    for (int i = 0; i < RF; ++i) acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i][1], xf[1][t], acc[i][t], 0, 0, 0);
            }
        };
        request(first, true);
        load_x(first * 4, 0);
        for (int k = 0; k < count; ++k) {
            const int sb = first + 8 * k;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the slice has landed
            load_w(sb);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // and is in registers
            request(sb + 8, k + 1 < count);
            contract(sb, k + 1 < count ? sb + 8 : sb);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the last request writes its slice, which the sums are about to take
    }
    constexpr int MP = sums_at_once<RF, MF>();
#pragma unroll
    for (int t0 = 0; t0 < MF; t0 += MP) {
        __syncthreads();  // the slices, or the sums in front, are consumed
#pragma unroll
        for (int i = 0; i < RF; ++i)
#pragma unroll
            for (int t = 0; t < MP; ++t)
                if (t0 + t < MF) sums[((wave * RF + i) * MP + t) * 64 + lane] = acc[i][t0 + t];
        __syncthreads();
        for (int f = wave; f < RF * MP; f += 8) {
            const int m = (t0 + f % MP) * 16 + r16, n = n0 + (f / MP) * 16 + 4 * c;  // activation row; weight rows n .. n + 3
            float4v s = sums[f * 64 + lane];
#pragma unroll
            for (int k = 1; k < 8; ++k) s += sums[(k * RF * MP + f) * 64 + lane];
            if (m >= M) continue;
            float *dst = y + (size_t)m * N + n;
            const float *r = res ? res + (size_t)m * N + n : nullptr;  // may alias dst: read before the store
            if (n + 3 < N && (N & 3) == 0) {
                if (r) s = *(const float4v *)r + s;
                *(float4v *)dst = s;
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (n + j < N) dst[j] = r ? r[j] + s[j] : s[j];
            }
        }
    }
#endif
}

// of 16 activation rows.  97 to 112 rows on seven instead of eight: 8192 x 4096 Q4_K 24.1 -> 22.5 us, 4096 x 2048 Q8_0 14.0 -> 13.0
static int fragments(int64_t m) { return m <= 48 ? 3 : m <= 64 ? 4 : m <= 80 ? 5 : m <= 96 ? 6 : m <= 112 ? 7 : 8; }

// What a call takes, us, here and on the 128 x 128 tiles of mmq_f16.hip, the tiles 2 % below their fit: both fitted to 3729 calls (five
// formats, 2048 .. 12288 weight rows, K 512 .. 8192, 36 .. 128 activation rows; the fits are 3 to 6 % off on average).  A line on any
// one size does not divide them: a round of super-blocks that most wavefronts sit out, a split that leaves the tiles short, an odd
// number of 210-byte blocks (rows 2 bytes off) each move it.
struct RowsCost {
    // a launch; a tile's super-block; a split's launch; MB of its copies; 1000 super-blocks of all tiles
    float tile[5];
    // a launch; a round of super-blocks: weight fragment, activation fragment; a super-block: activation fragment (read by every CU),
    // weight fragment, the same of odd rows of Q6_K; the sums of a fragment pair; MB of results
    float rows[8];
};
static const RowsCost &rows_cost(int fmt) {
    static constexpr RowsCost Q4K{{7.74f, 1.16f, 2.49f, 0.33f, 2.25f}, {4.49f, 0.32f, 0.02f, 0.10f, 0.01f, 0.0f, 0.05f, 0.33f}},
        Q5K{{8.22f, 1.24f, 3.32f, 0.27f, 2.51f}, {4.23f, 0.15f, 0.03f, 0.10f, 0.05f, 0.0f, 0.05f, 0.43f}},
        Q6K{{8.64f, 1.50f, 2.55f, 0.32f, 2.63f}, {4.16f, 0.27f, 0.00f, 0.10f, 0.07f, 0.01f, 0.07f, 0.63f}},
        Q80{{8.67f, 2.12f, 3.06f, 0.26f, 2.35f}, {4.18f, 0.00f, 0.05f, 0.10f, 0.13f, 0.0f, 0.00f, 0.70f}},
        Q40{{10.18f, 1.31f, 3.00f, 0.27f, 3.37f}, {4.34f, 0.14f, 0.01f, 0.11f, 0.03f, 0.0f, 0.07f, 0.35f}};
    return fmt == CANDY_HIP_Q4_K ? Q4K : fmt == CANDY_HIP_Q5_K ? Q5K : fmt == CANDY_HIP_Q6_K ? Q6K : fmt == CANDY_HIP_Q8_0 ? Q80 : Q40;
}

// 16-row weight fragments per workgroup with which one round of workgroups serves every row and this kernel is ahead of the tiles; 0:
// none, the tiles.  A second round would read the activations again, wider workgroups have no registers for their sums; fewer than
// 2048 weight rows leave half of the CUs idle.  All 3729 calls together take 0.3 % more than the faster kernel for each.  us of a call,
// tiles / here: Q8_0 4096 x 2304, 96 rows 20.4 / 12.1, Q4_K 4096 x 4096, 80 rows 18.9 / 14.3, 128 rows 21.8 / 20.4, 8200 x 2560,
// 96 rows 20.9 / 14.5, Q6_K 4096 x 4096, 96 rows 21.6 / 17.9, 11008 x 4096, 48 rows 29.8 / 17.1, 64 rows 30.7 / 18.4; one super-block in the
// last round, Q4_K 8192 x 2304, 128 rows 17.2 / 15.1, 4200 x 4352, 80 rows 18.3 / 16.2; odd Q6_K blocks, 8200 x 3840, 40 rows 22.8 / 16.1.
static int rows_fragments(int fmt, int64_t rows, int64_t cols, int64_t m, int num_cus) {
    const bool q6k = fmt == CANDY_HIP_Q6_K;
    // up to 64 rows the other formats are on the exact tiles (mmq_f16_big_covers)
    if (m > 128 || (m <= 64 && !q6k && fmt != CANDY_HIP_Q4_K) || rows < 2048 || cols % 256 != 0) return 0;
    // (seven fragments are weighed as eight: where those were behind the tiles, the exact kernel of rows_i8.hip is ahead, 4096 x
    // 4096, 104 rows Q4_K 15.1 there / 18.9 here)
    const int mf = m > 96 ? 8 : fragments(m);
    int rf = 1;
    while ((rows + 16 * rf - 1) / (16 * rf) > num_cus)
        if (++rf > 3) return 0;
    const int64_t blocks = cols / 256, rounds = (blocks + 7) / 8, tiles = (rows + 127) / 128;
    // 48 weight rows beside more than 96 activation rows: seven fragments of these fit the registers, but for Q6_K, and eight for
    // Q4_0.  us of a call, tiles / here: 11008 x 4096, 100 rows Q4_K 30.3 / 24.6, Q5_K 32.3 / 27.9, Q8_0 38.0 / 31.1, Q4_0 38.3 /
    // 26.4, Q6_K 35.8 / 34.8 (8208 x 4096 30.2 / 33.6); 128 rows Q5_K 33.5 / 33.8, Q8_0 39.4 / 40.6, Q4_0 40.0 / 29.4; 11008 x 2048,
    // 100 rows Q4_K 22.5 / 15.5, Q8_0 26.1 / 18.4.  Q4_K beside eight spills nine registers, which it makes up for where rows are
    // short, or where the tiles, whose number is past a third of the CUs, share their K by two and not by three: 128 rows 8208 x 3072
    // 23.9 / 22.6, 10300 x 3072 23.9 / 23.5, 8208 x 3328 24.8 / 25.4, 10880 x 3328 25.9 / 26.2, 8208 x 4096 26.5 / 28.0, 10752 x 4096
    // 28.6 / 29.1, 10880 x 4096 28.1 / 29.1; 10896 x 4096 31.1 / 29.1, 11008 x 4096 31.6 / 29.2, 12288 x 4096 31.8 / 29.7.
    if (rf == 3 && m > 96 && q6k) return 0;
    if (rf == 3 && m > 112 && fmt != CANDY_HIP_Q4_0 && (fmt != CANDY_HIP_Q4_K || (cols > 3072 && 3 * tiles <= num_cus))) return 0;
    if (mf * 32 * cols > 1200000) return 0;  // not measured
    // as plan_split() deals K to the tiles' workgroups
    int64_t splits = std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(num_cus / tiles, blocks / 2), 16));
    const int64_t per = (blocks + splits - 1) / splits;
    splits = (blocks + per - 1) / per;
    const RowsCost &c = rows_cost(fmt);
    const float out = (float)(rows * m) * 4e-6f;
    float tile = c.tile[0] + c.tile[1] * (float)per + c.tile[4] * 1e-3f * (float)(tiles * blocks);
    if (splits > 1) tile += c.tile[2] + c.tile[3] * (float)(splits + 1) * out;
    const float here = c.rows[0] + (float)rounds * (c.rows[1] * rf + c.rows[2] * mf) + (float)blocks * (c.rows[3] * mf + c.rows[4] * rf) +
                       (blocks & 1 ? c.rows[5] * (float)(blocks * rf) : 0.0f) + c.rows[6] * (float)(rf * mf) + c.rows[7] * out;
    return here < tile ? rf : 0;
}
template <class F, int RF, int MF>
constexpr bool reached() {
    constexpr bool q4k = std::is_same<F, BigQ4K>::value, q6k = std::is_same<F, BigQ6K>::value;
    constexpr bool most = q4k || std::is_same<F, BigQ4_0<false>>::value;
    return (MF > 4 || q4k || q6k) && (RF < 3 || MF <= 6 || (MF == 7 && !q6k) || (MF == 8 && most));
}

template <class F, int RF, int MF>
static int launch_rf(candy_hip_device *dev, const candy_hip_qtensor *w, const _Float16 *xh, int64_t m, float *y, const float *res) {
    constexpr size_t smem = lds_bytes<F, RF, MF>();
    void (*kern)(const uint8_t *, const _Float16 *, float *, const float *, int, int, int) = k_mmq_f16_rows<F, RF, MF>;
    CANDY_HIP_TRY(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
    hipLaunchKernelGGL(kern, dim3((unsigned)((w->rows + 16 * RF - 1) / (16 * RF))), dim3(512), smem, dev->stream,
                       (const uint8_t *)w->data, xh, y, res, (int)m, (int)w->rows, (int)w->cols);
    CANDY_LAUNCH_CHECK();
    return CANDY_HIP_OK;
}

template <class F>
static int launch_fmt(candy_hip_device *dev, const candy_hip_qtensor *w, const _Float16 *xh, int64_t m, float *y, const float *res) {
    const int mf = fragments(m), rf = rows_fragments(w->fmt, w->rows, w->cols, m, dev->num_cus);
#define CANDY_RF(RF, MF)                    \
    if constexpr (reached<F, RF, MF>())     \
        if (rf == RF && mf == MF) return launch_rf<F, RF, MF>(dev, w, xh, m, y, res);
#define CANDY_MF(MF) CANDY_RF(1, MF) CANDY_RF(2, MF) CANDY_RF(3, MF)
    CANDY_MF(3) CANDY_MF(4) CANDY_MF(5) CANDY_MF(6) CANDY_MF(7) CANDY_MF(8)
#undef CANDY_MF
#undef CANDY_RF
    return fail(CANDY_HIP_ERR_INVALID, "internal: fp16 contraction of %lld rows", (long long)m);
}

bool mmq_f16_rows_covers(const candy_hip_qtensor *w, int64_t m) {
    if (((uintptr_t)w->data & 15) != 0) return false;  // whole pieces
    switch (w->fmt) {
    case CANDY_HIP_Q4_K: case CANDY_HIP_Q5_K: case CANDY_HIP_Q6_K: case CANDY_HIP_Q8_0: case CANDY_HIP_Q4_0: case CANDY_HIP_Q4_0_GGML:
        return rows_fragments(w->fmt, w->rows, w->cols, m, w->dev->num_cus) > 0;
    default: return false;
    }
}

int launch_mmq_f16_rows(candy_hip_device *dev, const candy_hip_qtensor *w, const _Float16 *xh, int64_t m, float *y, const float *res) {
    CANDY_REQUIRE(m >= 1 && m <= 128 && w->cols % 256 == 0, "internal: shape of the fp16 contraction");
    switch (w->fmt) {
    case CANDY_HIP_Q4_K: return launch_fmt<BigQ4K>(dev, w, xh, m, y, res);
    case CANDY_HIP_Q5_K: return launch_fmt<BigQ5K>(dev, w, xh, m, y, res);
    case CANDY_HIP_Q6_K: return launch_fmt<BigQ6K>(dev, w, xh, m, y, res);
    case CANDY_HIP_Q8_0: return launch_fmt<BigQ8_0>(dev, w, xh, m, y, res);
    case CANDY_HIP_Q4_0: return launch_fmt<BigQ4_0<false>>(dev, w, xh, m, y, res);
    case CANDY_HIP_Q4_0_GGML: return launch_fmt<BigQ4_0<true>>(dev, w, xh, m, y, res);
    default: return fail(CANDY_HIP_ERR_INVALID, "internal: format of the fp16 contraction");
    }
}

}  // namespace candy

// The rule above, for its tests (no device needed).
extern "C" int candy_test_rows_fragments(int fmt, int64_t rows, int64_t cols, int64_t m, int num_cus) {
    return candy::rows_fragments(fmt, rows, cols, m, num_cus);
}
extern "C" int candy_test_rows_activation_fragments(int64_t m) { return candy::fragments(m); }
