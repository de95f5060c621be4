// Prompt-sized batches of Q4_K, Q5_K, Q6_K, Q8_0 and Q4_0 on the fp16 matrix cores: y[m, N] = x[m, K] . W^T.  (Up to 128 rows
// of one weight mostly run in mmq_f16_rows.hip.)
//
// Replaces mul_mat_q / load_tiles_q4_K / load_tiles_q6_K (tensor/internal/cuda/kernels/quantized.cu
// :455-578, :4116-4205) for prompt-sized batches.  With hundreds of activation rows the contraction
// is a dense GEMM, and the per-sub-block rescale that keeps the integer kernel exact costs several
// times the matrix-core time; here the scales are folded into the operands instead:
//   * weights are dequantized exactly as dequantize_block_q4_K / dequantize_block_q6_K do
//     (quantized.cu:1008-1041: (d*sc)*q - dmin*m; :1103-1128: d*sc*(q-32); evaluated in f32) and
//     rounded once to fp16;
//   * activations are the Q8_0 values d_x * q_x (exact in f32) rounded once to fp16;
//   * products accumulate in f32 (v_mfma_f32_16x16x32_f16).
// Both roundings are 2^-12 relative per element; the result stays a few 1e-4 (max-norm) from the
// CPU contraction, inside the 1e-3 bar.
//
// Tiling: a workgroup owns 128 weight rows x 256 (192, 128) activation rows and walks K in steps of 64.
//   k_mmq_f16_pc (what runs): four producer wavefronts dequantize 16 weights per thread and step into an LDS tile
//     (two or three buffers, one barrier per step); four consumer wavefronts read the weight fragments from LDS,
//     load their activation fragments straight from memory into operand registers (the fp16 image is stored
//     fragment by fragment, xh_index4) and issue the matrix instructions.
//   k_mmq_f16 (comparison: option mmq.f16_shape 3): every wavefront dequantizes, copies activations into a second LDS
//     tile and multiplies a 64 x 64 sub-tile.
// Global requests run ahead in registers: a thread's share of a whole super-block of weights four steps ahead
// (HBM), the activations one or two steps ahead (L2).  Workgroups are numbered so that those sharing an XCD (and its
// L2) work on neighbouring weight tiles of the same activation tile.  When the output has too few tiles to fill the
// chip (N = 4096 or 1024 projections), K is split over several workgroups per tile; their partial sums go to a
// scratch buffer and a second kernel adds them in a fixed order (bitwise reproducible).  One launch can serve up to
// three weight tensors that share their activations (q / k / v, gate / up).
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "attention_tiles.h"
#include "f16_weights.h"
#include "internal.h"

namespace candy {

constexpr int BIG_BK = 64;
// LDS tiles are stored as the matrix instruction reads them: a fragment of 16 rows x 32 values of K is 1 KB, its
// 16-byte pieces (8 values of K of one row) in the order lane = 16 * (piece of K) + row, so that a wavefront's
// operand read is 64 consecutive pieces.  (With rows laid end to end, padded or not, the 8 lanes of a group
// straddle both halves of the 64 banks and every 128-bit read takes close to twice the cycles; measured with a
// read-only probe: 2.8 against 4.7 ticks per instruction at 16 wavefronts.)  Offset in halves of piece (row, k):
__device__ __forceinline__ int frag_off(int row, int k) {
    const int piece = (k >> 3) & 3;
    return (((row >> 4) * 2 + (k >> 5)) << 9) + (((piece << 4) + ((row & 15) ^ piece)) << 3);
}
// ... and of the piece lane `lane` of a wavefront reads from a fragment
__device__ __forceinline__ int frag_lane_off(int lane) { return (((lane >> 4) << 4) + ((lane & 15) ^ (lane >> 4))) << 3; }

// ------------------------------------------------------------------ tile kernel
// One launch may serve up to three weight tensors that share the activations (q / k / v of a prompt pass): weight
// tiles [tile0, next tile0) belong to segment s, which has its own weights, row count, output and residual.
// Whether a policy offers the two-part dequantization (Pre, prepare, dequant_pre)
template <class F, class = void>
struct F16Pre {
    struct type {};
    static constexpr bool value = false;
};
template <class F>
struct F16Pre<F, std::void_t<typename F::Pre>> {
    typedef typename F::Pre type;
    static constexpr bool value = true;
};

struct F16Seg {
    const uint8_t *W;
    float *out;
    const float *res;
    int N, tile0;
};
struct F16Group {
    F16Seg seg[3];
    int count;
    _Float16 *act;  // EPI_SILU: the fp16 image that takes the place of both outputs
    __device__ __forceinline__ F16Seg pick(int nt) const {
        F16Seg s = seg[0];
        if (count > 1 && nt >= seg[1].tile0) s = seg[1];
        if (count > 2 && nt >= seg[2].tile0) s = seg[2];
        return s;
    }
};

// grid = tiles * n_split; workgroup (tile, split) contracts super-blocks [split*sb_per, ...) and writes
// its tile to out + split * split_stride (out = y when n_split == 1).
template <class F, int BN, int BM, int WN, int WM, bool RES>
__global__ __launch_bounds__(WN * WM * 64) void k_mmq_f16(const F16Group grp, const _Float16 *__restrict__ xh, int M, int K,
                                                          int n_tiles, int m_tiles, int sb_per, size_t split_stride) {
    constexpr int T = WN * WM * 64;
    constexpr int TN = BN / WN / 16, TM = BM / WM / 16;
    constexpr int ATK = BN * 4 / T;   // dequantization tasks per thread per step
    constexpr int BCH = BM * 8 / T;   // 16-byte activation chunks per thread per step
    static_assert(BN * 4 % T == 0 && BM * 8 % T == 0 && TN >= 1 && TM >= 1, "tile shape");
    extern __shared__ __align__(16) uint8_t smem_raw[];
    _Float16 *sA = (_Float16 *)smem_raw;               // [2][BN / 16][2] fragments
    _Float16 *sB = sA + 2 * BN * BIG_BK;               // [2][BM / 16][2] fragments

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wn = wave % WN, wm = wave / WN;
    // Weight staging lane map: neighbouring lanes take neighbouring quarters of a row (global loads of whole 64-byte
    // runs); the 32 lanes of a half-wavefront take rows {x, x+4, x+8, x+12}, which the row ^ piece term of the
    // layout spreads over all 16 bank windows.  The activations lie in memory fragment by fragment (xh_index4): the
    // tile's share of a step is 2 KB per 16 rows, copied piece by piece into the LDS order.
    const int a_c = lane & 3, a_r = 4 * ((lane >> 2) & 3) + (lane >> 4);

    // tile numbering: the hardware deals workgroups round-robin to the 8 XCDs; give each XCD a
    // contiguous run of weight tiles inside one activation tile
    const int total = n_tiles * m_tiles;
    const int split = blockIdx.x / total;
    int v = blockIdx.x - split * total;
    if ((total & 7) == 0) v = (v & 7) * (total >> 3) + (v >> 3);
    const int mt = v / n_tiles, nt = v - mt * n_tiles;
    const F16Seg seg = grp.pick(nt);
    const int N = seg.N;
    const int n0 = (nt - seg.tile0) * BN, m0 = mt * BM;

    const size_t rb = (size_t)(K >> 8) * F::BLOCK;
    const int sb0 = split * sb_per;
    const int n_sb = min(K >> 8, sb0 + sb_per) - sb0;  // >= 1 by construction of the grid
    const int steps = n_sb * 4;
    const uint8_t *__restrict__ W = seg.W + (size_t)sb0 * F::BLOCK;
    xh += (size_t)sb0 * 8 * 512;  // 8 fragments of 32 values further along K, in every row block
    float *out = seg.out + (size_t)split * split_stride;
    const float *res = seg.res;
    const _Float16 *xtile = xh + (size_t)(m0 >> 4) * (K >> 5) * 512;

    typename F::Raw raw[2][ATK];
    u32x4 xr[2][BCH];
    auto gload_a = [&](int sb, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < ATK; ++i) {
            const int row = ((tid + i * T) >> 6) * 16 + a_r;
            F::load(W + (size_t)min(n0 + row, N - 1) * rb + (size_t)sb * F::BLOCK, a_c, raw[slot][i]);
        }
    };
    auto gload_b = [&](int ks, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < BCH; ++i) {
            // LDS piece q of the tile: 16-row block q >> 7, half of the step (q >> 6) & 1, piece p = (q >> 4) & 3 of row
            // (q & 15) ^ p; in memory a fragment is 16 rows of 64 bytes
            const int q = tid + i * T, pc = (q >> 4) & 3, row = (q & 15) ^ pc;
            xr[slot][i] = *(const u32x4 *)(xtile + ((size_t)(q >> 7) * (K >> 5) + (size_t)ks * 2 + ((q >> 6) & 1)) * 512 +
                                           row * 32 + pc * 8);
        }
    };
    auto stage = [&](int g, int aslot, int bslot, int buf) __attribute__((always_inline)) {
        _Float16 *a = sA + buf * BN * BIG_BK;
        _Float16 *b = sB + buf * BM * BIG_BK;
#pragma unroll
        for (int i = 0; i < ATK; ++i) {
            const int row = ((tid + i * T) >> 6) * 16 + a_r;
            half8 o0, o1;
            int k0, k1;
            F::dequant(raw[aslot][i], g, a_c, o0, o1, k0, k1);
            *(half8 *)&a[frag_off(row, k0)] = o0;
            *(half8 *)&a[frag_off(row, k1)] = o1;
        }
#pragma unroll
        for (int i = 0; i < BCH; ++i) *(u32x4 *)&b[(tid + i * T) * 8] = xr[bslot][i];
    };

    float4v acc[TN][TM];
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) acc[a][b] = float4v{0.f, 0.f, 0.f, 0.f};

    auto compute = [&](int buf) __attribute__((always_inline)) {
        const _Float16 *a = sA + buf * BN * BIG_BK + wn * (BN / WN) * BIG_BK + frag_lane_off(lane);
        const _Float16 *b = sB + buf * BM * BIG_BK + wm * (BM / WM) * BIG_BK + frag_lane_off(lane);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            half8 af[TN], bf[TM];
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) af[tn] = *(const half8 *)&a[(tn * 2 + kk) * 512];
#pragma unroll
            for (int tm = 0; tm < TM; ++tm) bf[tm] = *(const half8 *)&b[(tm * 2 + kk) * 512];
#pragma unroll
            for (int tn = 0; tn < TN; ++tn)
#pragma unroll
                for (int tm = 0; tm < TM; ++tm)
                    acc[tn][tm] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[tn], bf[tm], acc[tn][tm], 0, 0, 0);
        }
    };

    // Step ks = 4*sb + g computes from LDS buffer (ks & 1) and, meanwhile, stages step ks+1 into the
    // other buffer.  Staging step 4*sb+4 (g == 3) is the first use of super-block sb+1, which was
    // requested when super-block sb was first used.  Super-blocks alternate between the two register
    // slots, so the loop body covers two of them.
    gload_a(0, 0);
    gload_b(0, 0);
    gload_b(1, 1);
    gload_a(min(1, n_sb - 1), 1);
    stage(0, 0, 0, 0);
    gload_b(2, 0);
    __syncthreads();
    for (int sb2 = 0; sb2 < n_sb; sb2 += 2) {
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int sb = sb2 + half;
            if (sb >= n_sb) break;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                // One straight-line block per step (loads past the end are clamped to valid addresses and
                // the last step stages a buffer nobody reads).
                const int ks = sb * 4 + g;
                compute(g & 1);
                // (g + 1) & 1 is both the activation slot and the LDS buffer of step ks + 1
                if (g < 3) stage(g + 1, half, (g + 1) & 1, (g + 1) & 1);
                else stage(0, half ^ 1, 0, 0);
                gload_b(min(ks + 3, steps - 1), (g + 1) & 1);
                if (g == 3) gload_a(min(sb + 2, n_sb - 1), half);
                __syncthreads();
            }
        }
    }

    // C layout of a 16x16 tile: lane holds activation row (lane & 15) and weight rows 4*(lane>>4)..+3
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
            const int m = m0 + wm * (BM / WM) + tm * 16 + (lane & 15);
            const int n = n0 + wn * (BN / WN) + tn * 16 + 4 * (lane >> 4);
            if (m >= M) continue;
            float *dst = out + (size_t)m * N + n;
            const float *r = RES && res ? res + (size_t)m * N + n : nullptr;  // may alias dst: read before the store
            if (n + 3 < N && (N & 3) == 0) {
                float4 o = make_float4(acc[tn][tm][0], acc[tn][tm][1], acc[tn][tm][2], acc[tn][tm][3]);
                if (r) {
                    const float4 rv = *(const float4 *)r;
                    o = make_float4(rv.x + o.x, rv.y + o.y, rv.z + o.z, rv.w + o.w);
                }
                *(float4 *)dst = o;
            } else {
#pragma unroll
                for (int l = 0; l < 4; ++l)
                    if (n + l < N) dst[l] = r ? r[l] + acc[tn][tm][l] : acc[tn][tm][l];
            }
        }
}

// ------------------------------------------------------------------ the same tile with the work split by role
// 128 weight rows x BM (256, 192 or 128) activation rows, 8 wavefronts: wavefronts 0-3 (one per SIMD) are producers, 4-7
// consumers.
// Producers request weights, dequantize them and fill the LDS weight buffer of step s + 1 (two buffers) while the
// consumers contract step s; one workgroup barrier per step hands a buffer over.  The activations never touch LDS:
// their fp16 image lies in memory fragment by fragment, 1 KB per B operand of a matrix instruction (xh_index4), so a
// consumer loads each fragment it needs with one 128-bit load per lane, 1 KB of consecutive memory per wavefront,
// straight into operand registers, one step ahead.  Each consumer owns all 128 weight rows and a quarter of the tile's
// activation rows, so every activation fragment is loaded by exactly one wavefront of the workgroup.
//   Why: with the activations staged through LDS by the producers (8 loads and 8 LDS writes per thread and step for
//   BM = 256), disabling parts of the kernel showed the producers alone taking 72 of the kernel's 81 us at
//   14336 x 4096 x 512 - 23 us of that the activation copy, 12 us the dequantization - against 55 us for the consumers
//   alone: moving a step's 32 KB of activations into the CU costs 700 to 950 cycles whichever wavefronts do it, and
//   LDS carried 144 KB per step (now 80 KB: 16 KB of weight tile written, 4 x 16 KB read).
// A consumer walks a step in four phases (two halves of K x two halves of the weight rows) of 16 or 8 matrix
// instructions, reading the next phase's four weight fragments from LDS and requesting a quarter of the next step's
// activation fragments while the current phase's instructions run; it runs at raised priority, so that its matrix
// instruction goes ahead of a producer's vector instruction when both are ready.
// The two roles are separate loops with the same number of barriers, so that their registers (accumulators and
// operand fragments here, raw blocks there) share one allocation.
// BN = 112 (seven 16-row fragments: the second half of the weight rows is three fragments instead of four) is for
// row counts that are a multiple of 7 * 16 and not of 256 * 128: 14336 = 128 * 112 rows are 128 tiles, one or two per
// CU, where 112 tiles of 128 rows leave an eighth of the chip idle or wait for a short last round.  The LDS buffers
// keep room for 128 rows; the producer wavefront whose second task would fall on rows 112 .. 127 repeats its first.
// EPI_SILU: one grid for gate (segment 0) and up (segment 1), 64 rows of each per tile in turns of 32, so that a lane
// ends with gate and up of the same eight values of a Q8_0 block and the four lanes that share an activation row hold
// the block: silu(gate) * up leaves as the fp16 image of its quantization, which the down projection reads.  Neither
// product is written or read as f32.  us per layer, its own launch / this one: Llama-3.2-1B shape 300 rows 157 / 151, 1500
// rows 368 / 348; Llama-3-8B shape (whose two tensors alone would take tiles of 112 rows) 300 rows 331 / 324, 512 rows 356 /
// 342, 2048 rows 1124 / 1052; Llama-2-7B shape 300 rows 311 / 308, 1400 rows 847 / 824.  A CU holds one such workgroup, so
// the epilogue's vector instructions are exposed: with q8_level's branch asked value by value and the full division in
// silu_f half of the gain was lost (1.035 against 1.058 at 1500 rows).
// EPI_TAIL: EPI_RES in a grid whose last round is split (a kernel of its own: the others' prologues stay as short as they are).
enum { EPI_PLAIN, EPI_RES, EPI_SILU, EPI_TAIL };
// silu_f with the quotient corrected once by its own residual: the same bits for every f32 from SILU_ONCE up.  Below, the divisor's
// reciprocal is too small for a normal number, and the full division is asked for, once for eight values (taken at a quarter instead,
// value by value, prompts took 0.6 to 1.5 % longer).
constexpr float SILU_ONCE = -87.3f;
__device__ __forceinline__ float silu_once(float x) {
    const float den = 1.0f + expf(-x), r = __builtin_amdgcn_rcpf(den), q = x * r;
    return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-den, q, x), r, q), den, x);
}
// STAGED: a producer's blocks come into a slice of LDS of its own, 16-byte pieces in the order they lie in memory, and from there
// to its lanes.  For Q8_0, whose lanes would ask for eight runs of 16 bytes and eight scales 34 bytes apart in every super-block:
// that many lines per load bound the tiles, not the dequantization.  us of a call, loads of single lanes / staged: 11008 x 4096, 140
// rows 44.3 / 39.7, 1400 rows 200.8 / 177.6; 4096 x 14336, 1400 rows 227 / 211; 4096 x 4096, 400 rows 37.7 / 35.6.  The other formats'
// blocks are fewer loads, and a slice is a wait for LDS once a super-block: Q4_0 level, Q5_K and Q4_K 3 to 5 % slower, Q6_K (14
// pieces from the one its even address lies in) 7 to 13 %.
template <class F>
constexpr bool f16_staged() { return std::is_same<F, BigQ8_0>::value; }
template <class F>
constexpr int f16_slice_loads() { return (32 * F::BLOCK / 16 + 63) / 64; }  // of 1 KB, for a producer's 32 rows
// A staged piece is found by a 32-bit offset from the tile's first row: the tile's rows within 4 GB (128 rows of Q8_0: 31.5 million
// values each).  Longer ones take the tiles whose lanes load their own runs, through pointers.
static bool f16_roles_fit(int fmt, int64_t tile_rows, int64_t cols) {
    return fmt != CANDY_HIP_Q8_0 || tile_rows * (cols / 256 * BigQ8_0::BLOCK) <= 0xFFFFFFFFll;
}

// Of a grid of more workgroups than CUs, the tiles of a short last round split K over the CUs that would be idle (plan_tail):
// tiles whole .. end are dealt to several workgroups of `sb` super-blocks each, behind the whole ones, which leave BM x BN sums in
// `part`, [split][tile], for k_tail_sum.
struct F16Tail {
    float *part;
    int whole, sb;
};

template <class F, int BN, int BM, int EPI>
__global__ __launch_bounds__(512) void k_mmq_f16_pc(const F16Group grp, const _Float16 *__restrict__ xh, int M, int K,
                                                    int n_tiles, int m_tiles, int sb_per, size_t split_stride, const F16Tail tail) {
    constexpr int PT = 256, BNB = 128;  // BNB: weight rows an LDS buffer has room for
    constexpr int ATK = BNB * 4 / PT;   // dequantization tasks per producer thread per step
    constexpr int TNF = BN / 16;        // 16-row weight fragments of the tile
    static_assert(BN == 128 || BN == 112, "weight rows per tile");
    constexpr int TM = BM / 64;       // 16-row activation fragments of a consumer's sub-tile (its rows: BM / 4)
    static_assert(BM == 256 || BM == 192 || BM == 128, "activation rows per tile");
    // BM = 256, 192: the producers work two steps ahead into the third of three weight buffers, and a consumer reads the
    // first weight fragments of step s + 1 during the last matrix instructions of step s (16 per phase cover the
    // read).  BM = 128 (8 matrix instructions per phase) is faster one step ahead with two buffers: 33.8 against
    // 35.2 us at 14336 x 4096 x 128.
    constexpr int LEAD = BM > 128 ? 2 : 1, NB = LEAD + 1;
    extern __shared__ __align__(16) uint8_t smem_raw[];
    _Float16 *sA = (_Float16 *)smem_raw;               // [NB][BNB / 16][2] fragments

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    const int total = n_tiles * m_tiles, whole = EPI == EPI_TAIL ? tail.whole : total;
    const bool in_tail = EPI == EPI_TAIL && (int)blockIdx.x >= whole;
    const int b = blockIdx.x - (in_tail ? whole : 0), group = in_tail ? total - whole : whole;
    const int split = b / group;
    int v = b - split * group;
    if (in_tail) v += whole;
    else if ((whole & 7) == 0) v = (v & 7) * (whole >> 3) + (v >> 3);
    if (in_tail) sb_per = tail.sb;
    const int mt = v / n_tiles, nt = v - mt * n_tiles;
    static_assert(EPI != EPI_SILU || BN == 128, "64 rows of gate and of up");
    const F16Seg seg = EPI == EPI_SILU ? grp.seg[wave >> 1 & 1] : grp.pick(nt);  // producers 0, 1 gate and 2, 3 up
    const int N = seg.N;
    const int n0 = EPI == EPI_SILU ? nt * (BN / 2) : (nt - seg.tile0) * BN, m0 = mt * BM;

    const size_t rb = (size_t)(K >> 8) * F::BLOCK;
    const int sb0 = split * sb_per;
    const int n_sb = min(K >> 8, sb0 + sb_per) - sb0;  // >= 1 by construction of the grid
    const int steps = n_sb * 4;
    const uint8_t *__restrict__ W = seg.W + (size_t)sb0 * F::BLOCK;
    xh += (size_t)sb0 * 8 * 512;  // 8 fragments of 32 values further along K, in every row block
    float *out = EPI == EPI_TAIL ? seg.out : seg.out + (size_t)split * split_stride;
    const float *res = seg.res;

    if (wave < 4) {
        // ---------------- producers: the weight tile of step t + LEAD (buffer (t + LEAD) % NB) while step t is contracted
        constexpr bool STAGED = f16_staged<F>();
        constexpr int SLOTS = STAGED ? 1 : 2;
        typename F::Raw raw[SLOTS][ATK];
        typename F16Pre<F>::type pre[SLOTS][ATK];
        // neighbouring lanes take neighbouring quarters of a row; a half-wavefront takes rows {x, x+4, x+8, x+12}
        const int a_c = lane & 3, a_row = 16 * wave + 4 * ((lane >> 2) & 3) + (lane >> 4);   // + a_step i
        const int a_step = BN == 112 && wave == 3 ? 0 : 64;
        const int w_row = EPI == EPI_SILU ? a_row & 31 : a_row, w_step = EPI == EPI_SILU ? 32 : a_step;  // in the tensor
        auto gload_a = [&](int sb, int slot) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < ATK; ++i)
                F::load(W + (size_t)min(n0 + w_row + w_step * i, N - 1) * rb + (size_t)sb * F::BLOCK, a_c, raw[slot][i]);
        };
        auto stage = [&](int g, int aslot, int buf) __attribute__((always_inline)) {
            _Float16 *a = sA + buf * BNB * BIG_BK;
#pragma unroll
            for (int i = 0; i < ATK; ++i) {
                half8 o0, o1;
                int k0, k1;
                if constexpr (F16Pre<F>::value) {
                    if (g == 0) F::prepare(raw[aslot][i], a_c, pre[aslot][i]);  // a super-block's first step
                    F::dequant_pre(raw[aslot][i], pre[aslot][i], g, a_c, o0, o1, k0, k1);
                } else {
                    F::dequant(raw[aslot][i], g, a_c, o0, o1, k0, k1);
                }
                *(half8 *)&a[frag_off(a_row + a_step * i, k0)] = o0;
                *(half8 *)&a[frag_off(a_row + a_step * i, k1)] = o1;
            }
        };
        if constexpr (STAGED) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass knows no buffer descriptors
            constexpr int P = F::BLOCK / 16, IT = f16_slice_loads<F>();
            static_assert(F::BLOCK % 16 == 0, "whole pieces");
            uint8_t *const slice = smem_raw + 3 * BNB * BIG_BK * 2 + wave * (IT * 1024);
            const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void *)(W + (size_t)n0 * rb), 0, -1, 0x00027000);
            const int row0 = EPI == EPI_SILU ? 16 * wave & 31 : 16 * wave;
            uint32_t from[IT];  // of a lane's piece, from the tile's first row and super-block
#pragma unroll
            for (int it = 0; it < IT; ++it) {
                const int e = min(it * 64 + lane, 32 * P - 1), r = e / P;  // lanes past the last piece fetch it once more
                from[it] = (uint32_t)(min(n0 + row0 + (r & 15) + (r >> 4) * w_step, N - 1) - n0) * (uint32_t)rb + (uint32_t)(e - r * P) * 16;
            }
            auto request = [&](int sb) __attribute__((always_inline)) {
#pragma unroll
                for (int it = 0; it < IT; ++it)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (__attribute__((address_space(3))) void *)(slice + it * 1024), 16, from[it],
                                                             sb * F::BLOCK, 0, 0);
            };
            auto take = [&]() __attribute__((always_inline)) {
                __builtin_amdgcn_s_waitcnt(0x0070);  // the slice has landed
                asm volatile("" ::: "memory");
#pragma unroll
                for (int i = 0; i < ATK; ++i) F::load(slice + ((a_row & 15) + 16 * i) * F::BLOCK, a_c, raw[0][i]);
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_waitcnt(0x0070);  // and is in registers
            };
            auto meet = [&]() __attribute__((always_inline)) {  // __syncthreads() without a wait for the slice
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_waitcnt(0xC07F);
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
            };
            request(0);
            take();
            request(min(1, n_sb - 1));
            stage(0, 0, 0);
            if (LEAD == 2) stage(1, 0, 1);
            meet();
            int buf = LEAD % NB;
            for (int t4 = 0; t4 < steps; t4 += 4) {
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int g = (u + LEAD) & 3, sb = (t4 + u + LEAD) >> 2;
                    if (g == 0) {
                        take();
                        request(min(sb + 1, n_sb - 1));
                    }
                    stage(g, 0, NB == 2 ? ((u + LEAD) & 1) : buf);
                    buf = buf == NB - 1 ? 0 : buf + 1;
                    meet();
                }
            }
            __builtin_amdgcn_s_waitcnt(0x0070);  // the last request writes LDS that is still this workgroup's
#endif
            return;
        }
        if constexpr (!STAGED) {
            gload_a(0, 0);
            gload_a(min(1, n_sb - 1), 1);
            stage(0, 0, 0);
            if (LEAD == 2) stage(1, 0, 1);
            __syncthreads();
            // Iteration t = 8 j + u stages step t + LEAD (past the end: a clamped super-block, into a buffer nobody
            // reads): super-blocks alternate between the two raw slots, so u fixes group and slot of the staged step.
            int buf = LEAD % NB;
            for (int t8 = 0; t8 < steps; t8 += 8) {
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int t = t8 + u;
                    if ((u & 3) == 0 && t >= steps) break;  // steps is a multiple of 4
                    const int g = (u + LEAD) & 3, slot = ((u + LEAD) >> 2) & 1;
                    stage(g, slot, NB == 2 ? ((u + LEAD) & 1) : buf);  // two buffers: a constant of the unrolled body
                    buf = buf == NB - 1 ? 0 : buf + 1;
                    if (g == 3) gload_a(min(((t + LEAD) >> 2) + 2, n_sb - 1), slot);
                    __syncthreads();
                }
            }
        }
        return;
    }

    // ---------------- consumers: wavefront cw owns the BN weight rows x activation rows [cw * BM / 4, + BM / 4)
    const int cw = wave - 4;
    __builtin_amdgcn_s_setprio(3);
    float4v acc[TNF][TM];
#pragma unroll
    for (int a = 0; a < TNF; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) acc[a][b] = float4v{0.f, 0.f, 0.f, 0.f};
    // activation fragment (16-row block rbk of the tile, 32-value block kb of K): 1 KB at ((m0 / 16 + rbk) * (K / 32) + kb)
    // * 1 KB; lane l takes row l & 15, values 8 (l >> 4) .. + 7: the wavefront's 64 loads cover the fragment once
    const _Float16 *xfrag = xh + ((size_t)((m0 >> 4) + cw * TM) * (K >> 5)) * 512 + (lane & 15) * 32 + (lane >> 4) * 8;
    // steps the activation loads run ahead, and register slots for them: two steps for the 128-row tiles, whose steps
    // are shorter than a load from L2 under this traffic takes (14336 x 4096 x 128: 31.5 us; one step 32.2, three 32.6)
    constexpr int BD = BM == 128 ? 2 : 1, NS = 2 * BD;
    half8 bf[NS][2][TM];  // [step % NS][half of the step][fragment]
    auto load_b = [&](int ks, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
                bf[slot][kk][tm] = *(const half8 *)(xfrag + ((size_t)tm * (K >> 5) + (size_t)ks * 2 + kk) * 512);
    };
    // A step is four phases, phase p = 2 * kk + h: weight rows 64 h .. min(64 h + 63, BN - 1), values 32 kk .. 32 kk + 31
    // (two phases of all the weight rows for the 128-row tiles, whose phases have 8 matrix instructions: 34.4 against
    // 33.8 us at 14336 x 4096 x 128; eight producer wavefronts for them: 33.6 against 33.0)
    constexpr int PH = 4, HN = 4;  // phases per step, weight fragments per phase
    half8 af[2][HN];
    auto fetch = [&](int abuf, int p) __attribute__((always_inline)) {
        const _Float16 *a = sA + abuf * BNB * BIG_BK + frag_lane_off(lane);
        const int kk = PH == 4 ? p >> 1 : p, t0 = PH == 4 ? (p & 1) * 4 : 0;
#pragma unroll
        for (int tn = 0; tn < HN; ++tn)
            if (t0 + tn < TNF) af[p & 1][tn] = *(const half8 *)&a[((t0 + tn) * 2 + kk) * 512];
    };
    auto mma = [&](int bslot, int p) __attribute__((always_inline)) {
        const int kk = PH == 4 ? p >> 1 : p, t0 = PH == 4 ? (p & 1) * 4 : 0;
#pragma unroll
        for (int tn = 0; tn < HN; ++tn)
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
                if (t0 + tn < TNF)
                    acc[t0 + tn][tm] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[p & 1][tn], bf[bslot][kk][tm],
                                                                            acc[t0 + tn][tm], 0, 0, 0);
    };
    load_b(0, 0);
    if (BD == 2) load_b(min(1, steps - 1), 1);
    __syncthreads();  // the weight tiles of the first LEAD steps are in LDS
    constexpr bool AHEAD = LEAD == 2;
    if (AHEAD) fetch(0, 0);
    int abuf = 0;
    for (int sb = 0; sb < n_sb; ++sb) {  // four steps per iteration: no exit inside the unrolled body
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int ks = sb * 4 + g;
            const int anext = abuf == NB - 1 ? 0 : abuf + 1;
            const int acur = NB == 2 ? (g & 1) : abuf;  // two buffers: a constant of the unrolled body
            const int ksn = min(ks + BD, steps - 1);  // a later step's activations, in flight during this one:
            if (!AHEAD) fetch(acur, 0);               // a quarter of them requested in front of each phase
#pragma unroll
            for (int p = 0; p < PH; ++p) {
#pragma unroll
                for (int l = 2 * TM * p / PH; l < 2 * TM * (p + 1) / PH; ++l) {
                    const int kk = l / TM, tm = l % TM;
                    bf[(g + BD) & (NS - 1)][kk][tm] = *(const half8 *)(xfrag + ((size_t)tm * (K >> 5) + (size_t)ksn * 2 + kk) * 512);
                }
                // the next phase's weight fragments - after the last phase: the next step's first, whose buffer has
                // been complete since the barrier before this step - are read while this phase multiplies
                if (p < PH - 1) fetch(acur, p + 1);
                else if (AHEAD) fetch(anext, 0);
                __builtin_amdgcn_sched_barrier(0);
                mma(g & (NS - 1), p);
                __builtin_amdgcn_sched_barrier(0);
            }
            abuf = anext;
            __syncthreads();
        }
    }

    if (in_tail) {
        float *to = tail.part + ((size_t)split * group + (v - whole)) * (BM * BN) + 4 * (lane >> 4);
#pragma unroll
        for (int tn = 0; tn < TNF; ++tn)
#pragma unroll
            for (int tm = 0; tm < TM; ++tm) {
                const int m = cw * (BM / 4) + tm * 16 + (lane & 15);
                if (m0 + m < M)
                    *(float4 *)(to + m * BN + tn * 16) = make_float4(acc[tn][tm][0], acc[tn][tm][1], acc[tn][tm][2], acc[tn][tm][3]);
            }
        return;
    }
    if constexpr (EPI == EPI_SILU) {
        // the arithmetic of k_silu_mul_quant (quantize_q8_lane4 + q8_lane4_to_half) value by value
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
            const int m = m0 + cw * (BM / 4) + tm * 16 + (lane & 15);
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                float z[2][4], amax = 0.0f, least = 0.0f;
#pragma unroll
                for (int hf = 0; hf < 2; ++hf)
#pragma unroll
                    for (int l = 0; l < 4; ++l) {
                        z[hf][l] = silu_once(acc[4 * b + hf][tm][l]) * acc[4 * b + 2 + hf][tm][l];
                        least = fminf(least, acc[4 * b + hf][tm][l]);
                    }
                if (__builtin_expect(least < SILU_ONCE, 0)) {
#pragma unroll
                    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
                        for (int l = 0; l < 4; ++l) z[hf][l] = silu_f(acc[4 * b + hf][tm][l]) * acc[4 * b + 2 + hf][tm][l];
                }
#pragma unroll
                for (int hf = 0; hf < 2; ++hf)
#pragma unroll
                    for (int l = 0; l < 4; ++l) amax = hf + l ? fmaxf(amax, fabsf(z[hf][l])) : fabsf(z[hf][l]);
                amax = quad16_max(amax);
                const float d = amax / 127.0f, df = __half2float(__float2half_rn(d)), inv = __builtin_amdgcn_rcpf(d);
                // q8_level: the rounded product is the level unless it lies within 6.1e-5 of a half (or is no number: an
                // empty block, a scale or a value that is not finite), asked once for the eight values
                float level[2][4];
                bool unsure = false;
#pragma unroll
                for (int hf = 0; hf < 2; ++hf)
#pragma unroll
                    for (int l = 0; l < 4; ++l) {
                        const float t = z[hf][l] * inv;
                        level[hf][l] = rintf(t);
                        unsure |= !(fabsf(t - level[hf][l]) < 0.5f - 6.1e-5f);
                    }
                if (__builtin_expect(unsure, 0)) {
#pragma unroll
                    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
                        for (int l = 0; l < 4; ++l) level[hf][l] = (float)(int8_t)(amax != 0.0f ? q8_level(z[hf][l], d) : 0);
                }
                const int n = n0 + 32 * b + 4 * (lane >> 4);
#pragma unroll
                for (int hf = 0; hf < 2; ++hf) {
                    half4v h;
#pragma unroll
                    for (int l = 0; l < 4; ++l) h[l] = (_Float16)(df * level[hf][l]);
                    if (m < M && n < N) *(half4v *)(grp.act + xh_index4(m, (n + 16 * hf) >> 2, N) * 4) = h;
                }
            }
        }
        return;
    }

    // C layout of a 16x16 tile: lane holds activation row (lane & 15) and weight rows 4*(lane>>4)..+3
#pragma unroll
    for (int tn = 0; tn < TNF; ++tn)
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
            const int m = m0 + cw * (BM / 4) + tm * 16 + (lane & 15);
            const int n = n0 + tn * 16 + 4 * (lane >> 4);
            if (m >= M) continue;
            float *dst = out + (size_t)m * N + n;
            // may alias dst: read before the store
            const float *r = (EPI == EPI_RES || EPI == EPI_TAIL) && res ? res + (size_t)m * N + n : nullptr;
            if (n + 3 < N && (N & 3) == 0) {
                float4 o = make_float4(acc[tn][tm][0], acc[tn][tm][1], acc[tn][tm][2], acc[tn][tm][3]);
                if (r) {
                    const float4 rv = *(const float4 *)r;
                    o = make_float4(rv.x + o.x, rv.y + o.y, rv.z + o.z, rv.w + o.w);
                }
                *(float4 *)dst = o;
            } else {
#pragma unroll
                for (int l = 0; l < 4; ++l)
                    if (n + l < N) dst[l] = r ? r[l] + acc[tn][tm][l] : acc[tn][tm][l];
            }
        }
}

// y[i] = (res[i] +) part[0][i] + part[1][i] + ... in that order (copies `stride` floats apart); res may alias y
__global__ __launch_bounds__(256) void k_splitk_sum(const float *__restrict__ part, float *y, const float *res, size_t count,
                                                    int n_split, size_t stride) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= count) return;
    if (i + 4 <= count && (((uintptr_t)y | (uintptr_t)part | (uintptr_t)res) & 15) == 0 && ((count | stride) & 3) == 0) {
        float4 s = *(const float4 *)(part + i);
        for (int k = 1; k < n_split; ++k) {
            const float4 v = *(const float4 *)(part + (size_t)k * stride + i);
            s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
        }
        if (res) {
            const float4 r = *(const float4 *)(res + i);
            s = make_float4(r.x + s.x, r.y + s.y, r.z + s.z, r.w + s.w);
        }
        *(float4 *)(y + i) = s;
    } else {
        for (size_t j = i; j < i + 4 && j < count; ++j) {
            float s = part[j];
            for (int k = 1; k < n_split; ++k) s += part[(size_t)k * stride + j];
            y[j] = res ? res[j] + s : s;
        }
    }
}

int launch_splitk_sum(candy_hip_device *dev, const float *part, float *y, const float *res, size_t count, int n_split,
                      size_t stride) {
    hipLaunchKernelGGL(k_splitk_sum, dim3((unsigned)((count / 4 + 256) / 256)), dim3(256), 0, dev->stream, part, y, res,
                       count, n_split, stride ? stride : count);
    CANDY_LAUNCH_CHECK();
    return CANDY_HIP_OK;
}

// The last round's tiles: y = (res +) the copies in the order of K.  grid: tile, 8 of its activation rows.
template <int BN, int BM>
__global__ __launch_bounds__(256) void k_tail_sum(const F16Group grp, const float *__restrict__ part, int whole, int tiles, int splits, int n_tiles,
                                                  int M) {
    constexpr int Q = BN / 4;  // threads of a row
    const int tid = threadIdx.x, row = blockIdx.y * 8 + tid / Q, col = (tid % Q) * 4;
    const int v = whole + blockIdx.x, mt = v / n_tiles, nt = v - mt * n_tiles;
    const F16Seg seg = grp.pick(nt);
    const int m = mt * BM + row, n = (nt - seg.tile0) * BN + col;
    if (tid >= 8 * Q || m >= M || n >= seg.N) return;
    const float *p = part + (size_t)blockIdx.x * (BM * BN) + row * BN + col;
    float4 s = *(const float4 *)p;
    for (int k = 1; k < splits; ++k) {
        const float4 a = *(const float4 *)(p + (size_t)k * tiles * (BM * BN));
        s.x += a.x; s.y += a.y; s.z += a.z; s.w += a.w;
    }
    float *y = seg.out + (size_t)m * seg.N + n;
    const float *r = seg.res ? seg.res + (size_t)m * seg.N + n : nullptr;  // may alias y: read before the store
    if (n + 3 < seg.N && (seg.N & 3) == 0) {
        if (r) {
            const float4 a = *(const float4 *)r;
            s = make_float4(a.x + s.x, a.y + s.y, a.z + s.z, a.w + s.w);
        }
        *(float4 *)y = s;
    } else {
        const float o[4] = {s.x, s.y, s.z, s.w};
        for (int l = 0; l < 4; ++l)
            if (n + l < seg.N) y[l] = r ? r[l] + o[l] : o[l];
    }
}

// Up to three contractions that share the activations, in one launch (a single one: count = 1).  Every tensor but the
// last has a multiple of BN rows (a tile belongs to one tensor).
struct F16Job {
    const candy_hip_qtensor *w;
    float *y;
    const float *res;
};

// Workgroups per tile along K: split K until the grid covers the chip, keeping at least two super-blocks (8 steps)
// per workgroup: as many workgroups per tile as leave every workgroup a CU of its own (measured against rounding up:
// 14336 x 4096 at 128 rows 44.8 us with 2 against 47.6 with 3; 11008 x 4096 at 256 rows 57.4 with 2 against 66.6 with
// 3, at 512 rows 88.8 with 1 against 105.7 with 2)
static int plan_split(const candy_hip_device *dev, int tiles, int n_sb) {
    int n_split = 1;
    if (tiles < (3 * dev->num_cus) / 4) {
        n_split = dev->num_cus / tiles;
        if (n_split > n_sb / 2) n_split = n_sb / 2;
        if (n_split > 16) n_split = 16;
        if (n_split < 1) n_split = 1;
    }
    if (dev->opt.f16_split > 0) n_split = std::min(dev->opt.f16_split, n_sb);  // comparison runs
    return n_split;
}

// A grid whose last round has tiles for half the CUs at the most (Q4_K, whose rounds are the shortest: 0.4): these tiles split K, so
// that the round is as much shorter (two super-blocks a workgroup or more, of the last part one; not for short K, where the second
// launch costs what the round does).  us of a call, whole tiles / last round split: 11008 x 4096, 700 rows (258 tiles, two rounds for one
// and two tiles) Q4_K 104 / 84, Q6_K 122 / 92, Q8_0 126 / 95; 1500 rows (516) 159 / 149, 187 / 163, 192 / 167; 14336 x 4096, 600 rows
// Q8_0 (336, the last 80 in three) 122 / 110.  Q4_K, half a round in two: prompts of the 7B shape, whose q / k / v are 384 tiles at 1000
// tokens, 2237 / 2261 (four layers and the head): a full chip's clock falls by what the round gains.
struct TailPlan {
    int whole, splits = 0, sb = 0;  // tiles not split; workgroups and super-blocks of each of the others, 0: there are none
};
static TailPlan plan_tail(const candy_hip_device *dev, int fmt, int64_t tiles, int n_sb) {
    TailPlan p{(int)tiles};
    const int t = (int)(tiles % dev->num_cus);
    if (dev->opt.f16_shape != 0 || dev->opt.f16_split != 0 || n_sb < 8 || tiles < dev->num_cus || t == 0) return p;
    if ((fmt == CANDY_HIP_Q4_K ? 5 : 4) * t > 2 * dev->num_cus) return p;
    const int s = std::min(std::min(dev->num_cus / t, n_sb / 2), 16), sb = (n_sb + s - 1) / s, splits = (n_sb + sb - 1) / sb;
    // of a round's super-blocks an eighth is left, with two for the first loads and the launch that sums, and 2.5 a chip full of
    // tiles summed
    if (8 * (2 * (n_sb - sb - 2) * dev->num_cus - 5 * t * splits) < 2 * n_sb * dev->num_cus) return p;
    p.whole = (int)tiles - t;
    p.sb = sb;
    p.splits = splits;
    return p;
}

// LDS of the role-split kernel: weight tiles, and the producers' slices
template <class F>
constexpr size_t pc_lds() { return (size_t)3 * 128 * BIG_BK * sizeof(_Float16) + (f16_staged<F>() ? (size_t)4 * 1024 * f16_slice_loads<F>() : 0); }

template <class F, int BN, int BM, int WN, int WM, bool PC = false>
static int launch_big(candy_hip_device *dev, const F16Job *jobs, int count, const _Float16 *xh, int64_t m) {
    static_assert(!PC || ((BN == 128 || BN == 112) && (BM == 256 || BM == 192 || BM == 128) && WN * WM == 8), "the role-split kernel's tiles");
    const int K = (int)jobs[0].w->cols;
    F16Group grp{};
    grp.count = count;
    int n_tiles = 0;
    int64_t n_total = 0;
    bool any_res = false;
    for (int s = 0; s < count; ++s) {
        grp.seg[s] = F16Seg{(const uint8_t *)jobs[s].w->data, jobs[s].y, jobs[s].res, (int)jobs[s].w->rows, n_tiles};
        n_tiles += (int)((jobs[s].w->rows + BN - 1) / BN);
        n_total += jobs[s].w->rows;
        any_res = any_res || jobs[s].res;
    }
    const int m_tiles = (int)((m + BM - 1) / BM);
    const int tiles = n_tiles * m_tiles, n_sb = K >> 8;
    int n_split = plan_split(dev, tiles, n_sb);
    const int sb_per = (n_sb + n_split - 1) / n_split;
    n_split = (n_sb + sb_per - 1) / sb_per;  // no empty splits
    const size_t split_stride = (size_t)m * (size_t)n_total;
    float *part = nullptr;
    if (n_split > 1) {
        // each workgroup writes its partial tile to copy `split` of a workspace laid out [split][tensor][m][rows]
        void *p = nullptr;
        if (int rc = splitk_workspace(dev, (size_t)n_split * split_stride * sizeof(float), &p)) return rc;
        part = (float *)p;
        size_t off = 0;
        for (int s = 0; s < count; ++s) {
            grp.seg[s].out = part + off;
            grp.seg[s].res = nullptr;  // the split sum adds it
            off += (size_t)m * (size_t)jobs[s].w->rows;
        }
    }
    TailPlan tail{tiles};
    F16Tail tail_args{};
    if (PC && n_split == 1) {
        tail = plan_tail(dev, jobs[0].w->fmt, tiles, n_sb);
        void *p = nullptr;
        if (tail.splits) {
            const int rc = splitk_workspace(dev, (size_t)tail.splits * (tiles - tail.whole) * BM * BN * sizeof(float), &p);
            if (rc && rc != CANDY_HIP_ERR_OOM) return rc;
            if (rc) {  // without the memory they stay whole
                (void)hipGetLastError();
                tail = TailPlan{tiles};
            } else {
                tail_args = F16Tail{(float *)p, tail.whole, tail.sb};
            }
        }
    }
    constexpr size_t smem = PC ? pc_lds<F>() : (size_t)2 * (BN + BM) * BIG_BK * sizeof(_Float16);
    const bool epi_res = any_res && n_split == 1;
    const unsigned wgs = (unsigned)(tiles * n_split + (tiles - tail.whole) * (tail.splits - (tail.splits ? 1 : 0)));
    auto launch = [&](auto kern, auto... more) -> int {
        CANDY_HIP_TRY(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        hipLaunchKernelGGL(kern, dim3(wgs), dim3(WN * WM * 64), smem, dev->stream, grp, xh, (int)m, K, n_tiles, m_tiles, sb_per,
                           split_stride, more...);
        CANDY_LAUNCH_CHECK();
        return CANDY_HIP_OK;
    };
    int rc;
    if constexpr (PC)
        rc = tail.splits ? launch(k_mmq_f16_pc<F, BN, BM, EPI_TAIL>, tail_args)
             : epi_res   ? launch(k_mmq_f16_pc<F, BN, BM, EPI_RES>, tail_args)
                         : launch(k_mmq_f16_pc<F, BN, BM, EPI_PLAIN>, tail_args);
    else
        rc = epi_res ? launch(k_mmq_f16<F, BN, BM, WN, WM, true>) : launch(k_mmq_f16<F, BN, BM, WN, WM, false>);
    if (rc) return rc;
    if (tail.splits) {
        hipLaunchKernelGGL((k_tail_sum<BN, BM>), dim3((unsigned)(tiles - tail.whole), BM / 8), dim3(256), 0, dev->stream, grp,
                           tail_args.part, tail.whole, tiles - tail.whole, tail.splits, n_tiles, (int)m);
        CANDY_LAUNCH_CHECK();
    }
    bool one_run = true;  // outputs end to end, no residual but a single job's
    for (int s = 1; s < count; ++s)
        one_run = one_run && !jobs[0].res && !jobs[s].res && jobs[s].y == jobs[s - 1].y + (size_t)m * (size_t)jobs[s - 1].w->rows;
    if (n_split > 1 && one_run && dev->defer_split) {
        SplitPending &sp = *dev->defer_split;  // the caller sums the copies
        sp.part = part; sp.y = jobs[0].y; sp.res = jobs[0].res;
        sp.count = split_stride; sp.stride = split_stride; sp.n_split = n_split;
    } else if (n_split > 1) {
        // one sum per run of outputs that lie end to end (the prompt pass allocates q, k and v that way)
        size_t off = 0;
        for (int s = 0; s < count;) {
            size_t run = (size_t)m * (size_t)jobs[s].w->rows;
            int e = s + 1;
            while (e < count && !jobs[s].res && !jobs[e].res && jobs[e].y == jobs[s].y + run) {
                run += (size_t)m * (size_t)jobs[e].w->rows;
                ++e;
            }
            hipLaunchKernelGGL(k_splitk_sum, dim3((unsigned)((run / 4 + 256) / 256)), dim3(256), 0, dev->stream, part + off,
                               jobs[s].y, jobs[s].res, run, n_split, split_stride);
            CANDY_LAUNCH_CHECK();
            off += run;
            s = e;
        }
    }
    return CANDY_HIP_OK;
}

template <class F, int BN, int BM, int WN, int WM, bool PC = false>
static int launch_big(candy_hip_device *dev, const candy_hip_qtensor *w, const _Float16 *xh, int64_t m, float *y,
                      const float *res) {
    const F16Job job{w, y, res};
    return launch_big<F, BN, BM, WN, WM, PC>(dev, &job, 1, xh, m);
}

bool mmq_f16_big_covers(const candy_hip_qtensor *w, int64_t m, int min_m) {
    // A lower threshold than the decoder's holds for single contractions through the API: Q4_K and Q6_K from `min_m`
    // rows, the other formats from 65: up to 64 rows are one tile of the int8 kernel, which is level with the fp16 tiles
    // there for Q8_0, Q4_0 and Q5_K (and exact).  Measured, us per call, int8 / fp16 tiles: Q6_K 14336 x 4096 at 33 rows
    // 43.8 / 36.6, 4096 x 14336 at 96 rows 71.5 / 39.2, at 255 rows 133 / 57; Q8_0 14336 x 4096 at 48 rows 46.2 / 41.9
    // (4096 x 4096 22.4 / 22.6), at 96 rows 77.8 / 44.7, at 255 rows 121 / 61; Q4_0 at 48 rows 38.9 / 38.0 (4096 x 4096
    // 19.9 / 22.4), at 96 rows 64.3 / 48.7; Q5_K 36.9 / 35.1 (19.9 / 19.9) and 58.6 / 47.2.
    if (min_m <= 0) min_m = w->dev->opt.f16_big_min_m;
    else if (w->fmt != CANDY_HIP_Q4_K && w->fmt != CANDY_HIP_Q6_K) min_m = std::max(min_m, 65);
    if (m < min_m || w->cols % 256 != 0) return false;
    if (w->fmt == CANDY_HIP_Q4_K || w->fmt == CANDY_HIP_Q5_K || w->fmt == CANDY_HIP_Q8_0) return ((uintptr_t)w->data & 15) == 0;
    if (w->fmt == CANDY_HIP_Q6_K || w->fmt == CANDY_HIP_Q4_0 || w->fmt == CANDY_HIP_Q4_0_GGML)
        return ((uintptr_t)w->data & 1) == 0;
    return false;
}

// Tile shape by batch and grid.  Every format: 128 x 128 tiles up to 128 activation rows, 128 x 256 or 128 x 192 above.  Q4_K, whose
// dequantization is the cheapest, also takes the narrower tiles on some grids above 128 rows (with the heavier formats
// the producers then set the pace: Q6_K 14336 x 4096 at 192 rows 58.3 us on 128 x 128 tiles against 53.8, Q8_0 68.5
// against 58.6), and tiles of 112 weight rows.
struct F16Tile {
    int bn, bm;   // weight rows, activation rows
    bool single;  // every wavefront in both roles
};
static F16Tile pick_tile(const candy_hip_device *dev, int fmt, const int64_t *rows, int count, int64_t cols, int64_t m) {
    const bool q4k = fmt == CANDY_HIP_Q4_K;
    const int shape = dev->opt.f16_shape;  // comparison runs
    const bool single = shape == 3 || !f16_roles_fit(fmt, std::min<int64_t>(128, *std::max_element(rows, rows + count)), cols);
    const int n_sb = (int)(cols >> 8);
    // What the busiest CU does: rounds of workgroups x weight rows per tile x super-blocks per workgroup, x 8000 (a step of 192
    // activation rows: 7000, of 256: 8000; measured 0.84 to 0.88, the producers' share being the same).  A last round that is split counts
    // with its super-blocks, what plan_tail sets off, and 3 % of it all where the sides are near each other, for Q4_K 6 (prompts of the
    // 7B shape, 1300 tokens, q / k / v on 192-row tiles, whole / 256-row tiles, last round split 3003 / 3040).  0: not for these rows.
    auto cost = [&](int bn, int bm) -> int64_t {
        const int m_tiles = (int)((m + bm - 1) / bm);
        int64_t tiles = 0;
        for (int s = 0; s < count; ++s) {
            if (bn == 112 && rows[s] % 112 != 0) return 0;
            tiles += (rows[s] + bn - 1) / bn;
        }
        const int ns = plan_split(dev, (int)(tiles * m_tiles), n_sb), sb_per = (n_sb + ns - 1) / ns;
        const TailPlan tail = single ? TailPlan{0} : plan_tail(dev, fmt, tiles * m_tiles, n_sb);
        if (tail.splits)
            return (((int64_t)(tail.whole / dev->num_cus) * n_sb + tail.sb + 2) * 1000 +
                    2500 * (tiles * m_tiles - tail.whole) * tail.splits * bm / (256 * dev->num_cus)) *
                   bn * (bm == 192 ? 7 : 8) * (q4k ? 106 : 103) / 100;
        const int64_t wgs = tiles * m_tiles * ((n_sb + sb_per - 1) / sb_per);
        return ((wgs + dev->num_cus - 1) / dev->num_cus) * bn * sb_per * (bm == 192 ? 7 : 8) * 1000;
    };
    // Tiles of 112 weight rows where every tensor's rows divide by 112 and the grid then takes fewer row-steps of its
    // busiest CU (14336 rows: 128 tiles instead of 112, so 256 instead of 224 workgroups at 512 activation rows, 512
    // instead of 448 for a gate / up pair).
    auto narrow = [&](int bm) {
        if (!q4k || single || shape == 4) return false;
        const int64_t c112 = cost(112, bm);
        return c112 > 0 && c112 < cost(128, bm);
    };
    auto tile = [&](int bm) { return F16Tile{narrow(bm) ? 112 : 128, bm, single}; };
    // up to 128 activation rows: 128 x 128 tiles, K split over workgroups to fill the chip
    if (shape == 2 || m <= 128) return tile(128);
    auto wide_cost = [&](int bm) { return narrow(bm) ? cost(112, bm) : cost(128, bm); };
    // up to 256 rows where the 128 x 128 tiles fill the chip and the 128 x 256 tiles would have to split K
    // (Q4_K 14336 x 4096 at 256 rows: 70.7 us against 80.3)
    int64_t n128 = 0;
    for (int s = 0; s < count; ++s) n128 += (rows[s] + 127) / 128;
    const int64_t fill = (3 * (int64_t)dev->num_cus) / 4;
    // up to 192 rows: one column of 192-row tiles, K split up to four ways, instead of two columns of 128.  us, 128 x 128 / 128 x
    // 192: 11008 x 4096, 140 rows 43.7 / 35.9, 180 rows 44.0 / 37.5; 14336 x 4096 42.6 / 36.2, 43.0 / 38.9; 8192 x 2048 23.2 / 19.5,
    // 23.5 / 21.8; level where eight would share a tile (4096 x 4096 22.9 / 22.9).  Not where the two columns are one round and need
    // no split (more tiles than half the CUs) and K is so short that the sum of the copies costs more than the empty half of a
    // column: 129 / 192 rows 9216 x 2048 24.6 / 24.1, 24.9 / 25.9, 12288 x 2048 26.3 / 27.0, 26.5 / 29.2, 14336 x 2048 24.7 / 26.2,
    // 24.9 / 27.8, 16384 x 2048 27.2 / 27.6, 27.4 / 29.1; 14336 x 2560 28.8 / 27.8, 29.1 / 30.6, 12288 x 2560 30.4 / 28.3, 30.8 /
    // 30.4; 14336 x 2816 31.8 / 30.3, 31.4 / 32.8, 14336 x 3072 32.9 / 30.3, 33.2 / 33.2; 18432 x 2048, two rounds, 44.4 / 29.9, 45.5
    // / 31.4.
    const bool whole128 = 4 * n128 > dev->num_cus && 2 * n128 <= dev->num_cus && n_sb <= (m <= 160 ? 9 : narrow(128) ? 11 : 10);
    if (q4k && shape == 0 && !single && m <= 192 && n_sb >= 8 && 4 * n128 >= dev->num_cus && !whole128) return tile(192);
    if (q4k && m <= 256 && n128 * ((m + 127) / 128) >= fill && n128 * ((m + 255) / 256) < fill) return tile(128);
    // short K (at most 16 super-blocks) on a grid that 128 x 256 tiles would have to split: 128 x 128 tiles halve the
    // split as long as they still fit one round (Q4_K 4096 x 4096 at 512 rows 35.5 against 36.8 us, at 1024 rows 50.9
    // against 54.2; 6144 x 4096 at 512 rows 44.8 against 47.1; with K = 14336 the split is cheap and the wider tile wins)
    // Not where the launch behind sums the copies anyway (the decoder's prompts: the norm, the rotation) and the wide tiles leave it
    // two: us of a prompt (four layers and the head), narrow / wide tiles: q / k / v of the 8B shape 300 tokens 1179 / 1143, 512 1381 /
    // 1366; o 700 tokens 1891 / 1852, 1B shape 1300 tokens 1327 / 1303, 7B 600 1700 / 1658.  (With four copies level: 8B 512 tokens, o as well
    // 1360, 256 tokens 894 / 915.)  Where the wide tiles are not split either there is nothing to sum, and the fuller round of narrow ones
    // is ahead: q / k / v of the 8B shape, 240 workgroups of 256, 520 tokens narrow / wide 1608 / 1621, 640 1815 / 1836.
    const bool cheap = dev->defer_split && plan_split(dev, (int)(n128 * ((m + 255) / 256)), n_sb) == 2;
    if (q4k && !cheap && shape == 0 && cols <= 4096 && n128 * ((m + 255) / 256) < fill && n128 * ((m + 127) / 128) <= dev->num_cus)
        return tile(128);
    if (single) return F16Tile{128, 256, true};
    // A grid of 128 x 256 tiles that fills the chip, where the 128 x 128 tiles take no more rounds of workgroups: the
    // wide grid's last round is then at most a third full and its last column of tiles half empty, and a round of the
    // narrower tiles is the shorter one (about 0.7).  us on 128 x 256 / 128 x 128 tiles, two rounds either way: 11008 x
    // 4096 at 513..640 rows (258 and 430 tiles) Q4_K 109 / 80, Q5_K 125 / 105, Q6_K 125 / 98, Q8_0 144 / 110, Q4_0
    // 138 / 116; 21760 x 2048 at 300 rows (340 and 510, the fullest grids that the rule takes) 60 / 47, 70 / 60, 69 / 59,
    // 80 / 64, 77 / 65; 9300 x 1024 at 890 rows 40 / 34, 45 / 41, 45 / 40, 52 / 44, 49 / 43.  Where it costs a round
    // more the wider tiles win: 32000 x 4096 at 300 rows, two against three, Q5_K and Q4_0 0.86x on the narrow ones.
    // Not where the wider tiles' last round is split and that leaves less to do (a step of 128 rows counts 6, for Q4_K 5): 11008 x 4096 at
    // 513 rows Q4_K 81 / 71, Q6_K 98 / 81, Q8_0 112 / 85; at 600 rows level, 98 / 91, 113 / 93.
    auto rounds = [&](int bm) { return (n128 * ((m + bm - 1) / bm) + dev->num_cus - 1) / dev->num_cus; };
    auto tail_pays = [&](int bm) {
        int64_t tiles = 0;
        const int bn = narrow(bm) ? 112 : 128;
        for (int s = 0; s < count; ++s) tiles += (rows[s] + bn - 1) / bn;
        return plan_tail(dev, fmt, tiles * ((m + bm - 1) / bm), n_sb).splits &&
               wide_cost(bm) < 950 * rounds(128) * n_sb * 128 * (q4k ? 5 : 6);
    };
    if (shape == 0 && !narrow(256) && n128 * ((m + 255) / 256) >= fill && rounds(128) <= rounds(256) && !tail_pays(192) && !tail_pays(256))
        return tile(128);
    // Tiles of 192 activation rows where they leave the busiest CU less to do: a last column of tiles that would be mostly
    // empty (300 rows are 2 x 192 as they are 2 x 256), or a grid that fills the rounds better (1300 rows against 4096
    // weight rows: 224 workgroups instead of 192).  Over thirteen weight shapes and seventeen row counts from 140 to 2048,
    // five formats, the rule takes them at 4 points of 10, 1.09x on the geometric mean there, 0.996x to 1.225x.  us before /
    // with them: Q4_K 14336 x 4096 at 300 rows 60.6 / 51.0, 4096 x 14336 at 560 rows 101 / 87.5; Q5_K 32000 x 4096 at 560
    // rows 199 / 179; Q8_0 11008 x 4096 at 300 rows 77 / 70; Q6_K 4096 x 4096 at 1300 rows 69.9 / 63.4.
    const bool rows192 = shape == 0 && wide_cost(192) < wide_cost(256);
    return tile(rows192 ? 192 : 256);
}

template <class F>
static int launch_shapes(candy_hip_device *dev, const F16Job *jobs, int count, const _Float16 *xh, int64_t m) {
    constexpr bool q4k = std::is_same<F, BigQ4K>::value;
    int64_t rows[3];
    for (int s = 0; s < count; ++s) rows[s] = jobs[s].w->rows;
    const F16Tile t = pick_tile(dev, jobs[0].w->fmt, rows, count, jobs[0].w->cols, m);
    if (t.single)
        return t.bm == 128 ? launch_big<F, 128, 128, 2, 4>(dev, jobs, count, xh, m) : launch_big<F, 128, 256, 2, 4>(dev, jobs, count, xh, m);
    if constexpr (q4k) {
        if (t.bn == 112 && t.bm == 128) return launch_big<F, 112, 128, 2, 4, true>(dev, jobs, count, xh, m);
        if (t.bn == 112 && t.bm == 192) return launch_big<F, 112, 192, 2, 4, true>(dev, jobs, count, xh, m);
        if (t.bn == 112) return launch_big<F, 112, 256, 2, 4, true>(dev, jobs, count, xh, m);
    }
    if (t.bm == 128) return launch_big<F, 128, 128, 2, 4, true>(dev, jobs, count, xh, m);
    if (t.bm == 192) return launch_big<F, 128, 192, 2, 4, true>(dev, jobs, count, xh, m);
    return launch_big<F, 128, 256, 2, 4, true>(dev, jobs, count, xh, m);
}

static int launch_jobs(candy_hip_device *dev, const F16Job *jobs, int count, const _Float16 *xh, int64_t m) {
    switch (jobs[0].w->fmt) {
    case CANDY_HIP_Q6_K: return launch_shapes<BigQ6K>(dev, jobs, count, xh, m);
    case CANDY_HIP_Q5_K: return launch_shapes<BigQ5K>(dev, jobs, count, xh, m);
    case CANDY_HIP_Q8_0: return launch_shapes<BigQ8_0>(dev, jobs, count, xh, m);
    case CANDY_HIP_Q4_0: return launch_shapes<BigQ4_0<false>>(dev, jobs, count, xh, m);
    case CANDY_HIP_Q4_0_GGML: return launch_shapes<BigQ4_0<true>>(dev, jobs, count, xh, m);
    default: return launch_shapes<BigQ4K>(dev, jobs, count, xh, m);
    }
}

// xh: fp16 activations [mmq_m_pad(m)][K]; rows past m may hold anything (EPI_SILU leaves what was there): a row reaches its own
// results only.
int launch_mmq_f16_big(candy_hip_device *dev, const candy_hip_qtensor *w, const _Float16 *xh, int64_t m, float *y,
                       const float *res) {
    if (mmq_f16_rows_covers(w, m) && dev->opt.f16_shape == 0 && dev->opt.f16_split == 0) return launch_mmq_f16_rows(dev, w, xh, m, y, res);
    const F16Job job{w, y, res};
    return launch_jobs(dev, &job, 1, xh, m);
}

// Two or three projections of the same activations (q / k / v) as one grid: their tiles fill the chip together where
// each alone would split K many ways (Llama-3-8B shape, 512 rows: 1024 x 4096 alone is 16 tiles).
bool mmq_f16_group_covers(const candy_hip_qtensor *const *ws, int count, int64_t m) {
    if (count < 2 || count > 3 || !ws[0]->dev->opt.prefill_qkv_group || ws[0]->dev->opt.mmq_fp16_only) return false;
    for (int s = 0; s < count; ++s) {
        if (!mmq_f16_big_covers(ws[s], m) || ws[s]->fmt != ws[0]->fmt || ws[s]->cols != ws[0]->cols) return false;
        if (s + 1 < count && ws[s]->rows % 128 != 0) return false;  // a tile belongs to one tensor
    }
    return true;
}

int launch_mmq_f16_group(candy_hip_device *dev, const candy_hip_qtensor *const *ws, float *const *ys, int count,
                         const _Float16 *xh, int64_t m) {
    CANDY_REQUIRE(mmq_f16_group_covers(ws, count, m), "internal: projections cannot share a grid");
    F16Job jobs[3];
    for (int s = 0; s < count; ++s) jobs[s] = F16Job{ws[s], ys[s], nullptr};
    return launch_jobs(dev, jobs, count, xh, m);
}

// Gate, up and silu(gate) * up in one launch (EPI_SILU), where a tile's sums are whole: the grid of 128 x 256 tiles has to
// fill the chip without a split of K.
static bool silu_fills(const candy_hip_device *dev, int64_t rows, int64_t m) {
    return (rows / 64) * ((m + 255) / 256) >= (3 * (int64_t)dev->num_cus) / 4;
}

bool mmq_f16_silu_covers(const candy_hip_qtensor *gate, const candy_hip_qtensor *up, int64_t m) {
    const candy_hip_qtensor *const ws[2] = {gate, up};
    const Options &opt = gate->dev->opt;
    return opt.prefill_fold_silu && opt.f16_shape == 0 && opt.f16_split == 0 && m > 128 && gate->rows == up->rows && gate->rows % 64 == 0 &&
           mmq_f16_group_covers(ws, 2, m) && silu_fills(gate->dev, gate->rows, m) && f16_roles_fit(gate->fmt, 64, gate->cols);
}

template <class F, int BM>
static int launch_silu(candy_hip_device *dev, const candy_hip_qtensor *gate, const candy_hip_qtensor *up, const _Float16 *xh, int64_t m,
                       _Float16 *act) {
    const int N = (int)gate->rows, K = (int)gate->cols, n_tiles = N / 64, m_tiles = (int)((m + BM - 1) / BM);
    F16Group grp{};
    grp.count = 2;
    grp.act = act;
    grp.seg[0] = F16Seg{(const uint8_t *)gate->data, nullptr, nullptr, N, 0};
    grp.seg[1] = F16Seg{(const uint8_t *)up->data, nullptr, nullptr, N, 0};
    constexpr size_t smem = pc_lds<F>();
    auto kern = k_mmq_f16_pc<F, 128, BM, EPI_SILU>;
    CANDY_HIP_TRY(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
    hipLaunchKernelGGL(kern, dim3((unsigned)(n_tiles * m_tiles)), dim3(512), smem, dev->stream, grp, xh, (int)m, K, n_tiles, m_tiles,
                       K >> 8, (size_t)0, F16Tail{});
    CANDY_LAUNCH_CHECK();
    return CANDY_HIP_OK;
}

int launch_mmq_f16_silu(candy_hip_device *dev, const candy_hip_qtensor *gate, const candy_hip_qtensor *up, const _Float16 *xh, int64_t m,
                        _Float16 *act) {
    CANDY_REQUIRE(mmq_f16_silu_covers(gate, up, m), "internal: gate and up cannot share tiles");
    // the tiles of fewer activation rows by the rules of launch_shapes
    auto rounds = [&](int bm) { return (gate->rows / 64 * ((m + bm - 1) / bm) + dev->num_cus - 1) / dev->num_cus; };
    const int bm = rounds(128) <= rounds(256) ? 128 : 7 * rounds(192) < 8 * rounds(256) ? 192 : 256;
#define CANDY_SILU(F)                                                                                                     \
    return bm == 128 ? launch_silu<F, 128>(dev, gate, up, xh, m, act)                                                     \
                     : bm == 192 ? launch_silu<F, 192>(dev, gate, up, xh, m, act) : launch_silu<F, 256>(dev, gate, up, xh, m, act)
    switch (gate->fmt) {
    case CANDY_HIP_Q6_K: CANDY_SILU(BigQ6K);
    case CANDY_HIP_Q5_K: CANDY_SILU(BigQ5K);
    case CANDY_HIP_Q8_0: CANDY_SILU(BigQ8_0);
    case CANDY_HIP_Q4_0: CANDY_SILU(BigQ4_0<false>);
    case CANDY_HIP_Q4_0_GGML: CANDY_SILU(BigQ4_0<true>);
    default: CANDY_SILU(BigQ4K);
    }
#undef CANDY_SILU
}

}  // namespace candy

// The rules above, for their tests (no device needed): weight rows * 1000 + activation rows of a tile, negative where every wavefront has
// both roles; whether gate and up of a prompt share tiles with SiLU.
extern "C" int candy_test_f16_tile(int fmt, const int64_t *rows, int count, int64_t cols, int64_t m, int num_cus, int deferred) {
    candy_hip_device dev;
    candy::SplitPending pend;
    dev.num_cus = num_cus;
    if (deferred) dev.defer_split = &pend;
    const candy::F16Tile t = candy::pick_tile(&dev, fmt, rows, count, cols, m);
    return (t.single ? -1 : 1) * (t.bn * 1000 + t.bm);
}
// tile, and plan: tiles, those of them that are whole, workgroups and super-blocks of each of the others (0: there are none),
// workgroups of every tile where K is split throughout.
extern "C" int candy_test_f16_tail(int fmt, const int64_t *rows, int count, int64_t cols, int64_t m, int num_cus, int deferred, int *plan) {
    const int code = candy_test_f16_tile(fmt, rows, count, cols, m, num_cus, deferred);
    const int bn = std::abs(code) / 1000, bm = std::abs(code) % 1000;
    candy_hip_device dev;
    dev.num_cus = num_cus;
    int64_t tiles = 0;
    for (int s = 0; s < count; ++s) tiles += (rows[s] + bn - 1) / bn;
    tiles *= (m + bm - 1) / bm;
    const int n_sb = (int)(cols >> 8), all = candy::plan_split(&dev, (int)tiles, n_sb);
    const candy::TailPlan t = all == 1 && code > 0 ? candy::plan_tail(&dev, fmt, tiles, n_sb) : candy::TailPlan{(int)tiles};
    plan[0] = (int)tiles; plan[1] = t.whole; plan[2] = t.splits; plan[3] = t.sb; plan[4] = all;
    return code;
}
extern "C" int candy_test_f16_silu(int fmt, int64_t rows, int64_t cols, int64_t m, int num_cus) {
    candy_hip_device dev;
    dev.num_cus = num_cus;
    candy_hip_qtensor w;
    w.dev = &dev; w.fmt = fmt; w.rows = rows; w.cols = cols;
    return candy::mmq_f16_silu_covers(&w, &w, m);
}
