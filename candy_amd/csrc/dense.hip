// bfloat16 weights [rows, cols]: upload, row gather and the contraction y = epilogue(x . W^T).
//   k_dense_mv      one activation row: every weight row is streamed once by one wavefront, the activations wait in LDS
//                   (bfloat16 or f32 activations; HBM-bound).  Optional prologue: the norms in front of the contraction.
//   k_dense_mm      prompt batches of up to 64 rows, bfloat16 activations: v_mfma_f32_16x16x32_bf16 over LDS tiles filled
//                   by direct global-to-LDS loads, two stages; optionally split along K
//   k_dense_big     longer prompts: the same with tiles of 128 .. 256 x 128 or 256, fragments read a half stage ahead
//   k_dense_mm_f32  prompt batches, f32 activations: v_mfma_f32_16x16x4_f32, weights widened exactly
// Prompt batches also come with block-diagonal weights, and with their rows dealt to experts (GroupedRows).
// Weights are stored with both sides padded to multiples of 64 by zeros, so no kernel has a ragged edge in K, and the
// padded rows come out as epilogue(0) = 0.  (No counterpart in the reference, which has no bfloat16.)
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "dense.h"

namespace candy {

constexpr int EPI_NONE = CANDY_HIP_EPI_NONE, EPI_RELU2 = CANDY_HIP_EPI_SQUARED_RELU, EPI_CAP = CANDY_HIP_EPI_SOFTCAP,
              EPI_ACT = CANDY_HIP_EPI_ACT;
constexpr bool to_act(int epi) { return epi == EPI_RELU2 || epi == EPI_ACT; }  // the result is in the activation format

struct EpiArgs {
    float scale, cap;
};

template <int EPI>
__device__ __forceinline__ float epilogue(float z, const EpiArgs &e) {
    if (EPI == EPI_RELU2) {
        const float r = fmaxf(z, 0.0f);
        return r * r;
    }
    if (EPI == EPI_CAP) {
        z *= e.scale;
        return e.cap > 0.0f ? e.cap * tanhf(z / e.cap) : z;
    }
    return z;
}

// ------------------------------------------------------------------ one row
// The norms in front of the contraction (launch_norm_chain's arithmetic), for a kernel that runs them in its prologue.  What its
// first loads need are plain arguments of the kernel (they arrive in registers with the wavefront); this is the rest.  A norm's bias
// lies behind its weights; of two norms both have one (every norm of a Suvazen model has) or none has (Gulisun).
struct NormPro {
    const float *step;
    float *x_out;
    float mult, eps;
    int cols;
};
struct MvNorms {  // the plain arguments
    const float *x, *y, *post_w, *pre_w;
    int flags;    // MV_*
    NormPro rest;
};
enum { MV_Y = 1, MV_BIAS = 2, MV_RMS = 4, MV_PRE = 8 };

// Sum over the workgroup's wavefronts (at most 16), in every thread.  red: 16 floats of this sum's own, zero from the last
// wavefront on; one barrier.
__device__ __forceinline__ float pro_sum(float v, float *red) {
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    f32x4 r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = *(const f32x4 *)(red + 4 * i);
    float t = r[0][0];
#pragma unroll
    for (int w = 1; w < 16; ++w) t += r[w >> 2][w & 3];
    return t;
}

template <class AT> constexpr int mv_lds_values() { return sizeof(AT) == 2 ? 16384 : 8192; }  // 32 KB: whole steps
template <int R> constexpr int mv_unroll() { return 8 / R; }                                  // 8 KB requested per step

// One workgroup of W wavefronts per CU where the rows go round (launch_mv picks W and R so that they do), R weight rows
// per wavefront.  Two steps of weights are in flight, the first two requested right behind the activations and in front of
// everything that waits.  NV > 0: the activations are made here, by the norm chain in front of the contraction
// (NV float4 per thread); every workgroup repeats it, workgroup 0 writes the new residual row.
//   What bounds it: long weights, memory (128256 x 2048 at 6.8 TB/s); a layer's projections, the launch, the first round trip and, with
// norms, their two to four sums over the workgroup.  Requests are served in the order they are made, so the row comes in front of the
// weights; a step that was only requested once the row was staged (or the norms were done) cost a second round trip.  A sum is one
// barrier with its sixteen terms read together, not two barriers and a loop.  us, one step and in that order / so: 128256 x 2048 87.6 /
// 77.5, 102400 x 2048 70.5 / 63.2, the router of 64 experts 6.4 / 4.4; a decode step of the 1B-shaped Suvazen decoder, 1700 positions,
// 705 / 665, of the fine Gulisun one 302 / 288.
template <class AT, int R, int EPI, int NV>
__global__ __launch_bounds__(1024) void k_dense_mv(const void *__restrict__ xv_, const bf16 *__restrict__ W, int K, int rows,
                                                   const float *__restrict__ ny, const float *__restrict__ post_w,
                                                   const float *__restrict__ pre_w, int flags, void *__restrict__ yv, int n_store, const EpiArgs ea, const NormPro np) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass knows no buffer descriptors
    constexpr int U = mv_unroll<R>(), STEP = U * 512, CH = mv_lds_values<AT>();
    __shared__ __align__(16) AT xs[CH];
    __shared__ __align__(16) float red[NV > 0 ? 64 : 4];  // sixteen for each sum
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int threads = blockDim.x;
    const int row0 = (blockIdx.x * (threads >> 6) + wave) * R;
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.0f;
    // A weight row through a descriptor of its own: a lane's place is one offset, and what lies past the row comes as zeros.
    constexpr int NT = 2;  // nontemporal
    __amdgpu_buffer_rsrc_t wr[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
        wr[r] = __builtin_amdgcn_make_buffer_rsrc((void *)(W + (size_t)min(row0 + r, rows - 1) * K), 0, (int)(2u * (uint32_t)K), 0x00027000);
    auto fetch = [&](u32x4v (&w)[R][U], int k0) __attribute__((always_inline)) {
        const uint32_t at = 2u * (uint32_t)k0 + (uint32_t)lane * 16;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int r = 0; r < R; ++r)
                w[r][u] = __builtin_bit_cast(u32x4v, __builtin_amdgcn_raw_buffer_load_b128(wr[r], at + u * 1024, 0, NT));
    };
    auto multiply = [&](const u32x4v (&w)[R][U], int k0) __attribute__((always_inline)) {
        const AT *xp = xs + (k0 & (CH - 1)) + lane * 8;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float xf[8];
            lds8(xp + u * 512, xf);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float wf[8];
                widen8(w[r][u], wf);
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[r] = fmaf(wf[e], xf[e], acc[r]);
            }
            if (u & 1) __builtin_amdgcn_sched_barrier(0);  // two pieces of x at a time: all of them do not fit beside two steps of weights
        }
    };
    constexpr int PER = 16 / sizeof(AT);
    const AT *x = (const AT *)xv_;
    auto piece = [&](int k) __attribute__((always_inline)) { return k < K ? *(const u32x4v *)(x + k) : u32x4v{0, 0, 0, 0}; };
    u32x4v wa[R][U], wb[R][U];
    if constexpr (NV > 0) {
        f32x4 xv[NV], yv4[NV];
        const f32x4 zero{0.f, 0.f, 0.f, 0.f};
        auto load = [&](const float *p, f32x4 (&d)[NV]) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < NV; ++i) d[i] = (tid + threads * i) * 4 < K ? *(const f32x4 *)(p + (tid + threads * i) * 4) : zero;
        };
        f32x4 wv[NV], bv[NV], pw[NV], pb[NV];
#pragma unroll
        for (int i = 0; i < NV; ++i) bv[i] = pb[i] = zero;
        load((const float *)xv_, xv);
        if (flags & MV_Y) {
            load(ny, yv4);
            load(post_w, pw);
            if (flags & MV_BIAS) load(post_w + K, pb);
        }
        if (flags & MV_PRE) {
            load(pre_w, wv);
            if (flags & MV_BIAS) load(pre_w + K, bv);
        }
        fetch(wa, 0);
        if (NV == 1) fetch(wb, STEP);
        const int n_waves = threads >> 6;
        if (tid < 64 && (tid & 15) >= n_waves) red[tid] = 0.0f;
        const float inv_n = 1.0f / (float)np.cols;
        auto normalize = [&](f32x4 (&d)[NV], const f32x4 (&w)[NV], const f32x4 (&b)[NV], float *sums) __attribute__((always_inline)) {
            float mean = 0.0f;
            if (!(flags & MV_RMS)) {
                float s = 0.0f;
#pragma unroll
                for (int i = 0; i < NV; ++i) s += (d[i][0] + d[i][1]) + (d[i][2] + d[i][3]);
                mean = pro_sum(s, sums) * inv_n;
            }
            float q = 0.0f;
#pragma unroll
            for (int i = 0; i < NV; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    d[i][j] = (tid + threads * i) * 4 + j < np.cols ? d[i][j] - mean : 0.0f;
                    q += d[i][j] * d[i][j];
                }
            const float rstd = 1.0f / sqrtf(pro_sum(q, sums + 16) * inv_n + np.eps);
#pragma unroll
            for (int i = 0; i < NV; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) d[i][j] = d[i][j] * rstd * w[i][j] + b[i][j];  // w = b = 0 past the row
        };
        if (flags & MV_Y) {
            normalize(yv4, pw, pb, red);
#pragma unroll
            for (int i = 0; i < NV; ++i) xv[i] += np.mult * yv4[i];
        }
        if (np.step) {
            load(np.step, yv4);
#pragma unroll
            for (int i = 0; i < NV; ++i) xv[i] += yv4[i];
        }
        if (np.x_out && blockIdx.x == 0) {
#pragma unroll
            for (int i = 0; i < NV; ++i)
                if ((tid + threads * i) * 4 < K) *(f32x4 *)(np.x_out + (tid + threads * i) * 4) = xv[i];
        }
        if (flags & MV_PRE) normalize(xv, wv, bv, red + 32);
        if (NV > 1) fetch(wb, STEP);  // no registers for it any sooner
        typedef AT at4 __attribute__((ext_vector_type(4)));
        const int n = (K + STEP - 1) / STEP * STEP;
#pragma unroll
        for (int i = 0; i < NV; ++i)
            if ((tid + threads * i) * 4 < n) *(at4 *)&xs[(tid + threads * i) * 4] = __builtin_convertvector(xv[i], at4);
        for (int i = (tid + threads * NV) * 4; i < n; i += threads * 4) *(at4 *)&xs[i] = __builtin_convertvector(zero, at4);
    } else {
        // The first pieces of the row are requested in front of the weights: requests are served in order, and behind them the row
        // would come last.
        constexpr int FIRST = 2;
        u32x4v held[FIRST];
#pragma unroll
        for (int i = 0; i < FIRST; ++i) held[i] = piece((tid + threads * i) * PER);
        fetch(wa, 0);
        fetch(wb, STEP);
        __builtin_amdgcn_sched_barrier(0);
        const int n = min(CH, (K + STEP - 1) / STEP * STEP);
#pragma unroll
        for (int i = 0; i < FIRST; ++i)
            if ((tid + threads * i) * PER < n) *(u32x4v *)&xs[(tid + threads * i) * PER] = held[i];
        for (int i = (tid + threads * FIRST) * PER; i < n; i += threads * PER) *(u32x4v *)&xs[i] = piece(i);
    }
    __syncthreads();
    for (int k0 = 0; k0 < K; k0 += 2 * STEP) {
        if (NV == 0 && k0 && (k0 & (CH - 1)) == 0) {
            __syncthreads();  // the previous chunk is consumed
            const int n = min(CH, (K - k0 + STEP - 1) / STEP * STEP);
            for (int i = tid * PER; i < n; i += threads * PER) *(u32x4v *)&xs[i] = piece(k0 + i);
            __syncthreads();
        }
        multiply(wa, k0);
        fetch(wa, k0 + 2 * STEP);  // (steps past the row ask for nothing)
        if (k0 + STEP >= K) break;
        multiply(wb, k0 + STEP);
        fetch(wb, k0 + 3 * STEP);
    }
    float mine = 0.0f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float t = wave_sum(acc[r]);
        if (lane == r) mine = t;
    }
    if (lane < R && row0 + lane < n_store) {
        const float z = epilogue<EPI>(mine, ea);
        if (to_act(EPI)) ((AT *)yv)[row0 + lane] = (AT)z;
        else ((float *)yv)[row0 + lane] = z;
    }
#endif
}

// ------------------------------------------------------------------ prompt batches, bfloat16
// Tile: BN = 128 weight rows x BM = 64 activation rows, 64 values of K per stage.  A row of a stage is 128 bytes = eight
// 16-byte chunks; chunk c of row r sits in slot c ^ ((r >> 1) & 7), so that the 16 rows a fragment read touches spread
// over all banks.  A direct load writes 64 consecutive 16-byte slots, so the permutation is in the addresses it reads.
// GROUPED: the row tiles come from a list in device memory (of BM rows at most each), one expert's weights per tile.
template <int EPI, bool GROUPED>
__global__ __launch_bounds__(256, 2) void k_dense_mm(const bf16 *__restrict__ W, const bf16 *__restrict__ X, void *__restrict__ yv,
                                                     int M, int Np, int ld, int ldx, int k_slice, int64_t ldy, int n_store,
                                                     size_t split_stride, int m_tiles, int n_tiles, int block_rows, const EpiArgs ea,
                                                     const GroupedRows gr) {
    constexpr int BN = 128, BM = 64, BK = 64, ROWS = BN + BM, LOADS = ROWS / 32;
    constexpr int TN = 4, TM = BM / 32;
    __shared__ __align__(16) u32x4v s[2][ROWS * 8];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // each XCD takes a run of neighbouring tiles (workgroups are dealt to the XCDs round robin); the activation tiles of
    // one weight tile are neighbours
    if (GROUPED) m_tiles = *gr.n_tiles;
    const int total = m_tiles * n_tiles;
    int t = blockIdx.x;
    if (GROUPED && t >= total) return;
    {
        const int per = total >> 3, full = per << 3;
        if (t < full) t = (t & 7) * per + (t >> 3);
    }
    int n0 = (t / m_tiles) * BN, m0 = (t % m_tiles) * BM;
    const int *perm = nullptr;
    if (GROUPED) {
        // expert by expert; within one, its row tiles of one weight tile are neighbours
        GroupTile tile = gr.tiles[t / n_tiles];
        const int local = t - tile.tile0 * n_tiles, nt = local / tile.of_expert;
        n0 = nt * BN;
        tile = gr.tiles[tile.tile0 + local - nt * tile.of_expert];
        W += (size_t)tile.expert * Np * ld;
        perm = gr.perm + tile.first;
        M = tile.count;
        m0 = 0;
    }
    if (block_rows) X += (size_t)(n0 / block_rows) * ld;
    const int kbeg = blockIdx.y * k_slice, kend = min(kbeg + k_slice, ld);
    const bf16 *src[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int r = (wave + 4 * i) * 8 + (lane >> 3);
        const int c = (lane & 7) ^ ((r >> 1) & 7);
        int xr = min(m0 + max(r - BN, 0), M - 1);
        if (GROUPED) xr = perm[xr] / gr.x_div;
        src[i] = (r < BN ? W + (size_t)min(n0 + r, Np - 1) * ld : X + (size_t)xr * ldx) + kbeg + c * 8;
    }
    auto load = [&](int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src[i],
                                             (__attribute__((address_space(3))) void *)&s[stage][(wave + 4 * i) * 64], 16, 0, 0);
            src[i] += BK;
        }
    };
    f32x4 acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int wn = (wave >> 1) * 64, wm = BN + (wave & 1) * (BM / 2);
    const int r16 = lane & 15, g = lane >> 4;
    const int sw = (r16 >> 1) & 7;  // every tile starts at a multiple of 16 rows: the same swizzle for all of a lane's reads
    auto compute = [&](int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            bf16x8 a[TN], b[TM];
            const int slot = (kk * 4 + g) ^ sw;
#pragma unroll
            for (int i = 0; i < TN; ++i) a[i] = __builtin_bit_cast(bf16x8, s[stage][(wn + i * 16 + r16) * 8 + slot]);
#pragma unroll
            for (int j = 0; j < TM; ++j) b[j] = __builtin_bit_cast(bf16x8, s[stage][(wm + j * 16 + r16) * 8 + slot]);
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    };
    const int n_it = (kend - kbeg) / BK;
    load(0);
    for (int it = 0; it < n_it; ++it) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();  // the stage has landed for every wavefront, and the other one is consumed
        if (it + 1 < n_it) load((it + 1) & 1);
        compute(it & 1);
    }
    // C layout: column r16 is the activation row, rows 4g .. 4g+3 are four neighbouring outputs of it
#pragma unroll
    for (int j = 0; j < TM; ++j) {
        int m = m0 + wm - BN + j * 16 + r16;
        if (m >= M) continue;
        if (GROUPED) m = perm[m];
#pragma unroll
        for (int i = 0; i < TN; ++i) {
            const int n = n0 + wn + i * 16 + 4 * g;
            f32x4 z = acc[i][j];
#pragma unroll
            for (int e = 0; e < 4; ++e) z[e] = epilogue<EPI>(z[e], ea);
            if (to_act(EPI)) {
                if (n < n_store) *(bf16x4 *)((bf16 *)yv + (size_t)m * ldy + n) = __builtin_convertvector(z, bf16x4);
            } else if (EPI == EPI_NONE) {
                float *y = (float *)yv + blockIdx.y * split_stride + (size_t)m * ldy + n;
                if (n + 3 < n_store && (ldy & 3) == 0) *(f32x4 *)y = z;
                else
                    for (int e = 0; e < 4; ++e)
                        if (n + e < n_store) y[e] = z[e];
            } else {
                float *y = (float *)yv + (size_t)m * ldy + n;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < n_store) y[e] = z[e];
            }
        }
    }
}

// ------------------------------------------------------------------ prompt batches, bfloat16, large tiles
// Tile: BN weight rows x BM activation rows, 64 values of K per stage, one workgroup of eight wavefronts (WN x WM) per CU;
// a stage lies in LDS as in k_dense_mm.  What bounds it: the chip's power (at 2000 rows the clock falls
// from 2.4 to 2.0 GHz) and the matrix instructions, busy 50 - 61 % of a CU's cycles (a step of 256 x 256 is 2 048 cycles of them),
// with fragment reads and the wait for a stage in between; no bank conflicts.  Against two workgroups per CU of 128 x 128 tiles whose four wavefronts read all fragments of a
// half stage and then multiply: a wavefront's tile is up to twice as large, so that a fragment read meets more matrix
// instructions (an eighth to a quarter fewer LDS reads); the fragments of the next half stage are read while this one is
// multiplied; a stage's loads are requested when its place is free and have a step (two with three stages) to arrive.
// us, 128 x 128 -> the tile big_tile() picks: 2000 rows, 14336 x 4096 260 -> 215, 5120 x 4096 128 -> 91, 4096 x 4096 79 -> 72,
// 4096 x 14336 248 -> 207; 512 rows, 14336 x 4096 80 -> 72, 4096 x 14336 79 -> 67.  The 32x32x16 instruction (same reads, half
// the instructions) is 4 - 7 % slower, stages of 32 values with five of them in LDS no faster (fewer cycles, lower clock).
struct BigArgs {
    const bf16 *W, *X;           // from the tile's first rows and this workgroup's first value of K on
    int64_t w_values, x_values;  // readable from there
    const int *perm;             // grouped: the tile's rows
    int x_div;
    int rows, ld, ldx, n_it;     // activation rows, stages
};
constexpr int big_stages(int rows) { return 3 * rows * 128 <= 160 * 1024 ? 3 : 2; }

// The products of one tile whose wavefronts hold TM fragments of 16 activation rows each, every WM-th from `wm` on.
template <int BN, int WN, int TN, int TM, int TMAX, bool GROUPED>
__device__ __forceinline__ void big_products(const BigArgs &a, u32x4v *s, f32x4 (&acc)[TN][TMAX], int wave, int lane) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass knows no buffer descriptors
    constexpr int WM = 8 / WN, BK = 64, ROWS = BN + TM * WM * 16;
    constexpr int PIECES = ROWS / 8, LOADS = (PIECES + 7) / 8;  // wavefront loads of 1 KB per stage, per wavefront
    constexpr int STAGES = big_stages(ROWS);
    // A wavefront load takes eight rows of one matrix through a buffer descriptor: rows past the matrix come as zeros, and
    // the step along K is a scalar offset.  (Loads of the global_load_lds form count as LDS reads to the compiler's wait
    // counting: every fragment read behind one would wait for all of them.)
    auto describe = [](const bf16 *p, int64_t values) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, values >= 1ll << 31 ? -1 : (int)(uint32_t)(values * 2), 0x00027000);
    };
    const __amdgpu_buffer_rsrc_t rw = describe(a.W, a.w_values), rx = describe(a.X, a.x_values);
    uint32_t off[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int piece = min(wave + 8 * i, PIECES - 1);  // a spare load repeats the last piece
        const int r = piece * 8 + (lane >> 3);
        const int c = (lane & 7) ^ ((r >> 1) & 7);
        int row = r < BN ? r : r - BN;
        if (GROUPED && r >= BN) row = a.perm[min(row, a.rows - 1)] / a.x_div;
        off[i] = (uint32_t)row * (uint32_t)(r < BN ? a.ld : a.ldx) * 2 + c * 16;
    }
    int k_off = 0;
    auto load = [&](int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int piece = min(wave + 8 * i, PIECES - 1);
            auto *to = (__attribute__((address_space(3))) void *)(s + stage * ROWS * 8 + piece * 64);
            if (8 * i + 7 < BN / 8) __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, to, 16, off[i], k_off, 0, 0);
            else if (8 * i >= BN / 8) __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, to, 16, off[i], k_off, 0, 0);
            else if (piece < BN / 8) __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, to, 16, off[i], k_off, 0, 0);
            else __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, to, 16, off[i], k_off, 0, 0);
        }
        k_off += BK * 2;
    };
    const int wn = (wave / WM) * (BN / WN), wm = BN + (wave % WM) * 16;
    const int r16 = lane & 15, g = lane >> 4;
    const int sw = (r16 >> 1) & 7;
    struct Frags { bf16x8 a[TN], b[TM]; };
    auto read = [&](Frags &f, int stage, int kk) __attribute__((always_inline)) {
        const u32x4v *p = s + stage * ROWS * 8 + r16 * 8 + ((kk * 4 + g) ^ sw);
#pragma unroll
        for (int i = 0; i < TN; ++i) f.a[i] = __builtin_bit_cast(bf16x8, p[(wn + i * 16) * 8]);
#pragma unroll
        for (int j = 0; j < TM; ++j) f.b[j] = __builtin_bit_cast(bf16x8, p[(wm + j * WM * 16) * 8]);
    };
    auto multiply = [&](const Frags &f) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
            for (int j = 0; j < TM; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.a[i], f.b[j], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
    };
    // s_waitcnt in the form the compiler's own counting sees: no LDS reads left, all vector loads or a stage's in flight
    constexpr int ARRIVED = 0x0070, ARRIVED_BUT_ONE = 0x0070 | (LOADS & 15) | (LOADS >> 4) << 14;
    const int n_it = a.n_it;
    load(0);
    if (n_it > 1) load(1);
    if (n_it > 1) __builtin_amdgcn_s_waitcnt(ARRIVED_BUT_ONE);
    else __builtin_amdgcn_s_waitcnt(ARRIVED);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    Frags f0, f1;
    read(f0, 0, 0);
    if (STAGES == 3 && n_it > 2) load(2);
    int cur = 0, nxt = 1, last = 2;  // stage in use, the next one, and (three stages) the one behind that
    // What a step does is fixed at compile time, so that the compiler's counts of reads in flight are exact.  fill: a
    // further stage is requested; left: a stage is in flight behind the next one when that one's arrival is waited for
    auto step = [&](auto fill, auto left, auto more) __attribute__((always_inline)) {
        read(f1, cur, 1);
        multiply(f0);
        if (more) {
            __builtin_amdgcn_s_waitcnt(left ? ARRIVED_BUT_ONE : ARRIVED);  // this stage is read, and the next one is there
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            read(f0, nxt, 0);
            if (fill) load(cur);
        }
        multiply(f1);
        const int was = cur;
        cur = nxt;
        nxt = STAGES == 3 ? last : was;
        last = was;
    };
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    int it = 0;
    for (; it + STAGES < n_it; ++it) step(yes, std::bool_constant<STAGES == 3>{}, yes);
    if (STAGES == 3 && it + 2 < n_it) { step(no, yes, yes); ++it; }
    for (; it + 1 < n_it; ++it) step(no, no, yes);
    step(no, no, no);
#endif
}

template <int BN, int BM, int WN, int EPI, bool GROUPED>
__global__ __launch_bounds__(512, 2) void k_dense_big(const bf16 *__restrict__ W, const bf16 *__restrict__ X, void *__restrict__ yv, int M, int Np,
                                                      int ld, int ldx, int k_slice, int64_t ldy, int n_store, size_t split_stride, int m_tiles,
                                                      int n_tiles, int block_rows, const EpiArgs ea, const GroupedRows gr) {
    constexpr int WM = 8 / WN, TN = BN / WN / 16, TMAX = BM / WM / 16;
    static_assert(BN % (16 * WN) == 0 && TMAX == 4, "whole fragments, four of them along the activation rows");
    constexpr int most = std::max(std::max(big_stages(BN + BM / 4) * (BN + BM / 4), big_stages(BN + BM / 2) * (BN + BM / 2)),
                                  std::max(big_stages(BN + BM / 4 * 3) * (BN + BM / 4 * 3), big_stages(BN + BM) * (BN + BM)));
    __shared__ __align__(16) u32x4v s[most * 8];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int n0, m0 = 0;
    const int *perm = nullptr;
    if (GROUPED) {
        // expert by expert, an XCD taking neighbours; within one, its row tiles of one weight tile are neighbours
        const int total = *gr.n_tiles * n_tiles, per = total >> 3, full = per << 3;
        int t = blockIdx.x;
        if (t >= total) return;
        if (t < full) t = (t & 7) * per + (t >> 3);
        GroupTile tile = gr.tiles[t / n_tiles];
        const int local = t - tile.tile0 * n_tiles, nt = local / tile.of_expert;
        n0 = nt * BN;
        tile = gr.tiles[tile.tile0 + local - nt * tile.of_expert];
        W += (size_t)tile.expert * Np * ld;
        perm = gr.perm + tile.first;
        M = tile.count;
    } else {
        int t = blockIdx.x;
        const int total = m_tiles * n_tiles, per = total >> 3, full = per << 3;
        if (t < full) t = (t & 7) * per + (t >> 3);
        n0 = t / m_tiles * BN;
        m0 = t % m_tiles * BM;
    }
    if (block_rows) X += (size_t)(n0 / block_rows) * ld;
    const int kbeg = blockIdx.y * k_slice, kend = min(kbeg + k_slice, ld);
    f32x4 acc[TN][TMAX];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TMAX; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int rows = min(M - m0, BM);
    const BigArgs a{W + (size_t)n0 * ld + kbeg, X + (size_t)m0 * ldx + kbeg, (int64_t)(Np - n0) * ld - kbeg,
                    GROUPED ? (int64_t)1 << 40 : (int64_t)(M - m0) * ldx - kbeg, perm, GROUPED ? gr.x_div : 1, rows, ld, ldx, (kend - kbeg) / 64};
    // a tile of fewer rows takes as many quarters as it fills: the wavefronts share them fragment by fragment
    switch ((rows + BM / 4 - 1) / (BM / 4)) {
    case 1: big_products<BN, WN, TN, 1, TMAX, GROUPED>(a, s, acc, wave, lane); break;
    case 2: big_products<BN, WN, TN, 2, TMAX, GROUPED>(a, s, acc, wave, lane); break;
    case 3: big_products<BN, WN, TN, 3, TMAX, GROUPED>(a, s, acc, wave, lane); break;
    default: big_products<BN, WN, TN, 4, TMAX, GROUPED>(a, s, acc, wave, lane); break;
    }
    const int r16 = lane & 15, g = lane >> 4, wn = (wave / WM) * (BN / WN);
#pragma unroll
    for (int j = 0; j < TMAX; ++j) {
        int m = m0 + (j * WM + wave % WM) * 16 + r16;
        if (m >= M) continue;
        if (GROUPED) m = perm[m];
#pragma unroll
        for (int i = 0; i < TN; ++i) {
            const int n = n0 + wn + i * 16 + 4 * g;
            f32x4 z = acc[i][j];
#pragma unroll
            for (int e = 0; e < 4; ++e) z[e] = epilogue<EPI>(z[e], ea);
            if (to_act(EPI)) {
                if (n < n_store) *(bf16x4 *)((bf16 *)yv + (size_t)m * ldy + n) = __builtin_convertvector(z, bf16x4);
            } else if (EPI == EPI_NONE) {
                float *y = (float *)yv + blockIdx.y * split_stride + (size_t)m * ldy + n;
                if (n + 3 < n_store && (ldy & 3) == 0) *(f32x4 *)y = z;
                else
                    for (int e = 0; e < 4; ++e)
                        if (n + e < n_store) y[e] = z[e];
            } else {
                float *y = (float *)yv + (size_t)m * ldy + n;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < n_store) y[e] = z[e];
            }
        }
    }
}

// ------------------------------------------------------------------ prompt batches, bfloat16, few tiles
// Tile: 32 weight rows x BM = 32 or 64 activation rows, four wavefronts, K whole: for contractions whose epilogue does not let K be
// split and whose large tiles leave most of the chip idle.  There a workgroup's walk along K is a chain of stage latencies
// (0.8 us each, 64 values); here up to five stages are in flight, and four times as many workgroups walk.  What bounds it: the
// activations, which every workgroup reads.  A value's sum goes along K in the order of the other tiles: the same bits.
// us of a call with two conversions around it (6 us), before -> now: 2816 x 2048, 16 / 64 / 200 rows 20.9 / 22.1 / 23.2 -> 11.6 / 13.5 /
// 16.9; 6144 x 4096, 40 / 100 rows 39.0 / 35.4 -> 20.8 / 26.9; 14336 x 4096, 16 / 64 rows 40.3 / 44.5 -> 31.0 / 35.6.
constexpr int NARROW_BN = 32;
template <int EPI, int BM>
__global__ __launch_bounds__(256, 2) void k_dense_narrow(const bf16 *__restrict__ W, const bf16 *__restrict__ X, bf16 *__restrict__ y, int M,
                                                         int Np, int ld, int ldx, int64_t ldy, int n_store, int m_tiles, const EpiArgs ea) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass knows no buffer descriptors
    constexpr int BN = NARROW_BN, BK = 64, ROWS = BN + BM, PIECES = ROWS / 8, LOADS = PIECES / 4, STAGES = 6, TM = BM / 32;
    static_assert(PIECES % 4 == 0 && to_act(EPI), "every wavefront has as many loads; results are activations");
    __shared__ __align__(16) u32x4v s[STAGES * ROWS * 8];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = blockIdx.x / m_tiles * BN, m0 = blockIdx.x % m_tiles * BM;
    const int n_it = ld / BK;
    f32x4 acc[TM];
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int r16 = lane & 15, g = lane >> 4, sw = (r16 >> 1) & 7;
    const int wn = (wave >> 1) * 16, wm = BN + (wave & 1) * (BM / 2);
    auto describe = [](const bf16 *p, int64_t values) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, values >= 1ll << 31 ? -1 : (int)(uint32_t)(values * 2), 0x00027000);
    };
    const __amdgpu_buffer_rsrc_t rw = describe(W + (size_t)n0 * ld, (int64_t)(Np - n0) * ld),
                                 rx = describe(X + (size_t)m0 * ldx, (int64_t)(M - m0 - 1) * ldx + ld);
    uint32_t off[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int r = (wave + 4 * i) * 8 + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
        // activation rows past the last one repeat it
        off[i] = (r < BN ? (uint32_t)r * (uint32_t)ld : (uint32_t)min(r - BN, M - m0 - 1) * (uint32_t)ldx) * 2 + c * 16;
    }
    int k_off = 0;
    auto load = [&](int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            auto *to = (__attribute__((address_space(3))) void *)(s + stage * ROWS * 8 + (wave + 4 * i) * 64);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(4 * i < BN / 8 ? rw : rx, to, 16, off[i], k_off, 0, 0);  // pieces 0 .. 3 are W's
        }
        k_off += BK * 2;
    };
    auto compute = [&](int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const u32x4v *p = s + stage * ROWS * 8 + r16 * 8 + ((kk * 4 + g) ^ sw);
            const bf16x8 a = __builtin_bit_cast(bf16x8, p[wn * 8]);
#pragma unroll
            for (int j = 0; j < TM; ++j)
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8, p[(wm + j * 16) * 8]), acc[j], 0, 0, 0);
        }
    };
    // stages in flight behind the one waited for: STAGES - 2, none once the last one is requested
    constexpr int ARRIVED = 0x0070, BEHIND = LOADS * (STAGES - 2), ARRIVED_BUT = 0x0070 | (BEHIND & 15) | (BEHIND >> 4) << 14;
#pragma unroll
    for (int i = 0; i < STAGES - 1; ++i)
        if (i < n_it) load(i);
    int cur = 0;
    for (int it = 0; it < n_it; ++it) {
        if (it + STAGES - 1 <= n_it) __builtin_amdgcn_s_waitcnt(ARRIVED_BUT);
        else __builtin_amdgcn_s_waitcnt(ARRIVED);
        __builtin_amdgcn_s_barrier();  // this stage is there for every wavefront, and the one in front of it is consumed
        asm volatile("" ::: "memory");
        if (it + STAGES - 1 < n_it) load(cur == 0 ? STAGES - 1 : cur - 1);
        compute(cur);
        cur = cur + 1 == STAGES ? 0 : cur + 1;
    }
#pragma unroll
    for (int j = 0; j < TM; ++j) {
        const int m = m0 + wm - BN + j * 16 + r16, n = n0 + wn + 4 * g;
        if (m >= M) continue;
        f32x4 z = acc[j];
#pragma unroll
        for (int e = 0; e < 4; ++e) z[e] = epilogue<EPI>(z[e], ea);
        if (n < n_store) *(bf16x4 *)(y + (size_t)m * ldy + n) = __builtin_convertvector(z, bf16x4);
    }
#endif
}

// ------------------------------------------------------------------ prompt batches, f32 activations
template <int EPI, bool GROUPED>
__global__ __launch_bounds__(256) void k_dense_mm_f32(const bf16 *__restrict__ W, const float *__restrict__ X, float *__restrict__ yv,
                                                      int M, int ld, int ldx, int64_t ldy, int n_store, int block_rows,
                                                      const EpiArgs ea, const GroupedRows gr) {
    constexpr int B = 64, BK = 32, P = BK + 4;
    __shared__ __align__(16) float sw[B * P], sx[B * P];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n0 = blockIdx.x * B;
    int m0 = blockIdx.y * B;
    const int *perm = nullptr;
    if (GROUPED) {
        if ((int)blockIdx.y >= *gr.n_tiles) return;
        const GroupTile tile = gr.tiles[blockIdx.y];
        W += (size_t)tile.expert * gr.expert_rows * ld;
        perm = gr.perm + tile.first;
        M = tile.count;
        m0 = 0;
    }
    if (block_rows) X += (size_t)(n0 / block_rows) * ld;
    const int r16 = lane & 15, g = lane >> 4;
    const int wn = (wave >> 1) * 32, wm = (wave & 1) * 32;
    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int lr = tid >> 2, lc = (tid & 3) * 8;  // a row of the stage, 8 of its 32 values
    int xr = min(m0 + lr, M - 1);
    if (GROUPED) xr = perm[xr] / gr.x_div;
    for (int k0 = 0; k0 < ld; k0 += BK) {
        float wf[8], xf[8];
        widen8(*(const u32x4v *)(W + (size_t)(n0 + lr) * ld + k0 + lc), wf);
        lds8(X + (size_t)xr * ldx + k0 + lc, xf);
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            sw[lr * P + lc + e] = wf[e];
            sx[lr * P + lc + e] = xf[e];
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < BK; kk += 4) {
            float a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                a[i] = sw[(wn + i * 16 + r16) * P + kk + g];
                b[i] = sx[(wm + i * 16 + r16) * P + kk + g];
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        int m = m0 + wm + j * 16 + r16;
        if (m >= M) continue;
        if (GROUPED) m = perm[m];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int n = n0 + wn + i * 16 + 4 * g + e;
                if (n < n_store) yv[(size_t)m * ldy + n] = epilogue<EPI>(acc[i][j][e], ea);
            }
    }
}

// ------------------------------------------------------------------ launches
// Rows over wavefronts: with up to 64 rows per CU one workgroup per CU takes them all, its shape the one that leaves the
// fewest slots empty (the more wavefronts the better, from eight on); longer weights take many workgroups of 8 x 4.
MvShape mv_shape(const candy_hip_device *dev, int64_t rows) {
    const int64_t per_cu = (rows + dev->num_cus - 1) / dev->num_cus;
    if (per_cu > 64) return {8, 4};
    if (per_cu <= 8) return {8, 1};
    MvShape best{16, 4};
    int64_t best_cost = 1 << 30;
    for (int r : {1, 2, 4})
        for (int w = 8; w <= 16; ++w) {
            const int64_t slots = (int64_t)w * r;
            if (slots < per_cu) continue;
            const int64_t cost = (slots - per_cu) * 64 - w;
            if (cost < best_cost) { best_cost = cost; best = {w, r}; }
        }
    return best;
}

template <class AT, int R, int EPI>
static void launch_mv_nv(candy_hip_device *dev, const DenseLaunch &L, int waves, int nv, const MvNorms &np) {
    const int64_t per_wg = (int64_t)waves * R;
    const dim3 g((unsigned)((L.n_store + per_wg - 1) / per_wg)), b((unsigned)(64 * waves));
    const EpiArgs ea{L.scale, L.cap};
    const bf16 *W = (const bf16 *)L.w->data;
    const int K = (int)L.w->ld, rows = (int)L.w->rows_pad, ns = (int)L.n_store;
    auto launch = [&](auto kern, const void *x) {
        hipLaunchKernelGGL(kern, g, b, 0, dev->stream, x, W, K, rows, np.y, np.post_w, np.pre_w, np.flags, L.y, ns, ea, np.rest);
    };
    if constexpr (sizeof(AT) == 2 || (R == 1 && EPI == EPI_NONE)) {
        switch (nv) {
        case 1: launch(k_dense_mv<AT, R, EPI, 1>, np.x); return;
        case 2: launch(k_dense_mv<AT, R, EPI, 2>, np.x); return;
        default: break;
        }
    }
    launch(k_dense_mv<AT, R, EPI, 0>, L.x);
}

template <class AT, int R>
static void launch_mv_epi(candy_hip_device *dev, const DenseLaunch &L, int waves, int nv, const MvNorms &np) {
    switch (L.epi) {
    case EPI_RELU2: launch_mv_nv<AT, R, EPI_RELU2>(dev, L, waves, nv, np); break;
    case EPI_CAP: launch_mv_nv<AT, R, EPI_CAP>(dev, L, waves, nv, np); break;
    case EPI_ACT: launch_mv_nv<AT, R, EPI_ACT>(dev, L, waves, nv, np); break;
    default: launch_mv_nv<AT, R, EPI_NONE>(dev, L, waves, nv, np); break;
    }
}

template <class AT>
static int launch_mv(candy_hip_device *dev, const DenseLaunch &L, const MvShape &s, int nv = 0, const MvNorms &np = MvNorms{}) {
    switch (s.rows) {
    case 1: launch_mv_epi<AT, 1>(dev, L, s.waves, nv, np); break;
    case 2: launch_mv_epi<AT, 2>(dev, L, s.waves, nv, np); break;
    default: launch_mv_epi<AT, 4>(dev, L, s.waves, nv, np); break;
    }
    CANDY_LAUNCH_CHECK();
    return CANDY_HIP_OK;
}

int launch_dense_norm(candy_hip_device *dev, const DenseLaunch &L, const NormArgs &A) {
    // every workgroup repeats the norms: one per CU, or the launch of their own is the cheaper one
    const MvShape s = mv_shape(dev, L.n_store);
    const int per = 256 * s.waves, nv = (int)((L.w->ld + per - 1) / per);
    if (L.m != 1 || (L.f32 && (s.rows != 1 || L.epi != EPI_NONE)) || A.rows != 1 || A.y.copies != 1 || A.slots || A.row_ids ||
        A.x == A.x_out || nv > 2 || L.w->ld > (L.f32 ? mv_lds_values<float>() : mv_lds_values<bf16>()) || L.n_store > 64 * (int64_t)dev->num_cus)
        return CANDY_HIP_ERR_UNSUPPORTED;
    CANDY_REQUIRE(pad64(A.cols) == L.w->ld, "internal: norm and contraction of different widths");
    // biases: of both norms or of none, each behind its weights (as every model has them; others take two launches)
    const bool bias = A.pre_b || (A.y.p && A.post_b);
    if (bias && ((A.pre_w && A.pre_b != A.pre_w + L.w->ld) || (A.y.p && A.post_b != A.post_w + L.w->ld))) return CANDY_HIP_ERR_UNSUPPORTED;
    if (L.partial) *L.partial = Partial{(const float *)L.y, 1, 0, (int)L.ldy};
    const int flags = (A.y.p ? MV_Y : 0) | (bias ? MV_BIAS : 0) | (A.rms ? MV_RMS : 0) | (A.pre_w ? MV_PRE : 0);
    const MvNorms np{A.x, A.y.p, A.post_w, A.pre_w, flags, NormPro{A.step, A.x_out, A.mult, A.eps, A.cols}};
    return L.f32 ? launch_mv<float>(dev, L, s, nv, np) : launch_mv<bf16>(dev, L, s, nv, np);
}

// A contraction's tile and how it is split along K.  big false: k_dense_mm, 128 x 64.
struct MmPlan {
    bool big = false;
    int bn = 128, bm = 64, splits = 1;
};
struct BigTile {
    int bn, bm;
    float step;  // us a step of 64 values takes with every CU at work
};
constexpr BigTile BIG_TILES[] = {{256, 256, 1.52f}, {224, 256, 1.38f}, {192, 256, 1.24f}, {160, 256, 1.10f}, {128, 256, 0.92f},
                                 {256, 128, 0.89f}, {192, 128, 0.74f}, {128, 128, 0.57f}};

// The large tiles' loads reach the rows of a tile through 32-bit byte offsets from its first one: all of them within 4 GB.  (Rows
// of 8 million values and more go to k_dense_mm, whose addresses are pointers.)
static bool tile_fits(int tile_rows, int64_t ld) { return tile_rows * ld * 2 <= 0xFFFFFFFFll; }

// The tile and split with the shortest time by the steps a CU has to take one after the other: rounds of workgroups x
// steps x the step's measured time, plus a pass over the copies of a split (written here, read by the launch behind).
// Over twelve shapes of 300 .. 4096 rows this finds the fastest of the tiles measured or one within 3 % of it.
// row_tiles(bm): tiles along the activation rows.  few: of the tiles with 128 or 256 weight rows only; even: whose weight
// rows divide `rows`.
template <class RowTiles>
static MmPlan big_tile(int num_cus, int64_t rows, int64_t K, int64_t ldx, RowTiles row_tiles, int64_t out_bytes, int min_splits, int max_splits,
                       bool few, bool even) {
    MmPlan best;
    best.splits = min_splits;
    float best_us = 1e30f;
    for (const BigTile &t : BIG_TILES) {
        if ((few && t.bn != 128 && t.bn != 256) || (even && rows % t.bn)) continue;
        if (!tile_fits(t.bn, K) || !tile_fits(t.bm, ldx)) continue;
        const int64_t tiles = row_tiles(t.bm) * ((rows + t.bn - 1) / t.bn);
        for (int sp = min_splits; sp <= max_splits; ++sp) {
            const int64_t steps = (K / 64 + sp - 1) / sp;
            if (sp > min_splits && steps < 8) break;
            const float us = (float)((tiles * sp + num_cus - 1) / num_cus * steps) * t.step + (float)(sp - 1) * (float)out_bytes * 4e-7f;
            if (us < best_us) {
                best_us = us;
                best.big = true;
                best.bn = t.bn;
                best.bm = t.bm;
                best.splits = sp;
            }
        }
    }
    return best;
}

// m rows of activations `ldx` apart against `rows` rows of K values
static MmPlan mm_plan(int num_cus, int m, int64_t rows, int64_t K, int64_t ldx, bool partial, bool steady, bool few, int block_rows) {
    MmPlan p;
    if (partial && (m <= 64 || steady)) {
        // two workgroups (of 128 x 64 or 128 x 128) fit a CU; a slice keeps at least 512 values of K
        const int bm = m <= 64 ? 64 : 128;
        const int64_t room = 2 * (int64_t)num_cus / ((m + bm - 1) / bm * ((rows + 127) / 128));
        p.splits = (int)std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(room, 8), K / 512));
    }
    if (m <= 64) return p;
    // block-diagonal: no tile may reach into a second block
    const int64_t blocks = block_rows ? rows / block_rows : 1;
    return big_tile(num_cus, rows / blocks, K, ldx, [&](int bm) { return (m + bm - 1) / bm * blocks; }, (int64_t)m * rows * 4, p.splits,
                    partial && !steady ? 8 : p.splits, few, block_rows != 0);
}

template <int EPI, bool GROUPED, class... Args>
static void launch_big(const MmPlan &p, dim3 g, hipStream_t stream, Args... args) {
#define CANDY_BIG(BN, BM, WN)                                                                                       \
    if (p.bn == BN && p.bm == BM) {                                                                                 \
        hipLaunchKernelGGL((k_dense_big<BN, BM, WN, EPI, GROUPED>), g, dim3(512), 0, stream, args...);              \
        return;                                                                                                     \
    }
    if constexpr (!GROUPED && (EPI == EPI_NONE || EPI == EPI_RELU2)) {
        CANDY_BIG(224, 256, 2)
        CANDY_BIG(192, 256, 2)
        CANDY_BIG(160, 256, 2)
        CANDY_BIG(192, 128, 4)
    }
    if constexpr (!GROUPED) {
        CANDY_BIG(256, 256, 2)
        CANDY_BIG(128, 256, 2)
    }
    CANDY_BIG(256, 128, 4)
    CANDY_BIG(128, 128, 4)
#undef CANDY_BIG
}

// Where the narrow tiles are at most two workgroups per CU: past that the activations they read again cost more than the shorter
// walk saves (us as above, large tiles / narrow ones: 6144 x 4096, 200 rows 38.1 / 46.3, 11008 x 4096, 100 rows 36.3 / 45.4; at 512
// workgroups, 8192 x 2048, 100 rows 22.5 / 20.8).  Where two a CU are nearly all there, a second column of tiles that is not even half full
// is too dear: 8192 x 8192, 65 / 96 / 97 rows 53.5 / 62.0, 55.0 / 59.5, 62.0 / 59.3, 8192 x 4096 30.9 / 31.9, 32.2 / 32.6, 36.0 / 32.7 (but 7168 x 8192,
// 65 rows 53.3 / 53.7, 6144 x 4096 30.6 / 26.3, and short K, 8192 x 1536 16.9 / 16.4).
static bool narrow_pays(int num_cus, int64_t m, int64_t rows, int64_t ld) {
    const int64_t m_tiles = m <= 32 ? 1 : (m + 63) / 64, tiles = m_tiles * (rows / NARROW_BN);
    return tiles <= 2 * (int64_t)num_cus && (4 * tiles <= 7 * (int64_t)num_cus || m <= 64 || ld < 2048 || m % 64 == 0 || m % 64 > 32);
}
static bool narrow_covers(int num_cus, const DenseLaunch &L) {
    if (L.f32 || L.partial || L.block_rows || L.group || !to_act(L.epi)) return false;
    return narrow_pays(num_cus, L.m, L.w->rows_pad, L.w->ld) && tile_fits(NARROW_BN, L.w->ld) && tile_fits(64, L.ldx);
}
static int launch_narrow(candy_hip_device *dev, const DenseLaunch &L) {
    const int K = (int)L.w->ld, rows = (int)L.w->rows_pad, bm = L.m <= 32 ? 32 : 64, m_tiles = (L.m + bm - 1) / bm;
    const dim3 g((unsigned)(m_tiles * (rows / NARROW_BN))), b(256);
    const EpiArgs ea{L.scale, L.cap};
    const bf16 *W = (const bf16 *)L.w->data, *X = (const bf16 *)L.x;
    auto launch = [&](auto kern) {
        hipLaunchKernelGGL(kern, g, b, 0, dev->stream, W, X, (bf16 *)L.y, L.m, rows, K, (int)L.ldx, L.ldy, (int)L.n_store, m_tiles, ea);
    };
    if (L.epi == EPI_RELU2) bm == 32 ? launch(k_dense_narrow<EPI_RELU2, 32>) : launch(k_dense_narrow<EPI_RELU2, 64>);
    else bm == 32 ? launch(k_dense_narrow<EPI_ACT, 32>) : launch(k_dense_narrow<EPI_ACT, 64>);
    CANDY_LAUNCH_CHECK();
    return CANDY_HIP_OK;
}

static int launch_mm(candy_hip_device *dev, const DenseLaunch &L) {
    const int K = (int)L.w->ld;
    const int64_t rows = L.w->rows_pad;
    const MmPlan p = mm_plan(dev->num_cus, L.m, rows, K, L.ldx, L.partial != nullptr, L.steady, L.epi != EPI_NONE && L.epi != EPI_RELU2,
                             L.block_rows);
    if (narrow_covers(dev->num_cus, L)) return launch_narrow(dev, L);
    const int m_tiles = (L.m + p.bm - 1) / p.bm, n_tiles = (int)((rows + p.bn - 1) / p.bn);
    const int64_t tiles = (int64_t)m_tiles * n_tiles;
    CANDY_REQUIRE(tiles <= 0x7FFFFFFF, "matrix too large");
    void *y = L.y;
    int64_t ldy = L.ldy, n_store = L.n_store;
    size_t stride = 0;
    if (p.splits > 1) {
        ldy = n_store = rows;
        stride = (size_t)L.m * ldy;
        if (int rc = splitk_workspace(dev, stride * p.splits * sizeof(float), &y)) return rc;
    }
    const int k_slice = (int)pad64((K + p.splits - 1) / p.splits);
    const int splits = (K + k_slice - 1) / k_slice;
    if (L.partial) {
        L.partial->p = (const float *)y;
        L.partial->copies = splits;
        L.partial->stride = stride;
        L.partial->ld = (int)ldy;
    }
    const dim3 g((unsigned)tiles, (unsigned)splits);
    const EpiArgs ea{L.scale, L.cap};
    const bf16 *W = (const bf16 *)L.w->data, *X = (const bf16 *)L.x;
#define CANDY_MM(EPI)                                                                                                                 \
    do {                                                                                                                              \
        if (p.big)                                                                                                                    \
            launch_big<EPI, false>(p, g, dev->stream, W, X, y, L.m, (int)rows, K, (int)L.ldx, k_slice, ldy, (int)n_store, stride,     \
                                   m_tiles, n_tiles, L.block_rows, ea, GroupedRows{});                                                \
        else                                                                                                                          \
            hipLaunchKernelGGL((k_dense_mm<EPI, false>), g, dim3(256), 0, dev->stream, W, X, y, L.m, (int)rows, K, (int)L.ldx,        \
                               k_slice, ldy, (int)n_store, stride, m_tiles, n_tiles, L.block_rows, ea, GroupedRows{});                \
    } while (0)
    switch (L.epi) {
    case EPI_RELU2: CANDY_MM(EPI_RELU2); break;
    case EPI_CAP: CANDY_MM(EPI_CAP); break;
    case EPI_ACT: CANDY_MM(EPI_ACT); break;
    default: CANDY_MM(EPI_NONE); break;
    }
#undef CANDY_MM
    CANDY_LAUNCH_CHECK();
    return CANDY_HIP_OK;
}

// 64-row tiles (two workgroups per CU) while experts have few rows each, and for short contractions, whose few steps do not pay for
// a large tile's first loads: us of a whole layer, 64 / 128 rows, 64 experts of 256 at width 512, 160 rows each 71.0 / 71.8, 256 85.6 /
// 92.4; of 512 at 1024, 112 rows 96.0 / 107.1, 160 108.6 / 115.9, 192 121.9 / 119.8; of 1408 at 2048, 96 rows 293 / 265.
int grouped_tile_rows(int experts, int64_t slots, int64_t widest) {
    const bool few = slots < 96 * (int64_t)experts, brief = widest <= 768 || (widest <= 1024 && slots < 160 * (int64_t)experts);
    // an activation row's place is a 32-bit offset in the large tiles' loads, from the first of all rows, and so is a weight row's
    return few || brief || slots * widest * 2 > 0xFFFFFFFFll || !tile_fits(256, widest) ? 64 : 128;
}

// Weight rows of the 128-row tiles: 256 for the longer share of a launch that reads every expert's weights either way, 128 where all
// of these are on the chip at once (by the rows an expert has on average, and a few more).  us of a whole layer, 128 / 256: 64 experts
// of 1408 at width 2048, 96 rows each 273 / 265, 192 396 / 362, 512 816 / 732; 16 of 2048 at 4096, 192 283 / 267; 8 of 4096 at
// 4096, 96 rows (one round) 211 / 239, 128 rows (two) 264 / 245; 4 of 2048 at 1024, 256 rows 68 / 86; 8 of 4096 at 1024, 96 rows 82 / 107.
static int grouped_weight_rows(int num_cus, int experts, int64_t slots, int expert_rows) {
    const int64_t row_tiles = (slots / experts + 16 + 127) / 128 * experts;
    return expert_rows <= 128 || row_tiles * ((expert_rows + 127) / 128) <= num_cus ? 128 : 256;
}

// Rows dealt to experts: the grid has room for max_tiles row tiles, workgroups past the list's end leave at once.
static int launch_mm_grouped(candy_hip_device *dev, const DenseLaunch &L) {
    const GroupedRows &gr = *L.group;
    const int K = (int)L.w->ld;
    MmPlan p;
    if (gr.tile_rows > 64) {
        p.big = true;
        p.bm = 128;
        p.bn = grouped_weight_rows(dev->num_cus, (int)(L.w->rows / gr.expert_rows), L.m, gr.expert_rows);
    }
    const int n_tiles = (gr.expert_rows + p.bn - 1) / p.bn;
    const int64_t tiles = (int64_t)gr.max_tiles * n_tiles;
    CANDY_REQUIRE(tiles <= 0x7FFFFFFF, "matrix too large");
    const dim3 g((unsigned)tiles);
    const EpiArgs ea{L.scale, L.cap};
    const bf16 *W = (const bf16 *)L.w->data, *X = (const bf16 *)L.x;
#define CANDY_MMG(EPI)                                                                                                                    \
    do {                                                                                                                                  \
        if (p.big)                                                                                                                        \
            launch_big<EPI, true>(p, g, dev->stream, W, X, L.y, L.m, gr.expert_rows, K, (int)L.ldx, K, L.ldy, (int)L.n_store, (size_t)0, \
                                  0, n_tiles, 0, ea, gr);                                                                                 \
        else                                                                                                                              \
            hipLaunchKernelGGL((k_dense_mm<EPI, true>), g, dim3(256), 0, dev->stream, W, X, L.y, L.m, gr.expert_rows, K, (int)L.ldx, K,   \
                               L.ldy, (int)L.n_store, (size_t)0, 0, n_tiles, 0, ea, gr);                                                  \
    } while (0)
    if (L.epi == EPI_RELU2) CANDY_MMG(EPI_RELU2);
    else CANDY_MMG(EPI_NONE);
#undef CANDY_MMG
    CANDY_LAUNCH_CHECK();
    return CANDY_HIP_OK;
}

int launch_dense(candy_hip_device *dev, const DenseLaunch &L) {
    const candy_hip_dense *w = L.w;
    CANDY_REQUIRE(L.m > 0 && w->rows_pad <= 0x7FFFFFFF && w->ld <= 0x7FFFFFFF && L.ldx >= w->ld && L.ldx <= 0x7FFFFFFF,
                  "internal: dense contraction of a shape the kernels do not take");
    CANDY_REQUIRE(L.n_store <= w->rows_pad && L.ldy >= L.n_store, "internal: dense output row too short");
    const int64_t out_rows = L.group ? L.group->expert_rows : w->rows_pad;
    CANDY_REQUIRE(!to_act(L.epi) || (L.n_store == out_rows && (L.ldy & 63) == 0), "internal: activation rows must be padded");
    CANDY_REQUIRE(L.block_rows == 0 || (!L.partial && L.block_rows % 128 == 0 && w->rows_pad % L.block_rows == 0 &&
                                        L.ldx >= w->rows_pad / L.block_rows * w->ld), "internal: block-diagonal contraction");
    if (L.group) {
        CANDY_REQUIRE((L.epi == EPI_NONE || L.epi == EPI_RELU2) && !L.partial && !L.block_rows && L.group->expert_rows % 64 == 0 &&
                          w->rows % L.group->expert_rows == 0 && L.group->max_tiles <= 65535,
                      "internal: grouped contraction");
        CANDY_REQUIRE(L.group->tile_rows == 64 || (!L.f32 && L.group->tile_rows == 128), "internal: row tiles");
        if (!L.f32) return launch_mm_grouped(dev, L);
    }
    if (L.partial) {
        L.partial->p = (const float *)L.y;
        L.partial->copies = 1;
        L.partial->stride = 0;
        L.partial->ld = (int)L.ldy;
    }
    if (L.m == 1 && !L.group && !L.block_rows) {
        const MvShape s = mv_shape(dev, L.n_store);
        return L.f32 ? launch_mv<float>(dev, L, s) : launch_mv<bf16>(dev, L, s);
    }
    if (!L.f32) return launch_mm(dev, L);
    const dim3 g((unsigned)(out_rows / 64), (unsigned)(L.group ? L.group->max_tiles : (L.m + 63) / 64)), b(256);
    CANDY_REQUIRE((L.m + 63) / 64 <= 65535, "prompt too long for one pass");
    const EpiArgs ea{L.scale, L.cap};
    const bf16 *W = (const bf16 *)w->data;
    const float *X = (const float *)L.x;
#define CANDY_MM32(EPI)                                                                                                 \
    do {                                                                                                                \
        if (L.group)                                                                                                    \
            hipLaunchKernelGGL((k_dense_mm_f32<EPI, true>), g, b, 0, dev->stream, W, X, (float *)L.y, L.m, (int)w->ld,  \
                               (int)L.ldx, L.ldy, (int)L.n_store, 0, ea, *L.group);                                     \
        else                                                                                                            \
            hipLaunchKernelGGL((k_dense_mm_f32<EPI, false>), g, b, 0, dev->stream, W, X, (float *)L.y, L.m, (int)w->ld, \
                               (int)L.ldx, L.ldy, (int)L.n_store, L.block_rows, ea, GroupedRows{});                     \
    } while (0)
    switch (L.epi) {
    case EPI_RELU2: CANDY_MM32(EPI_RELU2); break;
    case EPI_CAP: CANDY_MM32(EPI_CAP); break;
    default: CANDY_MM32(EPI_NONE); break;  // ACT: f32 is the activation format
    }
#undef CANDY_MM32
    CANDY_LAUNCH_CHECK();
    return CANDY_HIP_OK;
}

// rows ids[i] of a bfloat16 table, widened and scaled; an id outside the table raises the handle's fault word and gives zeros
__global__ __launch_bounds__(256) void k_dense_gather(const bf16 *__restrict__ W, int64_t rows, int64_t ld,
                                                      const int64_t *__restrict__ ids, float *__restrict__ out, int64_t ldo,
                                                      float scale, int *fault) {
    const int64_t id = ids[blockIdx.y];
    const int64_t c = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
    if (c >= ld) return;
    float f[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (id >= 0 && id < rows) widen8(*(const u32x4v *)(W + id * ld + c), f);
    else if (c == 0) *fault = 1;
    float *o = out + (int64_t)blockIdx.y * ldo + c;
    *(f32x4 *)o = f32x4{f[0], f[1], f[2], f[3]} * scale;
    *(f32x4 *)(o + 4) = f32x4{f[4], f[5], f[6], f[7]} * scale;
}

int launch_dense_gather(candy_hip_device *dev, const candy_hip_dense *w, const int64_t *ids, int64_t n, float *out, int64_t ldo,
                        float scale) {
    for (int64_t i0 = 0; i0 < n; i0 += 65535) {
        const int64_t part = std::min<int64_t>(n - i0, 65535);
        hipLaunchKernelGGL(k_dense_gather, dim3((unsigned)((w->ld / 8 + 255) / 256), (unsigned)part), dim3(256), 0, dev->stream,
                           (const bf16 *)w->data, w->rows, w->ld, ids + i0, out + i0 * ldo, ldo, scale, dev->fault);
        CANDY_LAUNCH_CHECK();
    }
    return CANDY_HIP_OK;
}

// f32 rows -> activation rows of ld values, zero past cols
template <class AT>
__global__ __launch_bounds__(256) void k_to_act(const float *__restrict__ src, AT *__restrict__ dst, int64_t rows, int64_t cols, int64_t ld) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= rows * ld) return;
    const int64_t r = i / ld, c = i % ld;
    dst[i] = c < cols ? (AT)src[r * cols + c] : (AT)0.0f;
}
// activation rows -> dense f32
template <class AT>
__global__ __launch_bounds__(256) void k_from_act(const AT *__restrict__ src, float *__restrict__ dst, int64_t rows, int64_t cols, int64_t ld) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= rows * cols) return;
    dst[i] = (float)src[i / cols * ld + i % cols];
}

int launch_to_act(candy_hip_device *dev, bool f32, const float *src, void *dst, int64_t rows, int64_t cols, int64_t ld) {
    const int64_t grid = (rows * ld + 255) / 256;
    CANDY_REQUIRE(grid <= 0x7FFFFFFF, "matrix too large");
    if (f32) hipLaunchKernelGGL((k_to_act<float>), dim3((unsigned)grid), dim3(256), 0, dev->stream, src, (float *)dst, rows, cols, ld);
    else hipLaunchKernelGGL((k_to_act<bf16>), dim3((unsigned)grid), dim3(256), 0, dev->stream, src, (bf16 *)dst, rows, cols, ld);
    CANDY_LAUNCH_CHECK();
    return CANDY_HIP_OK;
}
int launch_from_act(candy_hip_device *dev, bool f32, const void *src, float *dst, int64_t rows, int64_t cols, int64_t ld) {
    const int64_t grid = (rows * cols + 255) / 256;
    CANDY_REQUIRE(grid <= 0x7FFFFFFF, "matrix too large");
    if (f32) hipLaunchKernelGGL((k_from_act<float>), dim3((unsigned)grid), dim3(256), 0, dev->stream, (const float *)src, dst, rows, cols, ld);
    else hipLaunchKernelGGL((k_from_act<bf16>), dim3((unsigned)grid), dim3(256), 0, dev->stream, (const bf16 *)src, dst, rows, cols, ld);
    CANDY_LAUNCH_CHECK();
    return CANDY_HIP_OK;
}

}  // namespace candy

using namespace candy;

extern "C" {

int candy_hip_dense_upload(candy_hip_device *dev, int64_t rows, int64_t cols, const uint16_t *host_bf16, candy_hip_dense **out) {
    CANDY_REQUIRE(out, "out is nil");
    *out = nullptr;
    CANDY_REQUIRE(dev, "device handle is nil");
    CANDY_REQUIRE(rows > 0 && cols > 0 && rows <= 0x7FFFFF00 && cols <= 0x7FFFFF00, "invalid matrix dimensions %lld x %lld",
                  (long long)rows, (long long)cols);
    CANDY_REQUIRE(host_bf16, "host weight is nil");
    if (int rc = use_device(dev)) return rc;
    const int64_t rp = pad64(rows), ld = pad64(cols);
    void *d = nullptr;
    const size_t bytes = (size_t)rp * ld * 2;
    if (int rc = candy_hip_alloc(dev, bytes, &d)) return rc;
    int rc = CANDY_HIP_OK;
    if (rp != rows || ld != cols) rc = candy_hip_zero(dev, d, bytes);
    if (!rc) {
        hipError_t e = hipMemcpy2DAsync(d, (size_t)ld * 2, host_bf16, (size_t)cols * 2, (size_t)cols * 2, (size_t)rows,
                                        hipMemcpyHostToDevice, dev->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(dev->stream);
        if (e != hipSuccess) rc = fail(CANDY_HIP_ERR_HIP, "weight upload failed: %s", hipGetErrorString(e));
    }
    if (rc) {
        (void)candy_hip_free(dev, d);
        return rc;
    }
    candy_hip_dense *w = new candy_hip_dense();
    w->dev = dev; w->rows = rows; w->cols = cols; w->rows_pad = rp; w->ld = ld; w->data = d;
    *out = w;
    return CANDY_HIP_OK;
}

int candy_hip_dense_free(candy_hip_dense *w) {
    if (!w) return CANDY_HIP_OK;
    const int rc = candy_hip_free(w->dev, w->data);
    delete w;
    return rc;
}

int candy_hip_dense_info(const candy_hip_dense *w, int64_t *rows, int64_t *cols, size_t *nbytes) {
    CANDY_REQUIRE(w, "weight is nil");
    if (rows) *rows = w->rows;
    if (cols) *cols = w->cols;
    if (nbytes) *nbytes = (size_t)w->rows_pad * w->ld * 2;
    return CANDY_HIP_OK;
}

int candy_hip_dense_matmul(candy_hip_device *dev, const candy_hip_dense *w, const float *dev_x, int64_t m, int act, int epilogue,
                           float scale, float cap, float *dev_y) {
    CANDY_REQUIRE(w, "rhs weight is nil");
    CANDY_REQUIRE(dev && w->dev == dev, "rhs storage must live on the same HIP device");
    CANDY_REQUIRE(m >= 0 && m <= 1 << 20, "invalid matrix dimensions");
    CANDY_REQUIRE(act == CANDY_HIP_ACT_BF16 || act == CANDY_HIP_ACT_F32, "unknown activation format %d", act);
    CANDY_REQUIRE(epilogue >= EPI_NONE && epilogue <= EPI_ACT, "unknown epilogue %d", epilogue);
    if (m == 0) return CANDY_HIP_OK;
    CANDY_REQUIRE(dev_x && dev_y, "nil pointer");
    if (int rc = use_device(dev)) return rc;
    const bool f32 = act == CANDY_HIP_ACT_F32;
    const size_t x_bytes = (size_t)m * w->ld * 4, y_bytes = (size_t)m * w->rows_pad * 4;
    void *ws = nullptr;
    if (int rc = workspace(dev, x_bytes + y_bytes, &ws)) return rc;
    if (int rc = launch_to_act(dev, f32, dev_x, ws, m, w->cols, w->ld)) return rc;
    DenseLaunch L;
    L.w = w; L.x = ws; L.ldx = w->ld; L.f32 = f32; L.m = (int)m; L.epi = epilogue; L.scale = scale; L.cap = cap;
    if (!to_act(epilogue)) {
        L.y = dev_y; L.ldy = L.n_store = w->rows;
        return launch_dense(dev, L);
    }
    L.y = (uint8_t *)ws + x_bytes; L.ldy = L.n_store = w->rows_pad;
    if (int rc = launch_dense(dev, L)) return rc;
    return launch_from_act(dev, f32, L.y, dev_y, m, w->rows, w->rows_pad);
}

// The rules that choose a tile, for their tests (no device needed): plan[0..3] = large tiles, weight rows, activation rows, splits.
void candy_test_dense_plan(int num_cus, int m, int64_t rows, int64_t ld, int64_t ldx, int partial, int steady, int few, int block_rows, int *plan) {
    const candy::MmPlan p = candy::mm_plan(num_cus, m, rows, ld, ldx, partial != 0, steady != 0, few != 0, block_rows);
    plan[0] = p.big; plan[1] = p.bn; plan[2] = p.bm; plan[3] = p.splits;
}
int candy_test_narrow_pays(int num_cus, int64_t m, int64_t rows, int64_t ld) { return candy::narrow_pays(num_cus, m, rows, ld); }
int candy_test_grouped_tile_rows(int experts, int64_t slots, int64_t widest) { return candy::grouped_tile_rows(experts, slots, widest); }
int candy_test_grouped_weight_rows(int num_cus, int experts, int64_t slots, int expert_rows) {
    return candy::grouped_weight_rows(num_cus, experts, slots, expert_rows);
}

int candy_hip_dense_sweep(candy_hip_device *dev, const candy_hip_dense *const *ws, int n_ws, const float *dev_x, int64_t m,
                          int epilogue, int iters, float *elapsed_ms) {
    CANDY_REQUIRE(dev && ws && n_ws > 0 && dev_x && elapsed_ms && iters > 0 && m > 0 && m <= 1 << 20, "nil argument");
    CANDY_REQUIRE(epilogue >= EPI_NONE && epilogue <= EPI_ACT, "unknown epilogue %d", epilogue);
    for (int i = 0; i < n_ws; ++i)
        CANDY_REQUIRE(ws[i] && ws[i]->dev == dev && ws[i]->rows == ws[0]->rows && ws[i]->cols == ws[0]->cols,
                      "weights of one sweep share a device and a shape");
    if (int rc = use_device(dev)) return rc;
    const candy_hip_dense *w = ws[0];
    const size_t x_bytes = (size_t)m * w->ld * 2;
    void *buf = nullptr;
    if (int rc = workspace(dev, x_bytes + (size_t)m * w->rows_pad * 4, &buf)) return rc;
    if (int rc = launch_to_act(dev, false, dev_x, buf, m, w->cols, w->ld)) return rc;
    DenseLaunch L;
    Partial part;
    L.x = buf; L.ldx = w->ld; L.m = (int)m; L.epi = epilogue; L.scale = 1.0f; L.cap = 30.0f;
    L.y = (uint8_t *)buf + x_bytes; L.ldy = L.n_store = w->rows_pad;
    if (epilogue == EPI_NONE) L.partial = &part;
    CANDY_HIP_TRY(hipEventRecord(dev->ev_start, dev->stream));
    for (int i = 0; i < iters; ++i) {
        L.w = ws[i % n_ws];
        if (int rc = launch_dense(dev, L)) return rc;
    }
    CANDY_HIP_TRY(hipEventRecord(dev->ev_stop, dev->stream));
    CANDY_HIP_TRY(hipEventSynchronize(dev->ev_stop));
    CANDY_HIP_TRY(hipEventElapsedTime(elapsed_ms, dev->ev_start, dev->ev_stop));
    return CANDY_HIP_OK;
}

}  // extern "C"
