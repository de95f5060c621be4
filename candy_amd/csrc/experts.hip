// Routed experts with squared-ReLU feed-forwards (equations and layouts: include/candy_hip.h).
//   prompts: k_route        router scores of 16 tokens in f32 on the matrix cores (activations as the sum of three bfloat16
//                           parts, which is exact), softmax, the choice and its weights
//            k_deal         slots (token, choice) sorted by expert, and the list of row tiles
//            the experts' contractions over their rows, and the shared expert's (dense.hip); k_norm_chain sums the slots
//   decode:  the router as a contraction of one row (dense.hip)
//            k_expert_up    choice in the prologue; the chosen experts' and the shared one's rows, squared ReLU, weighted
//            k_expert_down  one contraction over the concatenation of their inner activations
// (No counterpart in the reference, which has no routed layer.)
#include <algorithm>

#include "dense.h"

namespace candy {

// What the choice orders scores by: every value has its place, so that the choice names `top` different experts even where
// a model's numbers have gone wrong.
__device__ __forceinline__ float ordered(float z) { return z == z ? z : -INFINITY; }

// One wavefront, lane e holding score e of a token's E <= 64 (ordered()): lane k leaves with the k-th choice and its weight.
struct Choice64 {
    float v, best, mine;   // the scores left, the largest of all, lane k: the k-th choice's
    int id;                // lane k: the k-th choice
    __device__ __forceinline__ void pick(float score, int E, int top) {
        const int lane = threadIdx.x & 63;
        uint64_t left = E == 64 ? ~0ull : (1ull << E) - 1;
        v = lane < E ? score : -INFINITY;
        best = wave_max(v);
        mine = -INFINITY;
        id = 0;
        float w = v, b = best;
        for (int k = 0; k < top; ++k) {
            if (k) b = wave_max(w);
            const int e = __ffsll((unsigned long long)(__ballot(w == b) & left)) - 1;   // not empty: `left` has top - k members
            left &= ~(1ull << e);
            if (lane == k) { id = e; mine = b; }
            if (lane == e) w = -INFINITY;
        }
    }
    // two tokens' choices at once
    static __device__ __forceinline__ void pick2(Choice64 (&c)[2], float s0, float s1, int E, int top) {
        const int lane = threadIdx.x & 63;
        const uint64_t all = E == 64 ? ~0ull : (1ull << E) - 1;
        uint64_t left[2] = {all, all};
        float w[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            c[t].v = w[t] = lane < E ? (t ? s1 : s0) : -INFINITY;
            c[t].mine = -INFINITY;
            c[t].id = 0;
        }
        for (int k = 0; k < top; ++k) {
            float b[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) b[t] = wave_max(w[t]);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                if (k == 0) c[t].best = b[t];
                const int e = __ffsll((unsigned long long)(__ballot(w[t] == b[t]) & left[t])) - 1;
                left[t] &= ~(1ull << e);
                if (lane == k) { c[t].id = e; c[t].mine = b[t]; }
                if (lane == e) w[t] = -INFINITY;
            }
        }
    }
    __device__ __forceinline__ float weight(int E, int top) const {
        const int lane = threadIdx.x & 63;
        const float mx = fmaxf(best, LOW), sum = wave_sum(lane < E ? expf(v - mx) : 0.0f);
        const float s = lane < top ? expf(mine - mx) / sum : 0.0f;
        return s / (wave_sum(s) + 1e-20f);
    }
};
__device__ __forceinline__ void choose64(float v, int E, int top, int &id, float &weight) {
    Choice64 c;
    c.pick(v, E, top);
    id = c.id;
    weight = c.weight(E, top);
}

// The same for any number of scores z[0 .. E) in LDS; choices and weights in order of their scores.
__device__ __forceinline__ void choose(const float *z, int E, int top, int *ids, float *weights) {
    const int lane = threadIdx.x & 63;
    if (E <= 64) {
        int id;
        float w;
        choose64(lane < E ? z[lane] : 0.0f, E, top, id, w);
        if (lane < top) {
            ids[lane] = id;
            weights[lane] = w;
        }
        return;
    }
    float mx = LOW;
    for (int e = lane; e < E; e += 64) mx = fmaxf(mx, z[e]);
    mx = wave_max(mx);
    float sum = 0.0f;
    for (int e = lane; e < E; e += 64) sum += expf(z[e] - mx);
    sum = wave_sum(sum);
    float chosen = 0.0f;
    for (int e0 = 0; e0 < E; e0 += 64) {
        const int e = e0 + lane;
        const float mine = e < E ? z[e] : 0.0f;
        int rank = 0;
#pragma unroll 8
        for (int f = 0; f < E; ++f) rank += z[f] > mine || (z[f] == mine && f < e);
        if (e < E && rank < top) {
            const float s = expf(mine - mx) / sum;
            ids[rank] = e;
            weights[rank] = s;
            chosen += s;
        }
    }
    chosen = wave_sum(chosen) + 1e-20f;
    __builtin_amdgcn_wave_barrier();
    for (int k = lane; k < top; k += 64) weights[k] /= chosen;
}

// ------------------------------------------------------------------ prompts
constexpr int ROUTE_T = 16, ROUTE_W = 8, ROUTE_K = 32 * ROUTE_W;   // tokens and wavefronts of a workgroup, values of K a stage
constexpr int ROUTE_STAGE = 64 * ROUTE_K * 2 + ROUTE_T * ROUTE_K * 4;   // bytes: router rows, token rows
// grid ceil(n / 16), 8 wavefronts that share K, a step of 32 values of a stage each; 64 experts per round.  What bounds it: latencies
// and the way of 384 KB into one CU, whatever the number of tokens.  Operands loaded as they are needed were 16 rows of 64 bytes, 4
// KB apart, to a load, and another wavefront's 64 bytes of the same lines came again; by direct loads of whole lines, three stages in
// LDS: us of a launch, 64 experts at width 2048, 128 / 2048 tokens 18.2 / 19.2 -> 11.3 / 13.0 (of which the choices, two tokens a
// wavefront side by side, 1.7).
template <int STAGES>
__global__ __launch_bounds__(64 * ROUTE_W) void k_route(const float *__restrict__ x, int64_t ldx, const bf16 *__restrict__ W, int ld, int E,
                                                        int top, int n, int *__restrict__ ids, float *__restrict__ weights) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass knows no buffer descriptors
    // [STAGES] of rows of 16-byte pieces, piece p of row r in slot p ^ (r & 15); once they are read, [8][64][17] sums of wavefronts.
    // Then [16][E] scores
    extern __shared__ __align__(16) uint8_t lds[];
    float *const red = (float *)lds, *const z = (float *)(lds + STAGES * ROUTE_STAGE);
    const int Ep = E | 1;                              // odd pitch
    int *const s_ids = (int *)lds;                     // once the scores stand: [16][top], [16][top]
    float *const s_w = red + ROUTE_T * top;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
    const int t0 = blockIdx.x * ROUTE_T, steps = ld >> 5, stages = (ld + ROUTE_K - 1) / ROUTE_K, rows = min(ROUTE_T, n - t0);
    const __amdgpu_buffer_rsrc_t rx =
                                     __builtin_amdgcn_make_buffer_rsrc((void *)(x + (size_t)t0 * ldx), 0, (int)(rows * ldx * 4), 0x00027000),
                                 rw = __builtin_amdgcn_make_buffer_rsrc((void *)W, 0, ((E + 15) & ~15) * ld * 2, 0x00027000);
    constexpr int LW = 64 / 2 / ROUTE_W, LX = ROUTE_T / ROUTE_W, LOADS = LW + LX;   // a wavefront's: two router rows, a token's row each
    for (int e0 = 0; e0 < E; e0 += 64) {
        uint32_t w_off[LW], x_off[LX];
#pragma unroll
        for (int i = 0; i < LW; ++i) {
            const int r = (wave * LW + i) * 2 + (lane >> 5);
            w_off[i] = (uint32_t)(e0 + r) * (uint32_t)ld * 2 + ((lane & 31) ^ (r & 15)) * 16;
        }
#pragma unroll
        for (int i = 0; i < LX; ++i) x_off[i] = (uint32_t)(wave * LX + i) * (uint32_t)ldx * 4 + (lane ^ (wave * LX + i)) * 16;
        auto request = [&](int k, int slot) __attribute__((always_inline)) {
            auto *to = (__attribute__((address_space(3))) uint8_t *)(lds + slot * ROUTE_STAGE);
#pragma unroll
            for (int i = 0; i < LW; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, to + (wave * LW + i) * 1024, 16, w_off[i], k * ROUTE_K * 2, 0, 0);
#pragma unroll
            for (int i = 0; i < LX; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, to + 64 * ROUTE_K * 2 + (wave * LX + i) * 1024, 16, x_off[i], k * ROUTE_K * 4,
                                                         0, 0);
        };
        f32x4 acc[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < STAGES - 1; ++k)
            if (k < stages) request(k, k);
        for (int k = 0, slot = 0; k < stages; ++k, slot = slot + 1 == STAGES ? 0 : slot + 1) {
            // this stage is there, those behind it may be on their way; the one in front of it is read
            asm volatile("" ::: "memory");
            if (STAGES == 3 && k + 1 < stages) __builtin_amdgcn_s_waitcnt(0x0070 | LOADS);
            else __builtin_amdgcn_s_waitcnt(0x0070);
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if (k + STAGES - 1 < stages) request(k + STAGES - 1, slot == 0 ? STAGES - 1 : slot - 1);
            if (k * ROUTE_W + wave >= steps) continue;
            const uint8_t *at = lds + slot * ROUTE_STAGE;
            bf16x8 w[4], part[3];
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = *(const bf16x8 *)(at + (i * 16 + r16) * (ROUTE_K * 2) + ((wave * 4 + g) ^ r16) * 16);
            f32x4 xv[2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
                xv[i] = *(const f32x4 *)(at + 64 * ROUTE_K * 2 + r16 * (ROUTE_K * 4) + ((wave * 8 + g * 2 + i) ^ r16) * 16);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float f = xv[j >> 2][j & 3];
                part[0][j] = (bf16)f;
                const float r1 = f - (float)part[0][j];
                part[1][j] = (bf16)r1;
                part[2][j] = (bf16)(r1 - (float)part[1][j]);
            }
#pragma unroll
            for (int p = 2; p >= 0; --p)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i], part[p], acc[i], 0, 0, 0);
        }
        __syncthreads();
        // lane: token r16, experts e0 + 16 i + 4 g + j
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) red[(wave * 64 + i * 16 + 4 * g + j) * 17 + r16] = acc[i][j];
        __syncthreads();
        for (int i = tid; i < 64 * ROUTE_T; i += 64 * ROUTE_W) {
            const int t = i & 15, e = i >> 4;
            if (e0 + e >= E) continue;
            float v[ROUTE_W], sum = 0.0f;
#pragma unroll
            for (int k = 0; k < ROUTE_W; ++k) v[k] = red[(k * 64 + e) * 17 + t];
#pragma unroll
            for (int k = 0; k < ROUTE_W / 2; ++k) sum += v[k + ROUTE_W / 2] + v[k];
            z[t * Ep + e0 + e] = ordered(sum);
        }
        __syncthreads();
    }
    static_assert(ROUTE_T == 2 * ROUTE_W, "two tokens a wavefront");
    if (E <= 64) {   // side by side: a choice is a chain of reductions
        Choice64 c[2];
        Choice64::pick2(c, lane < E ? z[wave * Ep + lane] : 0.0f, lane < E ? z[(wave + ROUTE_W) * Ep + lane] : 0.0f, E, top);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const float weight = c[k].weight(E, top);
            if (lane < top) {
                s_ids[(wave + k * ROUTE_W) * top + lane] = c[k].id;
                s_w[(wave + k * ROUTE_W) * top + lane] = weight;
            }
        }
    } else {
        for (int t = wave; t < ROUTE_T; t += ROUTE_W) choose(z + t * Ep, E, top, s_ids + t * top, s_w + t * top);
    }
    __syncthreads();
    for (int i = tid; i < ROUTE_T * top; i += 64 * ROUTE_W)
        if (t0 + i / top < n) {
            ids[(size_t)t0 * top + i] = s_ids[i];
            weights[(size_t)t0 * top + i] = s_w[i];
        }
#endif
}

constexpr int MAX_EXPERTS = 1024;
// One workgroup of 1024: perm[0 .. count) = the slots, expert by expert; tiles of at most `rows` of one expert each.
__global__ __launch_bounds__(1024) void k_deal(const int *__restrict__ ids, int count, int E, int rows, int *__restrict__ perm,
                                               GroupTile *__restrict__ tiles, int *__restrict__ n_tiles) {
    __shared__ int members[MAX_EXPERTS], totals[2][MAX_EXPERTS / 64];
    const int tid = threadIdx.x;
    members[tid] = 0;
    __syncthreads();
    // a thread's slots stay in registers between the count and the deal, up to 16 of them
    constexpr int AHEAD = 16;
    int e[AHEAD];
    auto request = [&](int i0) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < AHEAD; ++k)
            if (i0 + 1024 * k < count) e[k] = ids[i0 + 1024 * k];
    };
    for (int i0 = tid; i0 < count; i0 += 1024 * AHEAD) {
        request(i0);
#pragma unroll
        for (int k = 0; k < AHEAD; ++k)
            if (i0 + 1024 * k < count) atomicAdd(&members[e[k]], 1);
    }
    __syncthreads();
    const int mine = members[tid], my_tiles = (mine + rows - 1) / rows;
    // inclusive sums of a wavefront's 64 experts, then of the wavefronts in front
    const int lane = tid & 63, wave = tid >> 6;
    int end = mine, tile_end = my_tiles;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int m = __shfl_up(end, d, 64), t = __shfl_up(tile_end, d, 64);
        if (lane >= d) { end += m; tile_end += t; }
    }
    if (lane == 63) { totals[0][wave] = end; totals[1][wave] = tile_end; }
    __syncthreads();
    for (int w = 0; w < wave; ++w) { end += totals[0][w]; tile_end += totals[1][w]; }
    const int begin = end - mine, tile0 = tile_end - my_tiles;
    for (int k = 0; k < my_tiles; ++k) tiles[tile0 + k] = GroupTile{tid, begin + k * rows, min(rows, mine - k * rows), (uint16_t)tile0, (uint16_t)my_tiles};
    if (tid == E - 1) *n_tiles = tile_end;
    members[tid] = begin;
    __syncthreads();
    for (int i0 = tid; i0 < count; i0 += 1024 * AHEAD) {
        if (count > 1024 * AHEAD) request(i0);
#pragma unroll
        for (int k = 0; k < AHEAD; ++k)
            if (i0 + 1024 * k < count) perm[atomicAdd(&members[e[k]], 1)] = i0 + 1024 * k;
    }
}

// ------------------------------------------------------------------ decode
struct RowArgs {
    const bf16 *W, *shared;   // up: [E * rows_e][ld], [rows_s][ld]; down: [E * d_p][rows_e], [d_p][rows_s]
    int E, top, rows_e, rows_s, ld;   // rows_e / rows_s: padded inner widths of an expert and of the shared one
};

// 16-byte requests per row and step; two steps are in flight.  (With one of half the length, requested when the one before it was
// consumed, the down projections were six round trips one after the other.)  us of a decode step of the fine / coarse Gulisun decoder with
// four layers, before -> now: 288 / 396 -> 281 / 388.
template <int R> constexpr int exp_unroll() { return 8 / R; }

// k_expert_up: the row that a place of the grid stands for (those behind the last row: the last row), and whether the wavefront
// whose places start at row0 has rows of chosen experts, so that it needs the choice.  Where there is no shared expert the last row is a
// chosen expert's, and wavefronts wholly behind it read its weights as well.
__host__ __device__ __forceinline__ int up_row(int place, int total) { return place < total ? place : total - 1; }
__host__ __device__ __forceinline__ bool up_chooses(int row0, int total, int routed) { return up_row(row0, total) < routed; }

// Rows of the concatenated up matrices, R per wavefront.  FEW: at most 64 experts, every wavefront that has rows of chosen experts
// makes the choice for itself; scores and activations are requested in front of everything, the weights as soon as the choice
// stands, and its shares are worked out while they come.  LDS: x and eight zeros; else behind x the scores, where the zeros go once
// the choice stands, and the choice.
template <class AT, int R, bool FEW>
__global__ __launch_bounds__(1024) void k_expert_up(const float *__restrict__ x, const float *__restrict__ logits, AT *__restrict__ act,
                                                    int *__restrict__ sel, const RowArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass knows no buffer descriptors
    constexpr int U = exp_unroll<R>(), STEP = U * 512;
    extern __shared__ __align__(16) uint8_t lds[];
    AT *xs = (AT *)lds;
    AT *nothing = xs + a.ld;   // eight zeros
    float *z = (float *)nothing, *gate = z + a.E;
    int *ids = (int *)(gate + a.top);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), threads = blockDim.x;
    const int routed = a.top * a.rows_e, total = routed + a.rows_s, row0 = (blockIdx.x * (threads >> 6) + wave) * R;
    typedef AT at4 __attribute__((ext_vector_type(4)));
    constexpr int FIRST = 2;
    f32x4 held[FIRST];
    const float score = FEW ? logits[min(lane, a.E - 1)] : 0.0f;
#pragma unroll
    for (int i = 0; i < FIRST; ++i) held[i] = *(const f32x4 *)(x + min((tid + threads * i) * 4, a.ld - 4));
    auto stage = [&]() __attribute__((always_inline)) {
        if (tid < 8) nothing[tid] = (AT)0.0f;
#pragma unroll
        for (int i = 0; i < FIRST; ++i)
            if ((tid + threads * i) * 4 < a.ld) *(at4 *)&xs[(tid + threads * i) * 4] = __builtin_convertvector(held[i], at4);
        for (int i = (tid + threads * FIRST) * 4; i < a.ld; i += threads * 4)
            *(at4 *)&xs[i] = __builtin_convertvector(*(const f32x4 *)(x + i), at4);
    };
    Choice64 choice;
    const bool chooses = FEW && up_chooses(row0, total, routed);
    if (FEW) {
        if (chooses) {
            choice.pick(ordered(score), a.E, a.top);
            if (blockIdx.x == 0 && wave == 0 && lane < a.top) sel[lane] = choice.id;
        }
    } else {
        for (int e = tid; e < a.E; e += threads) z[e] = ordered(logits[e]);
        __syncthreads();
        if (wave == 0) {
            choose(z, a.E, a.top, ids, gate);
            if (blockIdx.x == 0)
                for (int k = lane; k < a.top; k += 64) sel[k] = ids[k];
        }
        __syncthreads();
    }
    // a row through a descriptor of its own: what lies past it comes as zeros
    constexpr int NT = 2;  // nontemporal
    __amdgpu_buffer_rsrc_t w[R];
    float scale[R];
    int of[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int row = up_row(row0 + r, total), k = row / a.rows_e;
        of[r] = k;
        const bf16 *p = a.shared + (size_t)max(row - routed, 0) * a.ld;
        if (k < a.top) {
            const int id = FEW ? __builtin_amdgcn_readlane(choice.id, k) : __builtin_amdgcn_readfirstlane(ids[k]);
            p = a.W + ((size_t)id * a.rows_e + (row - k * a.rows_e)) * a.ld;
        }
        w[r] = __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, 2 * a.ld, 0x00027000);
    }
    u32x4v va[R][U], vb[R][U];
    auto fetch = [&](u32x4v (&v)[R][U], int k0) __attribute__((always_inline)) {
        const int at = 2 * k0 + lane * 16;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int r = 0; r < R; ++r)
                v[r][u] = __builtin_bit_cast(u32x4v, __builtin_amdgcn_raw_buffer_load_b128(w[r], at + u * 1024, 0, NT));
    };
    fetch(va, 0);
    fetch(vb, STEP);
    __builtin_amdgcn_sched_barrier(0);
    float share = 0.0f;
    if (chooses) share = choice.weight(a.E, a.top);
#pragma unroll
    for (int r = 0; r < R; ++r)
        scale[r] = of[r] >= a.top ? 1.0f : FEW ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(share), of[r])) : gate[of[r]];
    stage();
    __syncthreads();
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.0f;
    auto multiply = [&](const u32x4v (&v)[R][U], int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u * 512 + lane * 8;
            float xf[8];
            lds8(k < a.ld ? xs + k : nothing, xf);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float f[8];
                widen8(v[r][u], f);
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[r] = fmaf(f[e], xf[e], acc[r]);
            }
            if (u & 1) __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int k0 = 0; k0 < a.ld; k0 += 2 * STEP) {
        multiply(va, k0);
        fetch(va, k0 + 2 * STEP);  // (steps past the row ask for nothing)
        if (k0 + STEP >= a.ld) break;
        multiply(vb, k0 + STEP);
        fetch(vb, k0 + 3 * STEP);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float t = fmaxf(wave_sum(acc[r]), 0.0f);
        if (lane == r && row0 + r < total) act[row0 + r] = (AT)(t * t * scale[r]);
    }
#endif
}

static __device__ __align__(16) const uint32_t zero_chunk[32] = {};   // 64 values
constexpr int DOWN_STEP = 4096;   // values the table of starts is padded to, at least one chunk of zeros behind the sum

// Rows of the result: an expert's inner activations meet its down matrix, all of them one long sum.  LDS: the
// activations, and per 64 of them where their weights start.
template <class AT, int R>
__global__ __launch_bounds__(1024) void k_expert_down(const AT *__restrict__ act, const int *__restrict__ sel, float *__restrict__ y,
                                                      int d_p, const RowArgs a) {
    constexpr int U = exp_unroll<R>(), STEP = U * 512;
    static_assert(DOWN_STEP % STEP == 0, "whole steps");
    extern __shared__ __align__(16) uint8_t lds[];
    const int K = a.top * a.rows_e + a.rows_s, chunks = K >> 6, entries = (K / DOWN_STEP + 1) * (DOWN_STEP / 64);
    int64_t *base = (int64_t *)lds;   // in bytes from a.W (a pointer out of LDS would be loaded through as a flat one)
    AT *xs = (AT *)(base + entries), *nothing = xs + K;   // eight zeros
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), threads = blockDim.x;
    const int row0 = (blockIdx.x * (threads >> 6) + wave) * R;
    // the first pieces of the activations are requested together, in front of what waits for the choice
    constexpr int PER = 16 / sizeof(AT), FIRST = 4;
    u32x4v held[FIRST];
#pragma unroll
    for (int i = 0; i < FIRST; ++i) held[i] = *(const u32x4v *)(act + min((tid + threads * i) * PER, K - PER));
    const int routed = a.top * a.rows_e;
    if (tid < 8) nothing[tid] = (AT)0.0f;
    const int64_t behind = (const char *)a.shared - (const char *)a.W, none = (const char *)zero_chunk - (const char *)a.W;
    for (int i = tid; i < entries; i += threads) {
        const int k = (i << 6) / a.rows_e;
        base[i] = i >= chunks ? none
                  : k < a.top ? 2 * ((int64_t)sel[k] * d_p * a.rows_e + ((i << 6) - k * a.rows_e))
                              : behind + 2 * (int64_t)((i << 6) - routed);
    }
#pragma unroll
    for (int i = 0; i < FIRST; ++i)
        if ((tid + threads * i) * PER < K) *(u32x4v *)&xs[(tid + threads * i) * PER] = held[i];
    for (int i = (tid + threads * FIRST) * PER; i < K; i += threads * PER) *(u32x4v *)&xs[i] = *(const u32x4v *)(act + i);
    __syncthreads();
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.0f;
    u32x4v va[R][U], vb[R][U];
    auto fetch = [&](u32x4v (&v)[R][U], int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = min(k0 + u * 512, (entries << 6) - 512) + lane * 8;
            const char *p = (const char *)a.W + base[k >> 6] + 2 * (k & 63);
            const int pitch = 2 * (k < routed ? a.rows_e : k < K ? a.rows_s : 0);
#pragma unroll
            for (int r = 0; r < R; ++r) v[r][u] = __builtin_nontemporal_load((const u32x4v *)(p + (size_t)min(row0 + r, d_p - 1) * pitch));
        }
    };
    auto multiply = [&](const u32x4v (&v)[R][U], int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u * 512 + lane * 8;
            float xf[8];
            lds8(k < K ? xs + k : nothing, xf);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float f[8];
                widen8(v[r][u], f);
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[r] = fmaf(f[e], xf[e], acc[r]);
            }
            if (u & 1) __builtin_amdgcn_sched_barrier(0);
        }
    };
    fetch(va, 0);
    fetch(vb, STEP);
    for (int k0 = 0; k0 < K; k0 += 2 * STEP) {
        multiply(va, k0);
        fetch(va, k0 + 2 * STEP);
        if (k0 + STEP >= K) break;
        multiply(vb, k0 + STEP);
        fetch(vb, k0 + 3 * STEP);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float t = wave_sum(acc[r]);
        if (lane == r && row0 + r < d_p) y[row0 + r] = t;
    }
}

// ------------------------------------------------------------------ host side
int expert_row_values(const candy_hip_expert_spec &s) { return (int)(s.top * pad64(s.d_ff) + pad64(s.shared_ff)); }

// LDS of the one-row kernels
static size_t up_lds(const candy_hip_expert_spec &s, int64_t ld, size_t es) {
    return (size_t)ld * es + std::max((size_t)(s.n_experts + 2 * s.top) * 4, 8 * es);
}
static size_t down_lds(const candy_hip_expert_spec &s, size_t es) {
    const size_t K = (size_t)expert_row_values(s);
    return (K / DOWN_STEP + 1) * (DOWN_STEP / 64) * 8 + (K + 8) * es;
}
constexpr int64_t MOST_INNER = 29952;   // values of a row's inner activations: in bfloat16 beside 12 bytes for 64 of them, 64 KB
// (what k_route asks for with two stages when there are many experts; the limit on their number is older than that)
static bool too_many_experts(const candy_hip_expert_spec &s) {
    return ((size_t)ROUTE_T * (s.n_experts | 1) + std::max<size_t>(ROUTE_W / 2 * 64 * 17, 2 * ROUTE_T * (size_t)s.top)) * 4 > 65536;
}
static size_t route_lds(const candy_hip_expert_spec &s, int stages) {
    return (size_t)stages * ROUTE_STAGE + (size_t)ROUTE_T * (s.n_experts | 1) * 4;
}

int check_expert_spec(const candy_hip_expert_spec &s, int d) {
    CANDY_REQUIRE(s.n_experts > 0 && s.n_experts <= MAX_EXPERTS / 2 && s.top > 0 && s.top <= s.n_experts, "choice of %d out of %d experts unsupported",
                  s.top, s.n_experts);
    CANDY_REQUIRE(s.d_ff > 0 && s.shared_ff >= 0 && s.d_ff <= 1 << 20 && s.shared_ff <= 1 << 20, "invalid expert widths %d / %d", s.d_ff, s.shared_ff);
    // one workgroup keeps a row's activations in the 64 KB of LDS a launch gets without asking
    CANDY_REQUIRE(up_lds(s, pad64(d), 4) <= 65536 && (int64_t)s.top * pad64(s.d_ff) + pad64(s.shared_ff) <= MOST_INNER,
                  "%d experts of %d (+ %d) at width %d are too wide for one row's kernels", s.top, s.d_ff, s.shared_ff, d);
    CANDY_REQUIRE(!too_many_experts(s), "too many experts (%d)", s.n_experts);
    return CANDY_HIP_OK;
}

static int deal_max_tiles(const candy_hip_expert_spec &s, int n, int rows) {
    const int64_t count = (int64_t)n * s.top;
    // an expert with members has at most one tile that is not full
    return (int)(count / rows + std::min<int64_t>(s.n_experts, count));
}
static size_t deal_perm(const candy_hip_expert_spec &s, int n) { return ((size_t)n * s.top + 4 + 3) & ~(size_t)3; }
size_t expert_list_ints(const candy_hip_expert_spec &s, int n) { return deal_perm(s, n) + 4 * (size_t)deal_max_tiles(s, n, 64); }

int launch_experts_prompt(candy_hip_device *dev, const ExpertLayer &A, int n) {
    const candy_hip_expert_spec &s = A.s;
    const int rows = A.f32 ? 64 : grouped_tile_rows(s.n_experts, (int64_t)n * s.top, std::max<int64_t>(A.ld_act, pad64(s.d_ff)));
    const bool three = route_lds(s, 3) <= 160 * 1024;
    const size_t lds = route_lds(s, three ? 3 : 2);
    auto route = three ? k_route<3> : k_route<2>;
    CANDY_HIP_TRY(hipFuncSetAttribute((const void *)route, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(route, dim3((unsigned)((n + ROUTE_T - 1) / ROUTE_T)), dim3(64 * ROUTE_W), lds, dev->stream, A.x, A.ldx,
                       (const bf16 *)A.w.router->data, (int)A.w.router->ld, s.n_experts, s.top, n, A.ids, A.weights);
    CANDY_LAUNCH_CHECK();
    int *n_tiles = A.list, *perm = A.list + 4;
    GroupTile *tiles = (GroupTile *)(A.list + deal_perm(s, n));
    CANDY_REQUIRE((int64_t)n * s.top <= 0x7FFFFFFF / 2, "prompt too long for one pass");
    hipLaunchKernelGGL(k_deal, dim3(1), dim3(1024), 0, dev->stream, A.ids, n * s.top, s.n_experts, rows, perm, tiles, n_tiles);
    CANDY_LAUNCH_CHECK();
    GroupedRows gr;
    gr.perm = perm; gr.tiles = tiles; gr.n_tiles = n_tiles; gr.max_tiles = deal_max_tiles(s, n, rows); gr.tile_rows = rows;
    const int64_t ff = pad64(s.d_ff), d = pad64(A.d);
    DenseLaunch D;
    D.f32 = A.f32; D.m = n * s.top; D.group = &gr;
    gr.x_div = s.top; gr.expert_rows = (int)ff;
    D.w = A.w.up; D.x = A.x_act; D.ldx = A.ld_act; D.epi = CANDY_HIP_EPI_SQUARED_RELU; D.y = A.act; D.ldy = D.n_store = ff;
    if (int rc = launch_dense(dev, D)) return rc;
    gr.x_div = 1; gr.expert_rows = (int)d;
    D.w = A.w.down; D.x = A.act; D.ldx = ff; D.epi = CANDY_HIP_EPI_NONE; D.y = A.slots; D.ldy = D.n_store = d;
    if (int rc = launch_dense(dev, D)) return rc;
    if (!s.shared_ff) return CANDY_HIP_OK;
    DenseLaunch S;
    S.f32 = A.f32; S.m = n;
    S.w = A.w.shared_up; S.x = A.x_act; S.ldx = A.ld_act; S.epi = CANDY_HIP_EPI_SQUARED_RELU; S.y = A.shared_act;
    S.ldy = S.n_store = A.w.shared_up->rows_pad;
    if (int rc = launch_dense(dev, S)) return rc;
    S.w = A.w.shared_down; S.x = A.shared_act; S.ldx = A.w.shared_down->ld; S.epi = CANDY_HIP_EPI_NONE; S.y = A.y; S.ldy = A.ldy;
    S.n_store = A.w.shared_down->rows_pad; S.partial = A.shared; S.steady = true;
    return launch_dense(dev, S);
}

template <class AT>
static int experts_row(candy_hip_device *dev, const ExpertLayer &A) {
    const candy_hip_expert_spec &s = A.s;
    const int64_t d = pad64(A.d);
    RowArgs u;
    u.E = s.n_experts; u.top = s.top; u.rows_e = (int)pad64(s.d_ff); u.rows_s = (int)pad64(s.shared_ff); u.ld = (int)d;
    u.W = (const bf16 *)A.w.up->data;
    u.shared = s.shared_ff ? (const bf16 *)A.w.shared_up->data : nullptr;
    const int total = expert_row_values(s);
    AT *act = (AT *)A.act;
    const MvShape su = mv_shape(dev, total), sd = mv_shape(dev, d);
    const dim3 gu((unsigned)((total + su.waves * su.rows - 1) / (su.waves * su.rows))), bu((unsigned)(64 * su.waves));
    const size_t lu = up_lds(s, d, sizeof(AT)), ldn = down_lds(s, sizeof(AT));
    CANDY_REQUIRE(lu <= 65536 && ldn <= 163840, "experts too wide for this activation format");
#define CANDY_UP(R)                                                                                                          \
    do {                                                                                                                     \
        if (s.n_experts <= 64) hipLaunchKernelGGL((k_expert_up<AT, R, true>), gu, bu, lu, dev->stream, A.x, A.logits, act, A.ids, u); \
        else hipLaunchKernelGGL((k_expert_up<AT, R, false>), gu, bu, lu, dev->stream, A.x, A.logits, act, A.ids, u);          \
    } while (0)
    switch (su.rows) {
    case 1: CANDY_UP(1); break;
    case 2: CANDY_UP(2); break;
    default: CANDY_UP(4); break;
    }
#undef CANDY_UP
    CANDY_LAUNCH_CHECK();
    u.W = (const bf16 *)A.w.down->data;
    u.shared = s.shared_ff ? (const bf16 *)A.w.shared_down->data : nullptr;
    const dim3 gd((unsigned)((d + sd.waves * sd.rows - 1) / (sd.waves * sd.rows))), bd((unsigned)(64 * sd.waves));
    switch (sd.rows) {
    case 1: hipLaunchKernelGGL((k_expert_down<AT, 1>), gd, bd, ldn, dev->stream, act, A.ids, A.y, (int)d, u); break;
    case 2: hipLaunchKernelGGL((k_expert_down<AT, 2>), gd, bd, ldn, dev->stream, act, A.ids, A.y, (int)d, u); break;
    default: hipLaunchKernelGGL((k_expert_down<AT, 4>), gd, bd, ldn, dev->stream, act, A.ids, A.y, (int)d, u); break;
    }
    CANDY_LAUNCH_CHECK();
    return CANDY_HIP_OK;
}
int launch_experts_row(candy_hip_device *dev, const ExpertLayer &A) {
    return A.f32 ? experts_row<float>(dev, A) : experts_row<bf16>(dev, A);
}

int check_expert_weights(const candy_hip_device *dev, const candy_hip_expert_spec &s, const candy_hip_expert_weights &w, int64_t d) {
    auto fits = [&](const candy_hip_dense *m, int64_t rows, int64_t cols) { return m && m->dev == dev && m->rows == rows && m->cols == cols; };
    CANDY_REQUIRE(fits(w.router, s.n_experts, d) && fits(w.up, s.n_experts * pad64(s.d_ff), d) &&
                      fits(w.down, s.n_experts * pad64(d), s.d_ff) &&
                      (s.shared_ff == 0 || (fits(w.shared_up, s.shared_ff, d) && fits(w.shared_down, d, s.shared_ff))),
                  "expert weights do not fit the spec");
    return CANDY_HIP_OK;
}

// sum of the slots and the shared row, for the entry point below
__global__ __launch_bounds__(256) void k_slot_sum(const float *slots, const float *weights, const Partial shared, int top, int d, int64_t ld,
                                                  float *out, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n * d) return;
    const int64_t t = i / d, c = i % d;
    float s = 0.0f;
    if (shared.p)
        for (int k = 0; k < shared.copies; ++k) s += shared.p[(size_t)k * shared.stride + t * shared.ld + c];
    for (int k = 0; k < top; ++k) s += weights[t * top + k] * slots[(t * top + k) * ld + c];
    out[i] = s;
}

}  // namespace candy

using namespace candy;

extern "C" int candy_hip_experts(candy_hip_device *dev, const candy_hip_expert_spec *spec, int act, const candy_hip_expert_weights *w,
                                 const float *x, int64_t n, int decode, float *out, int32_t *ids, float *weights) {
    CANDY_REQUIRE(dev && spec && w && w->router && x && out, "nil argument");
    const int64_t d = w->router->cols, ld = pad64(d);
    CANDY_REQUIRE(act == CANDY_HIP_ACT_BF16 || act == CANDY_HIP_ACT_F32, "unknown activation format %d", act);
    if (int rc = check_expert_spec(*spec, (int)d)) return rc;
    if (int rc = check_expert_weights(dev, *spec, *w, d)) return rc;
    CANDY_REQUIRE(n >= 1 && n <= 1 << 16 && (!decode || n == 1), "invalid number of rows %lld", (long long)n);
    if (int rc = use_device(dev)) return rc;
    const bool f32 = act == CANDY_HIP_ACT_F32;
    const size_t es = f32 ? 4 : 2, N = (size_t)n, slots = N * spec->top;
    auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
    size_t at = 0;
    auto take = [&](size_t bytes) { const size_t p = at; at += al(bytes); return p; };
    const size_t o_x = take(N * ld * 4), o_xa = take(N * ld * es), o_id = take(slots * 4), o_w = take(slots * 4),
                 o_act = take(std::max<size_t>(slots * pad64(spec->d_ff), expert_row_values(*spec)) * es),
                 o_sact = take(N * pad64(spec->shared_ff) * es + 4), o_list = take(expert_list_ints(*spec, (int)n) * 4),
                 o_slots = take(slots * ld * 4), o_y = take(N * ld * 4), o_lg = take(w->router->rows_pad * 4);
    void *ws = nullptr;
    if (int rc = workspace(dev, at, &ws)) return rc;
    uint8_t *b = (uint8_t *)ws;
    if (int rc = launch_to_act(dev, true, x, b + o_x, n, d, ld)) return rc;
    if (int rc = launch_to_act(dev, f32, x, b + o_xa, n, d, ld)) return rc;
    ExpertLayer A;
    Partial shared;
    A.s = *spec; A.w = *w; A.d = (int)d; A.f32 = f32;
    A.x = (const float *)(b + o_x); A.ldx = ld; A.x_act = b + o_xa; A.ld_act = ld;
    A.ids = (int *)(b + o_id); A.weights = (float *)(b + o_w); A.act = b + o_act; A.shared_act = b + o_sact; A.list = (int *)(b + o_list);
    A.slots = (float *)(b + o_slots); A.y = (float *)(b + o_y); A.ldy = ld; A.shared = &shared;
    if (decode) {
        CANDY_REQUIRE(!ids && !weights, "the decode kernels keep the weights to themselves");
        DenseLaunch D;
        D.w = w->router; D.x = A.x; D.ldx = ld; D.f32 = true; D.m = 1; D.y = b + o_lg; D.ldy = D.n_store = w->router->rows_pad;
        if (int rc = launch_dense(dev, D)) return rc;
        A.logits = (const float *)(b + o_lg);
        if (int rc = launch_experts_row(dev, A)) return rc;
        return candy_hip_d2d(dev, out, A.y, (size_t)d * 4);
    }
    if (int rc = launch_experts_prompt(dev, A, (int)n)) return rc;
    hipLaunchKernelGGL(k_slot_sum, dim3((unsigned)((n * d + 255) / 256)), dim3(256), 0, dev->stream, A.slots, A.weights, shared, spec->top, (int)d,
                       ld, out, n);
    CANDY_LAUNCH_CHECK();
    if (ids)
        if (int rc = candy_hip_d2d(dev, ids, A.ids, slots * 4)) return rc;
    return weights ? candy_hip_d2d(dev, weights, A.weights, slots * 4) : CANDY_HIP_OK;
}

// The limits of a spec and what its one-row launches ask for, for a test (no device needed): 0 refused, 1 taken, -1 taken without room.
extern "C" int candy_test_expert_spec(int n_experts, int top, int d_ff, int shared_ff, int d) {
    candy_hip_expert_spec s{};
    s.n_experts = n_experts; s.top = top; s.d_ff = d_ff; s.shared_ff = shared_ff;
    if (check_expert_spec(s, d)) return 0;
    for (size_t es : {2, 4})
        if (up_lds(s, pad64(d), es) > 65536 || down_lds(s, es) > 163840) return -1;
    return 1;
}

// How many wavefronts of the launch that experts_row() makes for these widths read the choice without having made it, for a test of
// the rule (no device needed).
extern "C" int candy_test_unmade_choices(int num_cus, int top, int rows_e, int rows_s) {
    candy_hip_device dev;
    dev.num_cus = num_cus;
    const int routed = top * rows_e, total = routed + rows_s;
    const MvShape s = mv_shape(&dev, total);
    const int per_wg = s.waves * s.rows, places = (total + per_wg - 1) / per_wg * per_wg;
    int unmade = 0;
    for (int row0 = 0; row0 < places; row0 += s.rows) {
        bool reads = false;
        for (int r = 0; r < s.rows; ++r) reads = reads || up_row(row0 + r, total) < routed;
        unmade += reads && !up_chooses(row0, total, routed);
    }
    return unmade;
}
