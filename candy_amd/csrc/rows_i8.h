// Launch descriptor of the row contraction (rows_i8.hip) and the layout of its activations.
#pragma once

#include "internal.h"

namespace candy {

struct RowsJob {
    const uint8_t *W;
    float *y;
    const float *res;  // optional, added to the result (may be y)
    int N;
    int wg_end;
};
struct RowsJobs {
    RowsJob j[3];
};
// Activations in operand order: tiles of 16 rows.  Per tile
//   frag  [K/256][4][64 lanes][16 bytes]: lane (row r = lane & 15, chunk c = lane >> 4) of pair p holds values 8c .. 8c + 7 of
//         sub-blocks 2p and 2p + 1 of row r, as int8
//   d     [K/256 + 1][16 rows][8 sub-blocks] scales;  m: the same shape, d * sum of the levels
// Rows past the last one may hold anything: a row reaches its own results only.
struct RowsImage {
    uint8_t *frag = nullptr;
    float *d = nullptr, *m = nullptr;
    size_t frag_stride = 0, scale_stride = 0;  // bytes / floats from one tile to the next
};
__host__ __device__ inline size_t rows_frag_bytes(int64_t K) { return ((size_t)16 * (size_t)K + 255) & ~(size_t)255; }
inline size_t rows_scales_bytes(int64_t K) { return (((size_t)((K >> 8) + 1) * 16 * 8 * sizeof(float)) + 255) & ~(size_t)255; }
// tiles of 16 activation rows in the image: whole workgroups of one to four
inline int64_t rows_tiles(int64_t m) { return m <= 48 ? (m + 15) / 16 : (m + 63) / 64 * 4; }
inline size_t rows_image_bytes(int64_t m, int64_t K) {
    return (size_t)rows_tiles(m) * (rows_frag_bytes(K) + 2 * rows_scales_bytes(K)) + 256;
}
inline RowsImage rows_image(void *p, int64_t m, int64_t K) {
    const size_t tiles = (size_t)rows_tiles(m);
    RowsImage x;
    x.frag_stride = rows_frag_bytes(K);
    x.scale_stride = rows_scales_bytes(K) / sizeof(float);
    x.frag = (uint8_t *)p;
    x.d = (float *)(x.frag + tiles * x.frag_stride);
    x.m = x.d + tiles * x.scale_stride;
    return x;
}
__device__ __forceinline__ size_t rows_frag_offset(int r, int k) {
    const int sb = k >> 8, t = (k >> 5) & 7, c = (k >> 3) & 3;
    return ((size_t)((sb * 4 + (t >> 1)) * 64 + c * 16 + r)) * 16 + (t & 1) * 8 + (k & 7);
}
// Values 4 c4 .. 4 c4 + 3 of a row, quantized (quantize_q8_lane4), into the image.
__device__ __forceinline__ void rows_put(const RowsImage &o, int row, int c4, uint32_t packed, __half h, int bsum) {
    const int tile = row >> 4, r = row & 15, k = 4 * c4;
    *(uint32_t *)(o.frag + tile * o.frag_stride + rows_frag_offset(r, k)) = packed;
    if ((k & 31) == 0) {
        const float d = __half2float(h);
        const size_t at = tile * o.scale_stride + ((size_t)(k >> 8) * 16 + r) * 8 + ((k >> 5) & 7);
        o.d[at] = d;
        o.m[at] = d * (float)bsum;
    }
}
struct RowsLaunch {
    int n = 0;
    const candy_hip_qtensor *w[3] = {nullptr, nullptr, nullptr};
    float *y[3] = {nullptr, nullptr, nullptr};
    const float *res[3] = {nullptr, nullptr, nullptr};
    RowsImage x;
};
bool rows_i8_covers(const candy_hip_qtensor *w);  // whether the kernel takes the weight
bool rows_i8_takes(const candy_hip_qtensor *w, int64_t m);  // the same with the batch and the options
// whether a single contraction of m rows goes there; exact: its quants are planar already and the alternatives are the exact kernels only
// (else f32 rows or Q8_0 blocks, and kernels with fp16 operands as well)
bool rows_i8_picks(const candy_hip_qtensor *w, int64_t m, bool exact);
int launch_rows_i8(candy_hip_device *dev, const RowsLaunch &L, int64_t m);
// f32 rows, Q8_0 blocks or planar quants -> the image
int launch_rows_quantize(candy_hip_device *dev, const float *x, int64_t m, int64_t K, const RowsImage &o);
int launch_rows_pack_blocks(candy_hip_device *dev, const void *blocks, int64_t m, int64_t K, const RowsImage &o);
int launch_rows_pack_planar(candy_hip_device *dev, const int8_t *qs, const Q8Scale *scales, int64_t m, int64_t K, const RowsImage &o);

}  // namespace candy
