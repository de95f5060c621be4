// Weight blocks -> fp16 operands for the kernels that contract on the fp16 matrix cores, one policy per format.
#pragma once

#include "blocks.h"

namespace candy {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ half2v bits_h2(uint32_t u) { return __builtin_bit_cast(half2v, u); }

// Unsigned levels become halves without a conversion: a byte b in the mantissa of the half 1024 is 1024 + b, exactly (bits 0x6400 | b),
// two of them one byte permutation.  From there a level takes half a packed subtraction and half a packed product where d * level
// is what is rounded (Q8_0, Q4_0: an fp16 product of two fp16 numbers rounds the same exact product once as the f32 product
// converted to fp16), or one mixed-precision multiply-add (Q6_K, Q5_K).  The same bits as level -> f32 -> product -> fp16, value by
// value, in fewer vector instructions per 16 weights: Q8_0 40 -> 31,
// Q4_0 72 -> 39 (ggml's order 96 -> 38), Q5_K 91 -> 67, Q6_K 59 -> 53.  us of a call: 11008 x 4096, 1000 rows Q5_K 133.3 -> 121.5, Q4_0 145.1 ->
// 136.1 (Q8_0 150.3 -> 149.7, Q6_K 131.6 -> 131.4: their requests bound those); 77 rows Q5_K 21.6 -> 18.7.
__device__ __forceinline__ half2v halves(uint32_t u, int pair) {  // bytes 0 and 1 of u, or 2 and 3
    return bits_h2(__builtin_amdgcn_perm(0x64646464u, u, pair ? 0x04030402u : 0x04010400u));
}
// Bytes 0 and 2, or 1 and 3: where every level goes on as one v_fma_mix that writes a half (of two levels out of one register the
// compiler makes two f32 multiply-adds and a conversion)
__device__ __forceinline__ half2v apart(uint32_t u, int odd) {
    return bits_h2(__builtin_amdgcn_perm(0x64646464u, u, odd ? 0x04030401u : 0x04020400u));
}
__device__ __forceinline__ half2v both(uint32_t h) { return bits_h2(__builtin_amdgcn_perm(h, h, 0x01000100u)); }  // the low half twice

// ------------------------------------------------------------------ per-format policies
// A task is (row, quarter c in 0..3) of one 64-wide step g in 0..3 of a super-block: 16 weights.
//   load():    the task's bytes of a whole super-block -> registers (requested four steps ahead)
//   dequant(): step g's 16 weights as two 8-value chunks and their positions (in halves) in the
//              64-wide LDS row
//   RUN16:     the chunks are 16 c .. + 7 and 16 c + 8 .. + 15 (else 8 c .. + 7 and 32 + 8 c .. + 7)

struct BigQ4K {
    static constexpr bool RUN16 = false;
    static constexpr int BLOCK = 144;
    struct Raw { u32x4 hdr; u32x2 q[4]; };  // header + bytes 8c..8c+7 of each 32-byte nibble group
    __device__ static __forceinline__ void load(const uint8_t *blk, int c, Raw &r) {
        r.hdr = *(const u32x4 *)blk;
#pragma unroll
        for (int g = 0; g < 4; ++g) r.q[g] = *(const u32x2 *)(blk + 16 + g * 32 + c * 8);
    }
    // group g holds sub-blocks 2g (low nibbles, k = 0..31 of the step) and 2g+1 (high nibbles, k = 32..63).
    // A nibble n is placed in the mantissa of the half 1024 (bits 0x6400 | n = 1024 + n, exact), two nibbles per
    // instruction, and each value is one mixed-precision multiply-add (f16 operand, f32 scale and offset, f32
    // arithmetic, rounded once to fp16): (1024 + n) * (d*sc) + (-(dmin*m) - 1024 * (d*sc)) = (d*sc)*n - dmin*m.
    // High nibbles stay where they are, four bits up (0x6400 | 16 n = 1024 + 16 n, exact as well), and take the
    // scale d*sc / 16 and the offset -(dmin*m) - 64 * (d*sc): one shift per word instead of three.
    // The offset's own f32 rounding (2^-24 of 1024 d*sc) is a thirtieth of the fp16 rounding that follows.
    __device__ static __forceinline__ uint32_t and_or(uint32_t x, uint32_t mask, uint32_t bits) {
        uint32_t r;  // (x & mask) | bits in one instruction; the mask rides on the constant bus, the bits in a register
        asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(mask), "v"(bits));
        return r;
    }
    __device__ static __forceinline__ void dequant(const Raw &r, int g, int c, half8 &o0, half8 &o1, int &k0, int &k1) {
        uint32_t sc2, m2;
        q4k_scale_min_pair(r.hdr.y, r.hdr.z, r.hdr.w, g, sc2, m2);
        const float d = half_bits_to_float((uint16_t)(r.hdr.x & 0xFFFF));
        const float dmin = half_bits_to_float((uint16_t)(r.hdr.x >> 16));
        const float d_lo = d * (float)(sc2 & 0xFF), d_hi = d * (float)((sc2 >> 8) & 0xFF);
        const float c_lo = fmaf(-1024.0f, d_lo, -(dmin * (float)(m2 & 0xFF)));
        const float c_hi = fmaf(-64.0f, d_hi, -(dmin * (float)((m2 >> 8) & 0xFF)));
        const float d_hi16 = d_hi * 0.0625f;
        const u32x2 q = r.q[g];
        const uint32_t MAGIC = 0x64006400u, LO = 0x000F000Fu, HI = 0x00F000F0u;
#pragma unroll
        for (int wi = 0; wi < 2; ++wi) {
            const uint32_t w = wi ? q.y : q.x, w8 = w >> 8;
            const half2v l02 = bits_h2(and_or(w, LO, MAGIC)), l13 = bits_h2(and_or(w8, LO, MAGIC));
            const half2v h02 = bits_h2(and_or(w, HI, MAGIC)), h13 = bits_h2(and_or(w8, HI, MAGIC));
            o0[4 * wi + 0] = (_Float16)fmaf((float)l02[0], d_lo, c_lo);
            o0[4 * wi + 1] = (_Float16)fmaf((float)l13[0], d_lo, c_lo);
            o0[4 * wi + 2] = (_Float16)fmaf((float)l02[1], d_lo, c_lo);
            o0[4 * wi + 3] = (_Float16)fmaf((float)l13[1], d_lo, c_lo);
            o1[4 * wi + 0] = (_Float16)fmaf((float)h02[0], d_hi16, c_hi);
            o1[4 * wi + 1] = (_Float16)fmaf((float)h13[0], d_hi16, c_hi);
            o1[4 * wi + 2] = (_Float16)fmaf((float)h02[1], d_hi16, c_hi);
            o1[4 * wi + 3] = (_Float16)fmaf((float)h13[1], d_hi16, c_hi);
        }
        k0 = c * 8;
        k1 = 32 + c * 8;
    }
    // The same in two parts for the kernel whose four neighbouring lanes hold the four quarters of one row: the scale
    // and offset of group g are the same for all four, so lane c works out those of group c once per super-block
    // (prepare) and each step fetches its group's from the lane that has them (four cross-lane moves instead of the
    // unpacking and six multiplies).  The same operations on the same values as dequant(): the same bits.
    struct Pre { float d_lo, d_hi16, c_lo, c_hi; };
    __device__ static __forceinline__ void prepare(const Raw &r, int c, Pre &p) {
        uint32_t sc2, m2;
        q4k_scale_min_pair(r.hdr.y, r.hdr.z, r.hdr.w, c, sc2, m2);
        const float d = half_bits_to_float((uint16_t)(r.hdr.x & 0xFFFF));
        const float dmin = half_bits_to_float((uint16_t)(r.hdr.x >> 16));
        const float d_lo = d * (float)(sc2 & 0xFF), d_hi = d * (float)((sc2 >> 8) & 0xFF);
        p.c_lo = fmaf(-1024.0f, d_lo, -(dmin * (float)(m2 & 0xFF)));
        p.c_hi = fmaf(-64.0f, d_hi, -(dmin * (float)((m2 >> 8) & 0xFF)));
        p.d_lo = d_lo;
        p.d_hi16 = d_hi * 0.0625f;
    }
    __device__ static __forceinline__ float quad_lane(float v, int g) {  // the value lane g of this lane's quad holds
        switch (g) {
        case 0: return dpp_move<0x00>(v);
        case 1: return dpp_move<0x55>(v);
        case 2: return dpp_move<0xAA>(v);
        default: return dpp_move<0xFF>(v);
        }
    }
    __device__ static __forceinline__ void dequant_pre(const Raw &r, const Pre &p, int g, int c, half8 &o0, half8 &o1,
                                                       int &k0, int &k1) {
        const float d_lo = quad_lane(p.d_lo, g), d_hi16 = quad_lane(p.d_hi16, g);
        const float c_lo = quad_lane(p.c_lo, g), c_hi = quad_lane(p.c_hi, g);
        const u32x2 q = r.q[g];
        const uint32_t MAGIC = 0x64006400u, LO = 0x000F000Fu, HI = 0x00F000F0u;
#pragma unroll
        for (int wi = 0; wi < 2; ++wi) {
            const uint32_t w = wi ? q.y : q.x, w8 = w >> 8;
            const half2v l02 = bits_h2(and_or(w, LO, MAGIC)), l13 = bits_h2(and_or(w8, LO, MAGIC));
            const half2v h02 = bits_h2(and_or(w, HI, MAGIC)), h13 = bits_h2(and_or(w8, HI, MAGIC));
            o0[4 * wi + 0] = (_Float16)fmaf((float)l02[0], d_lo, c_lo);
            o0[4 * wi + 1] = (_Float16)fmaf((float)l13[0], d_lo, c_lo);
            o0[4 * wi + 2] = (_Float16)fmaf((float)l02[1], d_lo, c_lo);
            o0[4 * wi + 3] = (_Float16)fmaf((float)l13[1], d_lo, c_lo);
            o1[4 * wi + 0] = (_Float16)fmaf((float)h02[0], d_hi16, c_hi);
            o1[4 * wi + 1] = (_Float16)fmaf((float)h13[0], d_hi16, c_hi);
            o1[4 * wi + 2] = (_Float16)fmaf((float)h02[1], d_hi16, c_hi);
            o1[4 * wi + 3] = (_Float16)fmaf((float)h13[1], d_hi16, c_hi);
        }
        k0 = c * 8;
        k1 = 32 + c * 8;
    }
};

// Q5_K: Q4_K's layout with 32 bytes of fifth bits between the header and the nibbles (quantized.cu:1044-1080):
// bit t of byte l is the fifth bit of value l of sub-block t.
struct BigQ5K {
    static constexpr bool RUN16 = false;
    static constexpr int BLOCK = 176;
    struct Raw { u32x4 hdr; u32x2 qh; u32x2 q[4]; };
    __device__ static __forceinline__ void load(const uint8_t *blk, int c, Raw &r) {
        r.hdr = *(const u32x4 *)blk;
        r.qh = *(const u32x2 *)(blk + 16 + c * 8);
#pragma unroll
        for (int g = 0; g < 4; ++g) r.q[g] = *(const u32x2 *)(blk + 48 + g * 32 + c * 8);
    }
    __device__ static __forceinline__ void dequant(const Raw &r, int g, int c, half8 &o0, half8 &o1, int &k0, int &k1) {
        uint32_t sc2, m2;
        q4k_scale_min_pair(r.hdr.y, r.hdr.z, r.hdr.w, g, sc2, m2);
        const float d = half_bits_to_float((uint16_t)(r.hdr.x & 0xFFFF));
        const float dmin = half_bits_to_float((uint16_t)(r.hdr.x >> 16));
        const float d_lo = d * (float)(sc2 & 0xFF), d_hi = d * (float)((sc2 >> 8) & 0xFF);
        const float m_lo = dmin * (float)(m2 & 0xFF), m_hi = dmin * (float)((m2 >> 8) & 0xFF);
        const u32x2 q = r.q[g];
        const half2v one_k = {(_Float16)1024.0f, (_Float16)1024.0f};
#pragma unroll
        for (int wi = 0; wi < 2; ++wi) {
            const uint32_t w = wi ? q.y : q.x, h = wi ? r.qh.y : r.qh.x;
            const uint32_t lo = (w & 0x0F0F0F0Fu) | (((h >> (2 * g)) & 0x01010101u) << 4);
            const uint32_t hi = ((w >> 4) & 0x0F0F0F0Fu) | (((h >> (2 * g + 1)) & 0x01010101u) << 4);
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const half2v l2 = halves(lo, p) - one_k, h2 = halves(hi, p) - one_k;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    o0[4 * wi + 2 * p + j] = (_Float16)fmaf((float)l2[j], d_lo, -m_lo);
                    o1[4 * wi + 2 * p + j] = (_Float16)fmaf((float)h2[j], d_hi, -m_hi);
                }
            }
        }
        k0 = c * 8;
        k1 = 32 + c * 8;
    }
};

// Q8_0: a "super-block" is eight 34-byte blocks (272 bytes); step g holds blocks 2g and 2g + 1, the task's quarter c
// the 16 quants of half a block and that block's scale.  d * q (DequantizeBlockQ8_0F32, quantized.go:131-136) as one packed fp16
// product: of two fp16 numbers, so that what is rounded, once, is the exact product.
struct BigQ8_0 {
    static constexpr bool RUN16 = true;
    static constexpr int BLOCK = 272;
    struct Raw { u32x4 q[4]; uint32_t d01, d23; };
    __device__ static __forceinline__ void load(const uint8_t *blk, int c, Raw &r) {
        uint32_t d[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const uint8_t *b = blk + 34 * (2 * g + (c >> 1));
            d[g] = *(const uint16_t *)b;
            r.q[g] = *(const u32x4_a2 *)(b + 2 + 16 * (c & 1));
        }
        r.d01 = d[0] | (d[1] << 16);
        r.d23 = d[2] | (d[3] << 16);
    }
    __device__ static __forceinline__ void dequant(const Raw &r, int g, int c, half8 &o0, half8 &o1, int &k0, int &k1) {
        const uint32_t dd = g < 2 ? r.d01 : r.d23;
        const half2v d = both(dd >> (16 * (g & 1))), mid = {(_Float16)1152.0f, (_Float16)1152.0f};
        const uint32_t w[4] = {r.q[g].x, r.q[g].y, r.q[g].z, r.q[g].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t u = w[i] ^ 0x80808080u;  // q + 128
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const half2v v = (halves(u, p) - mid) * d;
                half8 &o = i < 2 ? o0 : o1;
                o[4 * (i & 1) + 2 * p] = v[0];
                o[4 * (i & 1) + 2 * p + 1] = v[1];
            }
        }
        k0 = 32 * (c >> 1) + 16 * (c & 1);
        k1 = k0 + 8;
    }
};

// Q4_0: eight 18-byte blocks per "super-block" (144 bytes).  The task's 16 values of block 2g + c/2 are the two
// nibbles of 8 consecutive bytes in candy's element order (quantized.go:85-93) or one nibble of all 16 bytes in
// ggml's.  d * (q - 8) as for Q8_0: one packed fp16 product, the exact product rounded once.
template <bool GGML>
struct BigQ4_0 {
    static constexpr bool RUN16 = true;
    static constexpr int BLOCK = 144;
    struct Raw { u32x4 q[4]; uint32_t d01, d23; };
    __device__ static __forceinline__ void load(const uint8_t *blk, int c, Raw &r) {
        uint32_t d[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const uint8_t *b = blk + 18 * (2 * g + (c >> 1));
            d[g] = *(const uint16_t *)b;
            if (GGML) {
                r.q[g] = *(const u32x4_a2 *)(b + 2);
            } else {
                const u32x2 h = *(const u32x2_a2 *)(b + 2 + 8 * (c & 1));
                r.q[g] = u32x4{h.x, h.y, 0u, 0u};
            }
        }
        r.d01 = d[0] | (d[1] << 16);
        r.d23 = d[2] | (d[3] << 16);
    }
    __device__ static __forceinline__ void dequant(const Raw &r, int g, int c, half8 &o0, half8 &o1, int &k0, int &k1) {
        const uint32_t dd = g < 2 ? r.d01 : r.d23;
        const half2v d = both(dd >> (16 * (g & 1))), mid = {(_Float16)1032.0f, (_Float16)1032.0f};
        const uint32_t w[4] = {r.q[g].x, r.q[g].y, r.q[g].z, r.q[g].w};
        if (GGML) {
            const int sh = 4 * (c & 1);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t u = (w[i] >> sh) & 0x0F0F0F0Fu;
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    const half2v v = (halves(u, p) - mid) * d;
                    half8 &o = i < 2 ? o0 : o1;
                    o[4 * (i & 1) + 2 * p] = v[0];
                    o[4 * (i & 1) + 2 * p + 1] = v[1];
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const uint32_t even = w[i] & 0x0F0F0F0Fu, odd = (w[i] >> 4) & 0x0F0F0F0Fu;
#pragma unroll
                for (int j = 0; j < 4; ++j) {  // byte j: values 2j and 2j + 1
                    const half2v v = (bits_h2(__builtin_amdgcn_perm(odd, even, 0x0C040C00u + 0x00010001u * j) | 0x64006400u) - mid) * d;
                    half8 &o = i ? o1 : o0;
                    o[2 * j] = v[0];
                    o[2 * j + 1] = v[1];
                }
            }
        }
        k0 = 32 * (c >> 1) + 16 * (c & 1);
        k1 = k0 + 8;
    }
};

struct BigQ6K {
    static constexpr bool RUN16 = true;
    static constexpr int BLOCK = 210;
    // per half ip: ql bytes 64ip+16c..+15 (low nibbles: quarters 0/1, high nibbles: quarters 2/3) and qh bytes
    // 32ip+16(c&1)..+15; the four scales of this quarter-column (8ip + 4p + c) packed in one word; d
    struct Raw { u32x4 ql[2], qh[2]; uint32_t sc4; uint32_t d; };
    __device__ static __forceinline__ void load(const uint8_t *blk, int c, Raw &r) {
#pragma unroll
        for (int ip = 0; ip < 2; ++ip) {
            r.ql[ip] = *(const u32x4_a2 *)(blk + 64 * ip + 16 * c);
            r.qh[ip] = *(const u32x4_a2 *)(blk + 128 + 32 * ip + 16 * (c & 1));
        }
        const uint8_t *sc = blk + 192 + c;
        r.sc4 = (uint32_t)sc[0] | ((uint32_t)sc[4] << 8) | ((uint32_t)sc[8] << 16) | ((uint32_t)sc[12] << 24);
        r.d = *(const uint16_t *)(blk + 208);
    }
    // step g = 2*ip + p covers k = 128ip + 64p .. +63: quarters 2p and 2p+1 of half ip; this task owns
    // values 16c..16c+15 of the step, i.e. quarter 2p + (c>>1), il = 16(c&1)..+15, one scale
    __device__ static __forceinline__ void dequant(const Raw &r, int g, int c, half8 &o0, half8 &o1, int &k0, int &k1) {
        const int ip = g >> 1, p = g & 1;
        const int shift = 2 * (2 * p + (c >> 1));
        const float dsc = half_bits_to_float((uint16_t)r.d) * (float)(int)(int8_t)((r.sc4 >> (8 * g)) & 0xFF);
        const float off = -1056.0f * dsc;  // of 1024 + q; 18 bits times 33, exact, and so is the sum d*sc*(q-32)
        const uint32_t qlw[4] = {r.ql[ip].x, r.ql[ip].y, r.ql[ip].z, r.ql[ip].w};
        const uint32_t qhw[4] = {r.qh[ip].x, r.qh[ip].y, r.qh[ip].z, r.qh[ip].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t lo4 = (qlw[j] >> (4 * p)) & 0x0F0F0F0Fu;
            const uint32_t hi2 = ((qhw[j] >> shift) & 0x03030303u) << 4;
            const uint32_t q = lo4 | hi2;
#pragma unroll
            for (int p2 = 0; p2 < 2; ++p2) {
                const half2v h = apart(q, p2);
                half8 &o = j < 2 ? o0 : o1;
                o[4 * (j & 1) + p2] = (_Float16)fmaf((float)h[0], dsc, off);
                o[4 * (j & 1) + 2 + p2] = (_Float16)fmaf((float)h[1], dsc, off);
            }
        }
        k0 = 16 * c;
        k1 = 16 * c + 8;
    }
};

}  // namespace candy
