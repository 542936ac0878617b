// fp32 products on the bf16 matrix instructions.
//
// A float's 24 significant bits are three bf16 values' worth: x = h + m + l exactly, h the float rounded to bf16, m what is
// left rounded to bf16, l the rest.  A product of two floats is then six products of pieces, h h + (h m + m h) +
// (h l + m m + l h), and three that are left out, m l, l m and l l, of at most 2^-25 of it together: less than rounding a
// float leaves.  v_mfma_f32_32x32x16_bf16 sums 16 products in 32 cycles where v_mfma_f32_32x32x2_f32 takes 512, so six of
// them take 192: 2.7 times the rate, and a sixteenth as often rounded.
//
// What the bf16 instruction adds to a sum far above it is cut off below the sum's last place, so the small products go in
// first or have an accumulator of their own, and long sums are taken tile by tile and added up with ordinary additions.
// Relative error (2-norm) against 64 bits, fp32 instructions / this:  dot products of N(0,1) over d = 64 1.4e-7 / 4.9e-8,
// d = 128 2.0e-7 / 6.5e-8;  softmax weights times N(0,1) over 512 keys 4.1e-7 / 1.1e-7, 2048 keys 8.0e-7 / 1.7e-7;  sums of
// positive products over 2048 keys 7.0e-7 / 1.3e-7.
//
// Infinities have no such pieces (inf - inf, and 0 inf where a factor's lower pieces are zero), and pieces below 2^-126 count
// as zero in the instruction.  So the kernels watch the magnitudes of what they split, and a workgroup that meets anything
// outside Magnitudes' range does its work again with the fp32 instructions.
#pragma once

#include "ahpc_device.hpp"

namespace ahpc {

// The pieces of 8 values as operands of the 32x32x16 instruction.
struct F32x3 {
    u32x4 h, m, l;
};

__device__ inline F32x3 split_f32(const float (&x)[8]) {
    F32x3 out;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t h = pack2<bf16_t>(x[2 * i], x[2 * i + 1]);
        const float a = x[2 * i] - lo_f32<bf16_t>(h), b = x[2 * i + 1] - hi_f32<bf16_t>(h);
        const uint32_t m = pack2<bf16_t>(a, b);
        out.h[i] = h;
        out.m[i] = m;
        out.l[i] = pack2<bf16_t>(a - lo_f32<bf16_t>(m), b - hi_f32<bf16_t>(m));
    }
    return out;
}

// The magnitudes of the groups of 8 values seen so far: the largest, and the smallest among those of groups that hold
// something other than zeros.
struct Magnitudes {
    float largest = 0.0f, smallest = 1.0f;
    __device__ void see(const float (&x)[8]) {
        float top = fmaxf(__builtin_fabsf(x[0]), __builtin_fabsf(x[1]));
#pragma unroll
        for (int i = 2; i < 8; i += 2) top = fmaxf(fmaxf(top, __builtin_fabsf(x[i])), __builtin_fabsf(x[i + 1]));
        largest = fmaxf(largest, top);
        smallest = fminf(smallest, top > 0.0f ? top : 1.0f);
    }
    // Three pieces hold everything: from 2^-100, whose last piece is above 2^-126 down to a 24th bit, to where rounding to
    // bf16 would overflow.
    __device__ bool in_range() const { return largest < 3.38e38f && smallest >= 7.9e-31f; }
};

// lo += the five small products of 16 contracted values, hi += the large one.  Smallest first.
__device__ inline void mfma_x3(const F32x3& a, const F32x3& b, f32x16& hi, f32x16& lo) {
    lo = mfma_32x32x16<bf16_t>(a.h, b.l, lo);
    lo = mfma_32x32x16<bf16_t>(a.l, b.h, lo);
    lo = mfma_32x32x16<bf16_t>(a.m, b.m, lo);
    lo = mfma_32x32x16<bf16_t>(a.h, b.m, lo);
    lo = mfma_32x32x16<bf16_t>(a.m, b.h, lo);
    hi = mfma_32x32x16<bf16_t>(a.h, b.h, hi);
}

// The three planes of a tile of 32 rows in LDS, [plane][32 rows][D] bf16, 16-byte chunk c of row r at chunk c ^ f(r): what
// the 16-bit kernels have as tiles of 64 rows, with their swizzles (FlashTile).
template <int D> struct X3Tile {
    static constexpr int RB = 2 * D;
    static constexpr int CH = D / 8;
    static constexpr int kPlane = 32 * RB;
    static constexpr int kBytes = 3 * kPlane;
    __device__ static void put(unsigned char* tile, int row, int chunk_at, const F32x3& x) {
        unsigned char* const dst = tile + row * RB + (chunk_at << 4);
        *reinterpret_cast<u32x4*>(dst) = x.h;
        *reinterpret_cast<u32x4*>(dst + kPlane) = x.m;
        *reinterpret_cast<u32x4*>(dst + 2 * kPlane) = x.l;
    }
    __device__ static F32x3 row_operand(const unsigned char* at) {
        return F32x3{lds_read_b128(at), lds_read_b128(at + kPlane), lds_read_b128(at + 2 * kPlane)};
    }
};

}  // namespace ahpc
