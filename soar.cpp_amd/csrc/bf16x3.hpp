// bf16x3.hpp - fp32 products on the bf16 matrix cores.
//
// gfx950's bf16 matrix instructions run at 16 times the rate of its fp32
// ones.  An fp32 value is split into three bf16 parts, x = h + m + l, each
// the round-to-nearest bf16 (eight significant bits) of what the parts before
// it leave: |m| <= 2^-8 |x|, |l| <= 2^-17 |x|, and l leaves nothing.  A
// product then takes the six part products down to 2^-17 of it,
//   h h' + (h m' + m h') + (m m' + h l' + l h'),
// each exact in fp32 and added in fp32 by the matrix core; the three left
// out are together at most 2^-24 |x x'|, as much as rounding the product to
// fp32 (on average less: a sum of many products is nearer to exact than an
// fp32 one, mma_step; a single product's error can be twice as large).  It
// takes 6/16 of the fp32 matrix time plus the splits.
//
// Range.  The parts are those of 2^16 x (kBf3Up): fp32's last bit is 2^-149,
// bf16's 2^-133 (the conversions and the matrix cores keep denormals), so
// the split is exact for every x; unscaled, it lost bits from 2^-109 down.
// Sums come out 2^32 times as large and are scaled back by kBf3Down.  The
// scale costs 2-4%: 192 -> 384 channels at 128^2 pixels forward 22.4 -> 23.0,
// input gradient 25.8 -> 26.8, weight gradient with its finish 34.0 -> 35.0 us.
//
// Non-finite inputs: an infinity (or a finite value that the scale takes
// there, |x| >= 2^112) leaves a NaN remainder, so every output it reaches
// comes out non-finite, as does one above 2^96.  The kernels test their
// accumulators and run a tile that has a non-finite one again on the fp32
// instructions, so infinities, NaN and large values come out as fp32 products
// and sums give them.
#pragma once

#include <hip/hip_runtime.h>

namespace soar {
namespace gn {

typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

// One of the three parts of eight values, and all three.
typedef unsigned u4 __attribute__((ext_vector_type(4)));
struct Bf3 {
    u4 p[3];  // h, m, l: pairs of bf16 values
};

constexpr float kBf3Up = 0x1p16f, kBf3Down = 0x1p-32f;

// The parts of eight values, scaled: per pair two products, three packed
// conversions and four unpacked subtractions, thirteen instructions.  (A remainder as one bf16 dot
// product with (-1, 0) takes seven, but v_dot2_f32_bf16 does not run beside
// the matrix instructions of the SIMD as these do: 24 MFMAs with 144 of
// either took 1503 ns against 876-921 for two waves of a SIMD, 783 ns for
// the MFMAs alone.)
__device__ __forceinline__ Bf3 bf3_split(float v0, float v1, float v2, float v3, float v4,
                                         float v5, float v6, float v7) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    f2 v[4] = {{v0 * kBf3Up, v1 * kBf3Up},
               {v2 * kBf3Up, v3 * kBf3Up},
               {v4 * kBf3Up, v5 * kBf3Up},
               {v6 * kBf3Up, v7 * kBf3Up}};
    Bf3 o;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const unsigned b = __builtin_bit_cast(unsigned, __builtin_convertvector(v[i], bf2));
            o.p[p][i] = b;
            if (p < 2) {
                v[i].x -= __builtin_bit_cast(float, b << 16);
                v[i].y -= __builtin_bit_cast(float, b & 0xffff0000u);
            }
        }
    }
    return o;
}

__device__ __forceinline__ bf8 bf3_part(const Bf3& v, int p) {
    return __builtin_bit_cast(bf8, v.p[p]);
}

// The six part products of an MFMA step, smallest first: fn(a part, b part).
template <typename F>
__device__ __forceinline__ void bf3_products(F&& fn) {
    fn(2, 0);
    fn(1, 1);
    fn(0, 2);
    fn(1, 0);
    fn(0, 1);
    fn(0, 0);
}

}  // namespace gn
}  // namespace soar
