// bf16x3.hpp - fp32 products on the bf16 matrix cores.
//
// gfx950's bf16 matrix instructions run at 16 times the rate of its fp32
// ones.  An fp32 value is split into three bf16 parts, x = h + m + l, each
// the round-to-nearest bf16 of what the parts before it leave: |m| <= 2^-9
// |x|, |l| <= 2^-18 |x|, and what l leaves is at most 2^-27 |x|.  A product
// then takes the six part products down to 2^-18 of it,
//   h h' + (h m' + m h') + (m m' + h l' + l h'),
// each exact in fp32 and added in fp32 by the matrix core; the three left
// out and the splits' remainders are together at most 2^-25 |x x'|, half an
// fp32 rounding of the product itself.  So the result has the error of an
// fp32 dot product, at 6/16 of its matrix time plus the splits.
//
// Non-finite inputs: an infinity (or a finite value that rounds to one as
// bf16, |x| >= 2^128 (1 - 2^-9)) leaves a NaN remainder, so every output it
// reaches comes out non-finite.  The kernels test their accumulators and
// run a tile that has a non-finite one again on the fp32 instructions, so
// infinities and NaN come out as fp32 products and sums give them.  (Parts
// below 2^-126 are flushed: an absolute error below 2^-126 |x'|.)
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

// The parts of eight values: per pair three packed conversions and four
// unpacked subtractions, eleven instructions.  (A remainder as one bf16 dot
// product with (-1, 0) takes seven, but v_dot2_f32_bf16 does not run beside
// the matrix instructions of the SIMD as these do: 24 MFMAs with 144 of
// either took 1503 ns against 876-921 for two waves of a SIMD, 783 ns for
// the MFMAs alone.)
__device__ __forceinline__ Bf3 bf3_split(float v0, float v1, float v2, float v3, float v4,
                                         float v5, float v6, float v7) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    f2 v[4] = {{v0, v1}, {v2, v3}, {v4, v5}, {v6, v7}};
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
