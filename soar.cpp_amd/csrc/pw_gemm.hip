// pw_gemm.hip - block-tiled pointwise convolution for wide layers: forward
// (with the GroupNorm statistics of its output), input gradient and weight
// gradient as GEMMs on the bf16 matrix cores at fp32 accuracy (bf16x3.hpp).
//
// k_pw_conv gives every wave its own 64-row x 128-pixel tile and reads both
// operands from the caches into registers: 21 multiply-adds per byte, so a
// layer of more than about 64 rows and channels asks the caches for more
// than 10 TB/s and waits on them.  Here a block of four waves owns a 64 x
// 128 tile and stages each 32-deep K step of both operands through LDS
// once: the operands are split into their bf16 parts as they are staged
// (once per block and not once per wave), and the waves' 32 x 64 tiles read
// them back with conflict-free 16-byte reads.
//
// LDS: part p and group g of eight K values form a plane of 64 or 128 slots
// (the tile's rows or columns) of 16 bytes, the eight bf16 values of the
// slot: what a lane of the 32x32x16 MFMA takes.  Planes are padded by 64
// bytes, so the four planes of a part that a row-wise staging write touches
// start on different banks.  One stage of both operands (38 KB) per block:
// three blocks share a CU, and one block's loads, splits and waits run
// beside another's MFMAs.  What bounds a large grid is the LDS traffic (9
// KB read per 12 MFMAs of a wave, beside the staging) and the MFMAs
// together: 130 TFLOP/s of fp32 product for the input gradient of 128 -> 256
// channels over 2^20 pixels (k_pw_conv 92), 96 / 87 / 89 for 192 -> 384 at
// 128^2 (25.3 / 27.8 / 27.1 us forward with statistics / input gradient /
// weight gradient).  (Measured and not kept, before the operands' scale, us
// for those three, 23.9 / 26.5 / 26.0 as it was: 128 x 128 tiles 26.7 / 30.4
// / 37; loads two steps ahead 28.3 / 28.3 / 27.7; two stages with the
// next step's splits between the MFMAs, two blocks per CU, 30.6 / 29.9 / 35.7.)
//
// Operands whose K axis runs along the rows (W in the forward, dz and x in
// the weight gradient) are staged row by row: four lanes take 128
// consecutive bytes of a row.  Operands whose K axis runs across the rows (x
// in the forward; W and dz in the input gradient) are staged column by
// column: a lane takes four consecutive columns of eight rows.
//
// Rows and vectors need 4-byte alignment only (gfx950 loads and stores 16
// bytes at any dword address), so planes of any size take this path; where a
// row's last vector is partial, its loads are 4-byte ones.
#include <algorithm>
#include <type_traits>

#include "bf16x3.hpp"
#include "gn_internal.hpp"
#include "gn_math.hpp"
#include "gn_moments.hpp"
#include "soar_gn.h"

namespace soar {
namespace gn {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f16 __attribute__((ext_vector_type(16)));
typedef unsigned u2 __attribute__((ext_vector_type(2)));

constexpr int kGm = 64;                 // tile rows
constexpr int kGp = 128;                // tile columns (pixels)
constexpr int kGk = 32;                 // K values per step
constexpr int kPlaneA = kGm * 16 + 64;  // bytes of one (part, K group) plane
constexpr int kPlaneB = kGp * 16 + 64;
constexpr int kOperandA = 12 * kPlaneA, kOperandB = 12 * kPlaneB;
constexpr int kStatPitch = 34;          // float2 per row of the statistics transpose

enum GemmMode { kGemmPlain = 0, kGemmStats = 1, kGemmAccum = 2 };

// Row of a 32-row MFMA tile held in accumulator register r (half-wave 0;
// half-wave 1 holds the row 4 further).
__device__ __forceinline__ int mma_row(int r) { return (r & 3) + 8 * (r >> 2); }

// A raw buffer descriptor over `floats` floats at p: loads past them return
// zero, stores past them are dropped (gemm_fits: below 2^31 bytes).
__device__ __forceinline__ auto buffer_of(const float* p, int64_t floats) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), (short)0, (int)(4 * floats),
                                             0x00020000);
}
typedef decltype(buffer_of(nullptr, 0)) Buffer;

__device__ __forceinline__ f4 load4(Buffer b, uint32_t off) {
    return __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(b, off, 0, 0));
}
__device__ __forceinline__ float load1(Buffer b, uint32_t off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(b, off, 0, 0));
}

// Eight rows of four consecutive columns: rows k .. k + 7 (zero from the
// matrix's last row on) of the matrix in `b` (row length ld), columns c ..
// c + 3.  Columns past the row's end hold values of the next row: they reach
// only outputs that are not stored.  `whole` (block-uniform): no vector of
// the tile crosses a row's end, so none crosses the matrix's.
__device__ __forceinline__ void load_cols(f4 (&st)[8], Buffer b, uint32_t ld, uint32_t k,
                                          uint32_t c, bool whole) {
    uint32_t o = 4u * (k * ld + c);
    asm volatile("" : "+v"(o));  // (no offset is hoisted out of the step loop)
    if (whole) {
#pragma unroll
        for (int e = 0; e < 8; ++e) st[e] = load4(b, o + 4u * e * ld);
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int u = 0; u < 4; ++u) st[e][u] = load1(b, o + 4u * e * ld + 4u * u);
    }
}

// Splits them and writes K group g of slots slot0 + step u, u the column.
template <int PLANE>
__device__ __forceinline__ void stage_cols(const f4 (&st)[8], char* __restrict__ op, int g,
                                           int slot0, int step) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const Bf3 s = bf3_split(st[0][u], st[1][u], st[2][u], st[3][u], st[4][u], st[5][u],
                                st[6][u], st[7][u]);
        char* d = op + g * PLANE + (slot0 + step * u) * 16;
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<u4*>(d + 4 * p * PLANE) = s.p[p];
    }
}

// The same for the pixels 4 i + u of the forward: slots slot0 + 32 (u & 1) +
// 16 (u / 2).
__device__ __forceinline__ void stage_x(const f4 (&st)[8], char* __restrict__ op, int g,
                                        int slot0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const Bf3 s = bf3_split(st[0][u], st[1][u], st[2][u], st[3][u], st[4][u], st[5][u],
                                st[6][u], st[7][u]);
        char* d = op + g * kPlaneB + (slot0 + 32 * (u & 1) + 16 * (u >> 1)) * 16;
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<u4*>(d + 4 * p * kPlaneB) = s.p[p];
    }
}

// Eight consecutive K values k .. k + 7 (zero from kend on) of rows r, r +
// 16, r + 32 and r + 48 of the matrix in `b` (rows past it are zero).
// `whole` (block-uniform): kend is a multiple of 4.
__device__ __forceinline__ void load_rows(f4 (&st)[8], Buffer b, uint32_t ld, uint32_t r,
                                          uint32_t k, uint32_t kend, bool whole) {
    constexpr uint32_t kNone = 0x80000000u;  // past every descriptor's range
    uint32_t o = 4u * (r * ld + k);
    asm volatile("" : "+v"(o));
    if (whole) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t q = 4u * (e & 1);
            st[e] = load4(b, k + q < kend ? o + 64u * (e >> 1) * ld + 4u * q : kNone);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const uint32_t q = 4u * (e & 1) + u;
                st[e][u] = load1(b, k + q < kend ? o + 64u * (e >> 1) * ld + 4u * q : kNone);
            }
    }
}

// Splits them and writes K group g of slots slot, slot + 16, ...
template <int PLANE>
__device__ __forceinline__ void stage_rows(const f4 (&st)[8], char* __restrict__ op, int g,
                                           int slot) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const f4 a = st[2 * e], b = st[2 * e + 1];
        const Bf3 s = bf3_split(a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]);
        char* d = op + g * PLANE + (slot + 16 * e) * 16;
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<u4*>(d + 4 * p * PLANE) = s.p[p];
    }
}

template <int PLANE>
__device__ __forceinline__ bf8 read_slot(const char* __restrict__ op, int p, int g, int slot) {
    return *reinterpret_cast<const bf8*>(op + (4 * p + g) * PLANE + slot * 16);
}

// The step's MFMAs of a wave's 32 x 64 tile: row slots sa, column slots sc
// and sc + 32 (this lane's).  The products of the high parts go to acc, the
// five smaller ones (at most 2^-8 of them) to lo, added at the end: acc is
// then rounded once per 16 K values and not six times, and a sum over K has
// no larger error than the split sums of k_pw_conv (z over 192 / 320
// channels: 2.0e-7 / 2.7e-7 of its norm with one accumulator).
__device__ __forceinline__ void mma_step(f16 (&acc)[2], f16 (&lo)[2], const char* __restrict__ opa,
                                         const char* __restrict__ opb, int sa, int sc, int h) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        bf8 A[3], B[2][3];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            A[p] = read_slot<kPlaneA>(opa, p, 2 * ks + h, sa);
#pragma unroll
            for (int t = 0; t < 2; ++t) B[t][p] = read_slot<kPlaneB>(opb, p, 2 * ks + h, sc + 32 * t);
        }
        bf3_products([&](int p, int q) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                f16& d = p + q == 0 ? acc[t] : lo[t];
                d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[p], B[t][q], d, 0, 0, 0);
            }
        });
    }
}

// Whether some accumulator of the wave is infinite or NaN.
__device__ __forceinline__ bool any_nonfinite(const f16 (&acc)[2]) {
    float bad = 0.0f;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) bad = fmaf(acc[t][r], 0.0f, bad);
    return __any(bad != 0.0f);
}

__device__ __forceinline__ void clear(f16 (&acc)[2]) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] = 0.0f;
}

// Blocks that share an operand (the `inner` tiles of one outer tile) run on
// one XCD, one after another: block b is XCD b % 8's, whose L2 then holds
// the shared operand.  outer >= the number of outer tiles for the blocks of
// the padded grid.
__device__ __forceinline__ void xcd_tile(uint32_t b, uint32_t inner, int64_t* outer, int* in) {
    const uint32_t w = b / (8 * inner), r = b - w * 8 * inner;
    *outer = (int64_t)w * 8 + (r & 7);
    *in = (int)(r >> 3);
}

// z[m][p] = bias[m] + sum_k w[m][k] x[k][p] per sample (z += with
// kGemmAccum); TW: w[k][m].  kGemmStats: also the GroupNorm chunk partials
// part[(n*M + m)*cpp + chunk] (k_pw_conv's layout and arithmetic: sums of an
// item's values shifted by the item's first, folded in float64).
//
// Waves 0 and 1 stage x, wave 2 W.  Pixel 64 wn + 2 j + t of the item is
// column j of wave column wn's n-tile t, so a lane stores two consecutive
// pixels of a row.  Its slot is 64 wn + 32 t + (j / 2) + 16 (j % 2): the
// staging lane of pixels 4 i + u then writes slots consecutive in i.
template <int MODE, bool BIAS, bool TW>
__global__ __launch_bounds__(256, 3) void k_pw_gemm(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
    float* __restrict__ z, double2* __restrict__ part, int64_t K, int64_t M, int64_t HW,
    int64_t chunk, int64_t cpp, int64_t chunks, int mtiles) {
    __shared__ __attribute__((aligned(16))) char lds[kOperandA + kOperandB];
    __shared__ float shiftk[kGm];   // statistics: the item's shift of each row slot
    __shared__ float2 half[2][kGm]; // and its sums over each half of the columns
    static_assert(4 * 32 * kStatPitch * sizeof(float2) <= sizeof(lds), "statistics transpose");
    char* const opa = lds;
    char* const opb = lds + kOperandA;
    const int lane = threadIdx.x & 63;
    const int v = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int h = lane >> 5, j = lane & 31;
    const int wm = v >> 1, wn = v & 1;  // the wave's 32 rows and 64 columns
    int64_t gc;
    int mt;
    xcd_tile(blockIdx.x, (uint32_t)mtiles, &gc, &mt);
    if (gc >= chunks) return;  // whole block
    const int64_t n = gc / cpp, kc = gc - n * cpp;
    const int row0 = mt * kGm;
    const float* __restrict__ xn = x + n * K * HW;
    const Buffer bx = buffer_of(xn, K * HW), bw = buffer_of(w, M * K);
    const Buffer bz = buffer_of(z + n * M * HW, M * HW);
    const uint32_t hw = (uint32_t)HW;
    // row of the tile in row slot s (TW: the staging lane of rows 4 i + u
    // writes slots 16 u + i)
    auto slot_row = [&](int s) { return row0 + (TW ? 4 * (s & 15) + (s >> 4) : s); };
    const bool live = slot_row(32 * wm) < M;  // the wave has rows
    const int64_t px0 = kc * chunk, pend = min(px0 + chunk, HW);
    const bool wwhole = TW ? M % 4 == 0 || row0 + kGm <= M : K % 4 == 0;
    const int sc = 64 * wn + (j >> 1) + 16 * (j & 1);

    double run_n = 0.0, run_mean = 0.0, run_m2 = 0.0;  // of row slot threadIdx.x
    for (int64_t p0 = px0; p0 < pend; p0 += kGp) {
        f4 st[8];
        const bool xwhole = HW % 4 == 0 || p0 + kGp <= HW;
        auto gload = [&](int k0) {
            if (v < 2)
                load_cols(st, bx, hw, k0 + 8 * (2 * v + h), (uint32_t)p0 + 4 * j, xwhole);
            else if (v == 2 && TW)
                load_cols(st, bw, (uint32_t)M, k0 + 8 * (lane >> 4), row0 + 4 * (lane & 15),
                          wwhole);
            else if (v == 2)
                load_rows(st, bw, (uint32_t)K, row0 + (lane >> 2), k0 + 8 * (lane & 3),
                          (uint32_t)K, wwhole);
        };
        f16 acc[2], lo[2];
        clear(acc);
        clear(lo);
        gload(0);
        for (int k0 = 0; k0 < K; k0 += kGk) {
            lds_barrier();  // the stage is free
            if (v < 2)
                // columns 4 j + u: slots 64 (j / 16) + 32 (u & 1) + j % 16 + 16 (u / 2)
                stage_x(st, opb, 2 * v + h, 64 * (j >> 4) + (j & 15));
            else if (v == 2 && TW)
                stage_cols<kPlaneA>(st, opa, lane >> 4, lane & 15, 16);
            else if (v == 2)
                stage_rows<kPlaneA>(st, opa, lane & 3, lane >> 2);
            lds_barrier();  // and full
            if (k0 + kGk < K) gload(k0 + kGk);
            if (live) mma_step(acc, lo, opa, opb, 32 * wm + j, sc, h);
        }
        acc[0] += lo[0];
        acc[1] += lo[1];
        if (!any_nonfinite(acc)) {
            acc[0] *= kBf3Down;
            acc[1] *= kBf3Down;
        } else {
            // an infinity, NaN or large value: again on fp32 instructions
            clear(acc);
            const int64_t row = min<int64_t>(slot_row(32 * wm + j), M - 1);
            for (int64_t k = 0; k < K; k += 2) {
                const int64_t kk = k + h;
                const float a = kk < K ? (TW ? w[kk * M + row] : w[row * K + kk]) : 0.0f;
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const int64_t p = p0 + 64 * wn + 2 * j + t;
                    const float b = kk < K && p < HW ? xn[kk * HW + p] : 0.0f;
                    acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc[t], 0, 0, 0);
                }
            }
        }
        // ---- epilogue.  Rows past M fall outside the descriptor and are
        // dropped.  (The offsets are formed here, not hoisted out of the
        // item loop where 16 of them would stay live in registers.)
        const int64_t px = p0 + 64 * wn + 2 * j;
        const int nv = (int)max<int64_t>(0, min<int64_t>(2, HW - px));  // this lane's pixels
        uint32_t hw4 = 4u * hw;
        asm volatile("" : "+s"(hw4));
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = slot_row(32 * wm + mma_row(r) + 4 * h);
            if (BIAS) {
                const float b = bias[min<int64_t>(row, M - 1)];
                acc[0][r] += b;
                acc[1][r] += b;
            }
            const uint32_t o = (uint32_t)row * hw4 + 4u * (uint32_t)px;
            f2 o2 = {acc[0][r], acc[1][r]};
            if (nv == 2) {
                if (MODE == kGemmAccum)
                    o2 += __builtin_bit_cast(f2, __builtin_amdgcn_raw_buffer_load_b64(bz, o, 0, 0));
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, o2), bz, o, 0, 0);
            } else if (nv == 1) {
                if (MODE == kGemmAccum) o2[0] += load1(bz, o);
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, o2[0]), bz, o, 0, 0);
            }
        }
        if (MODE == kGemmStats) {
            // shift of each row: its value at the item's first pixel
            if (wn == 0 && j == 0) {
#pragma unroll
                for (int r = 0; r < 16; ++r) shiftk[32 * wm + mma_row(r) + 4 * h] = acc[0][r];
            }
            lds_barrier();  // every wave has read the stage; the shifts are there
            float2* sb = reinterpret_cast<float2*>(lds) + v * 32 * kStatPitch;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int s = mma_row(r) + 4 * h;
                const float s0 = shiftk[32 * wm + s];
                const float d0 = nv > 0 ? acc[0][r] - s0 : 0.0f;
                const float d1 = nv > 1 ? acc[1][r] - s0 : 0.0f;
                sb[s * kStatPitch + j] = make_float2(d0 + d1, fmaf(d1, d1, d0 * d0));
            }
            lds_barrier();
            // half h of the wave's 32 lane columns, for row slot 32 wm + j
            float S = 0.0f, Q = 0.0f;
            const float4* src = reinterpret_cast<const float4*>(sb + j * kStatPitch + 16 * h);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float4 u = src[i];
                S += u.x + u.z;
                Q += u.y + u.w;
            }
            S += __shfl_xor(S, 32);
            Q += __shfl_xor(Q, 32);
            if (h == 0) half[wn][32 * wm + j] = make_float2(S, Q);
            lds_barrier();
            if (threadIdx.x < kGm) {
                const float2 a = half[0][threadIdx.x], b = half[1][threadIdx.x];
                S = a.x + b.x;
                Q = a.y + b.y;
                const double cnt = (double)min<int64_t>(kGp, HW - p0);
                const double mean = (double)shiftk[threadIdx.x] + (double)S / cnt;
                const double m2 = fmax((double)Q - (double)S * (double)S / cnt, 0.0);
                // Chan's merge into the row's running moments
                const double tot = run_n + cnt, f = cnt / tot, d = mean - run_mean;
                run_m2 = run_n == 0.0 ? m2 : run_m2 + m2 + d * d * run_n * f;
                run_mean = run_n == 0.0 ? mean : run_mean + d * f;
                run_n = tot;
            }
        }
    }
    if (MODE == kGemmStats && threadIdx.x < kGm) {
        const int row = slot_row(threadIdx.x);
        if (row < M) part[(n * M + row) * cpp + kc] = make_double2(run_mean, run_m2);
    }
}

// dW partial of one pixel chunk: part_w[gb][co][ci] = sum_p dz[co][p]
// x[ci][p] over the chunk's pixels, and, from the blocks of the first ci
// tile, part_b[gb][co] = sum_p dz[co][p].  Tiles of 64 co x 128 ci; waves 0
// and 1 stage x, wave 2 dz.
__global__ __launch_bounds__(256, 3) void k_pw_gemm_wgrad(
    const float* __restrict__ dz, const float* __restrict__ x, float* __restrict__ part_w,
    float* __restrict__ part_b, int64_t C_in, int64_t C_out, int64_t HW, int64_t chunk,
    int64_t cpp, int64_t chunks, int tiles_ci, int tiles) {
    __shared__ __attribute__((aligned(16))) char lds[kOperandA + kOperandB];
    char* const opa = lds;
    char* const opb = lds + kOperandA;
    const int lane = threadIdx.x & 63;
    const int v = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int h = lane >> 5, j = lane & 31;
    const int wm = v >> 1, wn = v & 1;  // the wave's 32 rows and 64 columns
    int64_t gb;
    int tile;
    xcd_tile(blockIdx.x, (uint32_t)tiles, &gb, &tile);
    if (gb >= chunks) return;  // whole block
    const int64_t n = gb / cpp, kc = gb - n * cpp;
    const int64_t co0 = (int64_t)(tile / tiles_ci) * kGm, ci0 = (int64_t)(tile % tiles_ci) * kGp;
    const bool want_b = part_b != nullptr && ci0 == 0;
    const int64_t px0 = kc * chunk, pend = min(px0 + chunk, HW);
    const float* __restrict__ dzn = dz + n * C_out * HW;
    const float* __restrict__ xn = x + n * C_in * HW;
    const bool live = co0 + 32 * wm < C_out && ci0 + 64 * wn < C_in;
    const bool sdz = v == 2;
    const Buffer bs = buffer_of(sdz ? dzn : xn, (sdz ? C_out : C_in) * HW);
    const uint32_t r0 = (uint32_t)(sdz ? co0 : ci0 + 64 * v) + (lane >> 2);

    f4 st[8];
    auto gload = [&](int64_t p) {
        if (v < 3)
            load_rows(st, bs, (uint32_t)HW, r0, (uint32_t)p + 8 * (lane & 3), (uint32_t)pend,
                      pend % 4 == 0);
    };
    f16 acc[2], lo[2];
    clear(acc);
    clear(lo);
    float sb[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    gload(px0);
    for (int64_t p = px0; p < pend; p += kGk) {
        lds_barrier();  // the stage is free
        if (sdz) {
            stage_rows<kPlaneA>(st, opa, lane & 3, lane >> 2);
            if (want_b) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const f4 t = st[2 * e] + st[2 * e + 1];
                    sb[e] += (t[0] + t[1]) + (t[2] + t[3]);
                }
            }
        } else if (v < 2) {
            stage_rows<kPlaneB>(st, opb, lane & 3, 64 * v + (lane >> 2));
        }
        lds_barrier();  // and full
        if (p + kGk < pend) gload(p + kGk);
        if (live) mma_step(acc, lo, opa, opb, 32 * wm + j, 64 * wn + j, h);
    }
    acc[0] += lo[0];
    acc[1] += lo[1];
    if (!any_nonfinite(acc)) {
        acc[0] *= kBf3Down;
        acc[1] *= kBf3Down;
    } else {
        // an infinity, NaN or large value: again on fp32 instructions
        clear(acc);
        for (int64_t p = px0; p < pend; p += 2) {
            const int64_t pp = p + h;
            const float a = pp < pend ? dzn[min(co0 + 32 * wm + j, C_out - 1) * HW + pp] : 0.0f;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const float b =
                    pp < pend ? xn[min(ci0 + 64 * wn + 32 * t + j, C_in - 1) * HW + pp] : 0.0f;
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc[t], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int64_t co = co0 + 32 * wm + mma_row(r) + 4 * h;
            const int64_t ci = ci0 + 64 * wn + 32 * t + j;
            if (co < C_out && ci < C_in) part_w[(gb * C_out + co) * C_in + ci] = acc[t][r];
        }
    if (want_b && sdz) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float t = sb[e];
            t += __shfl_xor(t, 2);
            t += __shfl_xor(t, 1);
            const int64_t co = co0 + (lane >> 2) + 16 * e;
            if ((lane & 3) == 0 && co < C_out) part_b[gb * C_out + co] = t;
        }
    }
}

template <typename F>
void bsel(bool b, F&& f) {
    if (b)
        f(std::true_type{});
    else
        f(std::false_type{});
}

}  // namespace

// Byte offsets inside a sample's planes and inside W, tiles past their ends
// included, stay below 2^31; the grid too.
static bool gemm_fits(int64_t N, int64_t K, int64_t M, int64_t HW) {
    const int64_t lim = (int64_t)1 << 29;  // floats
    if (K > lim || M > lim || HW > lim || N > lim) return false;
    const int64_t k = K + kGp, m = M + kGp;
    return m <= lim / k && m <= lim / (HW + kGp) && k <= lim / (HW + kGp) &&
           N * ((HW + 31) / 32 + 8) < lim / (m / kGm + 1) / (k / kGm + 1);
}

// From 48 rows and 48 channels on the tile pays at every plane size (one
// sample; fused forward / input gradient, here against k_pw_conv: 48 -> 96
// channels at 16384 pixels 19.0 / 11.1 against 23.3 / 14.6 us, 128 -> 256
// at 65536 pixels 68.9 / 34.5 against 75.0 / 52.5 us, at 2^20 pixels 961 /
// 519 against 1453 / 747 us; 64 -> 64 at 2^20 pixels 215 against 217 us).
// A block walks all of K at about 1.3 us per step of 32 when it has a CU to
// itself, so a grid of few tiles and a deep K stays with the kernels that
// split K (512 -> 256 at 1024 pixels, 32 tiles: 31.4 here, 20.2 us there;
// 256 -> 128 at 4096, 64 tiles: 22.4 and 21.6 us; 512 -> 256 at 4096, 128
// tiles: 34.1 and 37.8 us).
static int64_t gemm_tiles(int64_t N, int64_t M, int64_t HW) {
    return N * ((HW + kGp - 1) / kGp) * ((M + kGm - 1) / kGm);
}

bool pw_gemm_use(int64_t N, int64_t K, int64_t M, int64_t HW) {
    if (M < 48 || K < 48 || !gemm_fits(N, K, M, HW)) return false;
    const int64_t tiles = gemm_tiles(N, M, HW);
    return tiles >= 32 && K <= 4 * tiles;
}

// Whether k_pw_small, within its own limit, is still faster.  Its time goes
// with the multiply-adds; here a tile that is partly filled (a plane of fewer
// than 128 pixels) takes as long as a full one, and the time goes with the K
// steps and, beyond about two blocks per CU, with the tiles.  us, k_pw_small /
// here: 512 -> 512 channels, 32 samples of 1 pixel 7.1 / 30.1; 256 -> 256, 16
// of 4 3.5 / 13.6; 64 -> 64, 32 of 49 4.5 / 7.0; 128 -> 128, 16 of 64 6.3 /
// 8.5 and 32 of 49 (2^24.6 multiply-adds) 11.2 / 10.2; 256 -> 256, 128 of 4
// 10.2 / 14; input gradients 192 <- 384, 48 of 9 20 / 16, 512 <- 512, 128 of 1
// 11 / 74.  Over 700 calls of at most 2^25 multiply-adds the line's choice
// takes 0.3% longer than the faster one on average and 20% at most; the tile
// everywhere 58%, at most 6.8 times as long.  `norm`: a GroupNorm of small
// units follows, which takes one launch over z but two on the tile's
// statistics (16 x 64 -> 64 at 16 x 16: 10.2 / 11.4, without it 6.2 / 6.0).
bool pw_gemm_loses(int64_t N, int64_t K, int64_t M, int64_t HW, bool norm) {
    const double steps = (double)((K + kGk - 1) / kGk);
    const double waves = std::max(1.0, (double)gemm_tiles(N, M, HW) / 512.0);
    const double macs = (double)N * (double)K * (double)M * (double)HW;
    return macs <= ((norm ? 11.0 : 7.0) + 3.5 * steps * waves) * 1048576.0;
}

// 192 -> 384 channels at 128^2 pixels: forward with statistics 49.5 -> 23.9
// us, input gradient 44.8 + 4.4 (transpose of W) -> 26.5 us.
hipError_t launch_pw_gemm(const PwArgs& a, int64_t N, int64_t K, int64_t M, int64_t HW,
                          int64_t chunk, double2* part, bool accumulate, bool trans,
                          hipStream_t s) {
    const int64_t cpp = (HW + chunk - 1) / chunk, chunks = N * cpp;
    const int mtiles = (int)((M + kGm - 1) / kGm);
    const dim3 grid((unsigned)((chunks + 7) / 8 * 8 * mtiles));
    auto go = [&](auto MD, auto B, auto T) {
        k_pw_gemm<MD(), B(), T()><<<grid, 256, 0, s>>>(a.x, a.w, a.bias, a.z, part, K, M, HW, chunk,
                                                       cpp, chunks, mtiles);
    };
    using F = std::false_type;
    using P = std::integral_constant<int, kGemmPlain>;
    if (trans) {
        bsel(accumulate, [&](auto A) {
            go(std::integral_constant<int, A() ? kGemmAccum : kGemmPlain>{}, F{}, std::true_type{});
        });
    } else if (accumulate) {
        return hipErrorInvalidValue;  // only input gradients are added
    } else {
        bsel(a.bias != nullptr, [&](auto B) {
            if (part)
                go(std::integral_constant<int, kGemmStats>{}, B, F{});
            else
                go(P{}, B, F{});
        });
    }
    return hipGetLastError();
}

// Against k_pw_wgrad (with its finish; one sample): 48 -> 96 channels at
// 65536 pixels 21.4 against 23.4 us, 64 -> 64 at 2^18 35.0 / 38.1, 128 ->
// 256 at 65536 40.0 / 57.4, at 2^18 149 / 187; at 2^20, where the rows of a
// step, a power of two apart, meet few memory channels and k_pw_wgrad's
// longer runs per row pay, 787 / 734 and 64 -> 64 190 / 117.
bool pw_gemm_wgrad_use(int64_t N, int64_t C_in, int64_t C_out, int64_t HW) {
    return C_in >= 48 && C_out >= 48 && HW <= (int64_t)1 << 18 && gemm_fits(N, C_in, C_out, HW);
}

// Pixels per chunk, for about 768 blocks (three per CU; at 384 x 192 over
// 16384 pixels 512 / 768 / 1024 blocks took 32.1 / 26.0 / 30.3 us), at least
// four steps each.
int64_t pw_gemm_wgrad_chunk(int64_t N, int64_t C_in, int64_t C_out, int64_t HW) {
    const int64_t tiles = ((C_out + kGm - 1) / kGm) * ((C_in + kGp - 1) / kGp);
    int64_t c = (N * HW * tiles / 768 + kGk - 1) / kGk * kGk;
    c = std::max<int64_t>(c, 4 * kGk);
    return std::min(c, (HW + kGk - 1) / kGk * kGk);
}

hipError_t launch_pw_gemm_wgrad(const float* dz, const float* x, float* part_w, float* part_b,
                                int64_t N, int64_t C_in, int64_t C_out, int64_t HW, int64_t chunk,
                                hipStream_t s) {
    const int64_t cpp = (HW + chunk - 1) / chunk, chunks = N * cpp;
    const int tco = (int)((C_out + kGm - 1) / kGm), tci = (int)((C_in + kGp - 1) / kGp);
    const dim3 grid((unsigned)((chunks + 7) / 8 * 8 * tco * tci));
    k_pw_gemm_wgrad<<<grid, 256, 0, s>>>(dz, x, part_w, part_b, C_in, C_out, HW, chunk, cpp, chunks,
                                         tci, tco * tci);
    return hipGetLastError();
}

}  // namespace gn
}  // namespace soar
