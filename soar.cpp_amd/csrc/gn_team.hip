// gn_team.hip - GroupNorm(+SiLU) of large tensors with every unit kept on
// chip between its two passes.
//
// The two-launch path reads a unit twice (statistics, then apply; reduction,
// then dx): 3 tensor passes forward and 5 backward, each at the rate of the
// memory.  Here a team of blocks owns a unit: every block loads its share
// once, reduces it to the chunk partials of the two-launch path, publishes
// them, waits for the team's other partials, finishes the unit's sums itself
// and writes y (dx) from what it holds: 2 tensor passes forward, 3 backward.
//
// What bounds it: memory, in phases.  A team loads, waits and stores, and
// while it waits only the next team's blocks load; a copy from registers in
// such phases takes 375-390 us per 2 GiB moved, a streaming copy 332.  So
// teams are kept small against the chip (several in flight).  Measured with
// SiLU, two launches -> one, forward; backward, us:
//   48 x 512^2, 8 groups         30.6 -> 23.0; 45.7 -> 37.0
//   64 x 512^2, 16               36.6 -> 27.1; 57.6 -> 43.9
//   16 x 1024^2, 8               37.5 -> 27.0; 56.9 -> 45.1
//   24 x 1024^2, 4               52.2 -> 36.9; (too large)
//   32 x 1024^2, 8               65.9 -> 51.5; (too large)
//   2 x 64 x 1024^2, 32          246 -> 191;   406 -> 330
//   2 x 128 x 1024^2, 32, +x     483 -> 386;   (too large)
// Held on chip per block: 512 threads at 128 VGPRs, two blocks per CU, so 64
// floats of x per thread in registers and 32 more in LDS forward, 32 of x and
// 32 of dy backward.  (Backward with a further chunk in LDS gained 4% and
// needed the whole chip to itself; reading x again instead of holding it was
// slower than two launches.)
//
// Every chunk (8192 floats of a plane, 256 threads of 8 vectors) and output
// uses the arithmetic of k_stats / k_apply / k_bwd_reduce / k_bwd_dx in the
// same order.  The finishes add the chunks' partials lane by lane (thread by
// thread) and then the lanes by a tree; a block takes the chunks of whole
// lanes ("items") and publishes the lanes' sums, at most a few hundred per
// unit.  So the sums are the two-launch path's up to the order of their
// float64 additions.  (The forward's moments are taken about the unit's first
// value and not about its first partial's mean, which no other block knows.)
//
// Hand-off.  A sum is two 64-bit words in a slot that the launch before
// (k_team_clear) set to all ones, a NaN that no partial is (publish maps it to
// another).  Words are written and read with relaxed atomics of device scope,
// which go past the XCDs' private caches; a reader needs no flag and no fence,
// since it takes a slot's words as they turn valid.
//
// Every wait ends.  The blocks of a team are consecutive, so they normally
// run together; but nothing guarantees it (kernels of other streams, fewer
// CUs).  A block that has waited `limit` clock ticks leaves its share
// unwritten, with a mark on the unit.  It has published its own sums, so the
// launch after (k_team_fwd_rest / k_team_bwd_rest) finds all sums of a marked
// unit in the slots, reads the unit again and writes it, the second pass of
// two launches; the bits are the same.  No loop ends by another block's
// store, and once a block of the call has left, the others do not wait
// either: a call that meets other work costs its limit once (with every
// block leaving, forward; backward: 64 x 512^2 55.8; 88.9 us, 32 x 1024^2
// forward 96).  A marked unit is read after blocks of it wrote theirs, which
// is why outputs that overlap inputs take the two launches.  Where nothing is
// marked the launch ends at once (1.2 us).
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "gn_internal.hpp"
#include "gn_math.hpp"
#include "gn_moments.hpp"
#include "soar_gn.h"

// Lambdas that take a chunk's registers are always inlined: a call would put
// them in memory.
#define SOAR_INLINE __attribute__((always_inline))

namespace soar {
namespace gn {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned long long u64;

constexpr int kTeamThreads = 512;
constexpr int kHalf = 256;     // threads of a half-block, which walks whole chunks
constexpr int kVec = 8;        // vectors of a chunk per thread
constexpr int kTeamChunk = 4 * kVec * kHalf;  // 8192 floats
constexpr int kMaxCpg = 128;                  // channels per unit
// Blocks of a team: a quarter of the 512 that 256 CUs hold.  Calls of other
// streams take their part of every CU, and a team that is only partly there
// waits for its limit; the part that is left for it must hold it.  Two streams
// of the same calls, us a pair, in two launches -> with teams of 128; 192;
// 256; 342 blocks (a limit of 50-100 us): 1012 -> 861 (forward, 2 x 128 x
// 1024^2), 100 -> 91 (backward, 16 x 1024^2); 149 -> 151; 206 -> 317 and 1629
// -> 2755 (backward, 32 and 2 x 128 x 1024^2; alone such a team gains 10%).
// Three streams: 0.92-0.99 of two launches' time at 128, 1.4 at 192; four up
// to 1.2 at 128, since blocks then leave.
constexpr int kMaxTeam = 128;
// Chunks of the tensor, forward (48 MB) and backward (24 MB).  Below, both
// ways live in the caches and the launches decide, of which this way has one
// more each way (three, at 2.4 us each for the host) and dgamma's with several
// samples.  Two launches -> one, us, replayed from a graph and called one by
// one: forward of 768 chunks 18.0 -> 15.3 and 18.9 -> 21.7, 1024 21.3 -> 17.8
// and 21.7 -> 20.6 (two streams 38.4 -> 42.2), 1536 30.6 -> 23.0; backward of
// 768 27.6 -> 20.5, 1024 33.8 -> 23.8.
constexpr int64_t kTeamMinFwd = 1536, kTeamMinBwd = 768;
// Chunks up to which a backward with residual and SiLU comes here (64 MB): its
// dy stays held and the SiLU's derivative is formed again after the wait.  Two
// launches -> one, us: 64 x 512^2 57.9 -> 43.7; larger, with more spilled
// registers than now, 64 x 1024^2 203 -> 206, 2 x 128 x 1024^2 812 -> 830.
// (gamma r dz + dy in dy's place instead: 73 spilled registers, 1199.)
constexpr int64_t kTeamMaxResChunks = 2048;
constexpr u64 kUnset = ~0ull;

__device__ __forceinline__ u64 load_word(const u64* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void publish(u64* slot, double a, double b) {
    u64 wa = __builtin_bit_cast(u64, a), wb = __builtin_bit_cast(u64, b);
    if (wa == kUnset) wa = 0x7ff8000000000000ull;
    if (wb == kUnset) wb = 0x7ff8000000000000ull;
    __hip_atomic_store(slot, wa, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(slot + 1, wb, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ __launch_bounds__(256) void k_team_clear(TeamWs w, int64_t words, int64_t units) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < words) w.slots[i] = kUnset;
    if (i < units) w.left[i] = 0;  // (a unit has at least two words)
    if (i == 0) *w.any = 0;
}

// Marks of a unit's blocks that left: some block, its first block.
constexpr unsigned kLeft = 1, kLeftFirst = 2;

// A block leaves (thread 0).
__device__ __forceinline__ void team_leave(const TeamWs& w, int64_t u, int kb) {
    __hip_atomic_fetch_or(w.left + u, kb == 0 ? kLeft | kLeftFirst : kLeft, __ATOMIC_RELAXED,
                          __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(w.any, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Geometry of a team launch.  Item `it` of a unit is the chunks that lane
// r = it % lanes of span it / lanes adds: r, r + lanes, ... of the span's
// chunks (forward: one span, the unit; backward: a span per plane).
struct Team {
    int64_t C, G, HW;
    int cpg, cpp, P;      // channels per unit, chunks per plane and per unit
    int span, lanes, nq;  // chunks of a span, its lanes, chunks of a lane (at most)
    int items, ipb;       // of a unit, of a block
    int blocks;           // per unit
    u64 limit;            // clock ticks (100 MHz) a block waits for the others
    int leave;            // every block leaves
};

// Chunk number of item it's i-th chunk, or -1.
__device__ __forceinline__ int item_chunk(const Team& g, int it, int i) {
    const int sp = it / g.lanes, c = it - sp * g.lanes + i * g.lanes;
    return it < g.items && c < g.span ? sp * g.span + c : -1;
}

// Chunk c of unit u: its plane, first element and length (0 for c < 0).
struct TeamChunk {
    int64_t plane, base;
    int len;
};
__device__ __forceinline__ TeamChunk team_chunk(const Team& g, int64_t u, int c) {
    const int c0 = max(c, 0), pl = c0 / g.cpp, k = c0 - pl * g.cpp;
    TeamChunk r;
    r.plane = u * g.cpg + pl;
    r.base = r.plane * g.HW + (int64_t)k * kTeamChunk;
    r.len = c < 0 ? 0 : (int)min<int64_t>(kTeamChunk, g.HW - (int64_t)k * kTeamChunk);
    return r;
}

// A chunk's vectors, thread t's at t, t + 256, ...: through a raw buffer
// descriptor of the chunk, so vectors past its end (all of them for a chunk
// that is not there) load zeros and store nothing, without a branch.
__device__ __forceinline__ auto chunk_buffer(const float* x, const TeamChunk& c) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x + c.base), (short)0, 4 * c.len,
                                             0x00020000);
}
constexpr int kNonTemporal = 2;  // cache policy bit of the buffer accesses

__device__ __forceinline__ void load_chunk(f4 (&v)[kVec], const float* __restrict__ x,
                                           const TeamChunk& c, int t) {
    const auto rs = chunk_buffer(x, c);
#pragma unroll
    for (int k = 0; k < kVec; ++k)
        v[k] = __builtin_bit_cast(
            f4, __builtin_amdgcn_raw_buffer_load_b128(rs, 16 * (t + k * kHalf), 0,
                                                      kNonTemporal));
}

__device__ __forceinline__ void store_vec(f4 o, float* __restrict__ y, const TeamChunk& c, int i) {
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, o), chunk_buffer(y, c), 16 * i, 0,
                                           kNonTemporal);
}

// The value of slot `it` once it is set; false when the limit passes first or
// another block of the call has left (wave-uniform).  A wait costs one round
// trip past the caches per look.  (With a slot per chunk, 2048 per 64 MB unit,
// the looks of 256 blocks were 19 MB each and a unit waited 7 us.  16-byte
// loads with the scope bits of a volatile buffer load, sc0 sc1, kept returning
// old words; these are sc1.)
__device__ __forceinline__ bool poll(double2& v, const u64* __restrict__ slots, int it,
                                     const Team& g, const TeamWs& w, u64 t0) {
    const u64* s = slots + 2 * min(it, g.items - 1);
    for (;;) {
        const u64 a = load_word(s), b = load_word(s + 1);
        v = make_double2(__builtin_bit_cast(double, a), __builtin_bit_cast(double, b));
        if (!__any(a == kUnset || b == kUnset)) return true;
        const bool others = __builtin_amdgcn_readfirstlane((int)load_word(w.any)) != 0;
        if (others || __builtin_amdgcn_s_memrealtime() - t0 > g.limit) return false;
        __builtin_amdgcn_s_sleep(2);
    }
}
// The same after the launch that set it.
__device__ __forceinline__ double2 read_slot(const u64* __restrict__ slots, int it, const Team& g) {
    const u64* s = slots + 2 * min(it, g.items - 1);
    return make_double2(__builtin_bit_cast(double, s[0]), __builtin_bit_cast(double, s[1]));
}

// Chunk m of block kb: chunk m % nq of its item m / nq (-1: none).
__device__ __forceinline__ int block_chunk(const Team& g, int kb, int m) {
    const int o = m / g.nq;
    return o < g.ipb ? item_chunk(g, kb * g.ipb + o, m - o * g.nq) : -1;
}

// ---- forward -----------------------------------------------------------------

// k_stats' sums of a chunk, for a thread of 256: shift K, sums, count.
struct ChunkSums {
    float K, s, q;
    int cnt;
};
__device__ __forceinline__ ChunkSums chunk_sums(const f4 (&v)[kVec], int len, int t) {
    ChunkSums r;
    r.K = v[0].x;
    const int n4 = len >> 2;
    r.cnt = t < n4 ? 4 * ((n4 - 1 - t) / kHalf + 1) : 0;
    float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f, q0 = 0.f, q1 = 0.f, q2 = 0.f, q3 = 0.f;
    // (a vector past the chunk's end counts as K: it adds zeros)
    const bool whole = len == kTeamChunk;
#pragma unroll
    for (int k = 0; k < kVec; ++k) {
        f4 x = v[k];
        if (!whole && 4 * k >= r.cnt) x = f4{r.K, r.K, r.K, r.K};
        const float d0 = x.x - r.K, d1 = x.y - r.K, d2 = x.z - r.K, d3 = x.w - r.K;
        s0 += d0;
        s1 += d1;
        s2 += d2;
        s3 += d3;
        q0 = fmaf(d0, d0, q0);
        q1 = fmaf(d1, d1, q1);
        q2 = fmaf(d2, d2, q2);
        q3 = fmaf(d3, d3, q3);
    }
    r.s = (s0 + s1) + (s2 + s3);
    r.q = (q0 + q1) + (q2 + q3);
    return r;
}

// The unit's sums over its items, by half-block 0 (thread t of it) into sums:
// get(it, p): item it's sums, false if they are not there.
template <typename F>
__device__ __forceinline__ void gather_fwd(const Team& g, int t, double2* sums, int* late, F get) {
    double2 v = make_double2(0.0, 0.0);
    for (int it = t; it - t < g.items; it += kHalf) {
        double2 p;
        if (!get(it, p)) *late = 1;
        if (it < g.items) {
            v.x += p.x;
            v.y += p.y;
        }
    }
    v.x = wave_sum(v.x);
    v.y = wave_sum(v.y);
    if ((t & 63) == 0) sums[t >> 6] = v;
}

// Mean, rstd and the mean's low part from them, into bc (thread 0); R: the
// moments' reference.
__device__ __forceinline__ void finish_fwd(const Team& g, const double2* sums, double R, float eps,
                                           int64_t u, bool first, float* __restrict__ mean,
                                           float* __restrict__ rstd, float* __restrict__ mean_lo,
                                           float* bc) {
    double S = sums[0].x, Q = sums[0].y;
#pragma unroll
    for (int i = 1; i < kHalf / 64; ++i) {
        S += sums[i].x;
        Q += sums[i].y;
    }
    const double n = (double)(g.cpg * g.HW);
    const double2 mm = centred_moments(S, Q, n, R);
    const double var = mm.y / n;
    const float hi = (float)mm.x, lo = (float)(mm.x - (double)hi);
    const float r = (float)(1.0 / sqrt(var + (double)eps));
    bc[0] = hi;
    bc[1] = r;
    bc[2] = lo;
    if (first) {
        mean[u] = hi;
        rstd[u] = r;
        if (mean_lo) mean_lo[u] = lo;
    }
}

// k_apply of a chunk that is held.
template <bool SILU, bool RES>
__device__ __forceinline__ void apply_chunk(const f4 (&d)[kVec], const Team& g, const TeamChunk& ck,
                                            const float* __restrict__ gamma,
                                            const float* __restrict__ beta, const float* bc,
                                            float* __restrict__ y, int t) {
    const float mu = bc[0], rs = bc[1], e = -bc[2] * rs;
    const int64_t ch = ck.plane % g.C;
    const float gm = gamma ? gamma[ch] : 1.0f;
    const float a = gm * rs, b = fmaf(gm, e, beta ? beta[ch] : 0.0f);
#pragma unroll
    for (int k = 0; k < kVec; ++k) {
        f4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float z = fmaf(d[k][i] - mu, a, b);
            o[i] = SILU ? silu_fast(z) : z;
            if (RES) o[i] += d[k][i];
        }
        store_vec(o, y, ck, t + k * kHalf);
    }
}

// NR chunks per half-block in registers (32 VGPRs each), NL in LDS (64 KB
// for both half-blocks); RES: y += x.
template <int NR, int NL, bool SILU, bool RES>
__global__ __launch_bounds__(kTeamThreads, 4) void k_team_fwd(
    const float* __restrict__ x, const float* __restrict__ gamma, const float* __restrict__ beta,
    float* __restrict__ y, float* __restrict__ mean, float* __restrict__ rstd,
    float* __restrict__ mean_lo, TeamWs ws, Team g, float eps) {
    constexpr int NQ = NR + NL;  // chunks per half-block
    static_assert(NL <= 1 && NR >= 1, "at most one LDS chunk per half-block");
    __shared__ f4 hold[NL > 0 ? NL * 2 * kVec * kHalf : 1];
    __shared__ double mom[2 * NQ][16];  // (n, S, Q, Rw) x 4 waves of each chunk
    __shared__ double2 cm[2 * NQ];      // and its (mean, M2)
    __shared__ double2 sums[kHalf / 64];
    __shared__ float bc[3];
    __shared__ int late;
    const int hb = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8);  // half-block
    const int t = threadIdx.x & (kHalf - 1), w = t >> 6;
    const int64_t u = blockIdx.x / (unsigned)g.blocks;
    const int kb = (int)(blockIdx.x - (unsigned)u * g.blocks);
    u64* __restrict__ slots = ws.slots + 2 * u * g.items;
    auto chunk_no = [&](int q) { return block_chunk(g, kb, 2 * q + hb); };
    const double R = (double)x[u * g.cpg * g.HW];  // the moments' reference
    // an item's sums about R from its chunks' moments, in order (finish_unit)
    auto add_chunk = [&](double2& s, const double2& m, int c) {
        const int k = c % g.cpp;
        const double n = (double)min<int64_t>(kTeamChunk, g.HW - (int64_t)k * kTeamChunk);
        const double d = m.x - R, nd = n * d;
        s.x += nd;
        s.y += fma(nd, d, m.y);
    };
    auto sum_chunk = [&](const f4 (&v)[kVec], int q, int len) SOAR_INLINE {
        const ChunkSums r = chunk_sums(v, len, t);
        wave_moments(r.K, r.s, r.q, r.cnt, &mom[2 * q + hb][w], 4);
    };

    f4 v[NR][kVec];
    auto load_q = [&](f4 (&r)[kVec], int q) SOAR_INLINE {
        load_chunk(r, x, team_chunk(g, u, chunk_no(q)), t);
    };
    if constexpr (NL > 0) {
        // (the last register chunk waits for the LDS chunk's registers)
        f4 l[kVec];
        load_q(l, 0);
#pragma unroll
        for (int i = 0; i < NR - 1; ++i) load_q(v[i], NL + i);
        __builtin_amdgcn_sched_barrier(0);
        sum_chunk(l, 0, team_chunk(g, u, chunk_no(0)).len);
#pragma unroll
        for (int k = 0; k < kVec; ++k) hold[(hb * kVec + k) * kHalf + t] = l[k];
        __builtin_amdgcn_sched_barrier(0);
        load_q(v[NR - 1], NL + NR - 1);
    } else {
#pragma unroll
        for (int i = 0; i < NR; ++i) load_q(v[i], i);
    }
#pragma unroll
    for (int i = 0; i < NR; ++i)
        sum_chunk(v[i], NL + i, team_chunk(g, u, chunk_no(NL + i)).len);
    lds_barrier();
    if (threadIdx.x < 2 * NQ) cm[threadIdx.x] = combine_wave_moments<4>(mom[threadIdx.x], 4);
    lds_barrier();
    if ((int)threadIdx.x < g.ipb && kb * g.ipb + (int)threadIdx.x < g.items) {
        double2 s = make_double2(0.0, 0.0);
        for (int i = 0; i < g.nq; ++i) {
            const int m = threadIdx.x * g.nq + i, c = block_chunk(g, kb, m);
            if (c >= 0) add_chunk(s, cm[m], c);
        }
        publish(slots + 2 * (kb * g.ipb + threadIdx.x), s.x, s.y);
    }
    if (threadIdx.x == 0) late = g.leave;
    lds_barrier();
    if (hb == 0 && !g.leave) {
        const u64 t0 = __builtin_amdgcn_s_memrealtime();
        gather_fwd(g, t, sums, &late,
                   [&](int it, double2& p) { return poll(p, slots, it, g, ws, t0); });
    }
    lds_barrier();
    if (late) {
        if (threadIdx.x == 0) team_leave(ws, u, kb);
        return;  // whole block
    }
    if (threadIdx.x == 0) finish_fwd(g, sums, R, eps, u, kb == 0, mean, rstd, mean_lo, bc);
    lds_barrier();
    auto apply = [&](const f4 (&d)[kVec], int c) SOAR_INLINE {
        apply_chunk<SILU, RES>(d, g, team_chunk(g, u, c), gamma, beta, bc, y, t);
    };
#pragma unroll
    for (int i = 0; i < NR; ++i) apply(v[i], chunk_no(NL + i));
    if constexpr (NL > 0) {
        f4 l[kVec];
#pragma unroll
        for (int k = 0; k < kVec; ++k) l[k] = hold[(hb * kVec + k) * kHalf + t];
        apply(l, chunk_no(0));
    }
}

// The units that blocks left: `blocks` as k_team_fwd's, 2 depth chunks each.
template <bool SILU, bool RES>
__global__ __launch_bounds__(kTeamThreads) void k_team_fwd_rest(
    const float* __restrict__ x, const float* __restrict__ gamma, const float* __restrict__ beta,
    float* __restrict__ y, float* __restrict__ mean, float* __restrict__ rstd,
    float* __restrict__ mean_lo, TeamWs ws, Team g, float eps, int64_t blocks, int depth) {
    __shared__ double2 sums[kHalf / 64];
    __shared__ float bc[3];
    if (*ws.any == 0) return;
    const int hb = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8);
    const int t = threadIdx.x & (kHalf - 1);
    for (int64_t b = blockIdx.x; b < blocks; b += gridDim.x) {
        const int64_t u = b / g.blocks;
        const int kb = (int)(b - u * g.blocks);
        if (ws.left[u] == 0) continue;
        const u64* __restrict__ slots = ws.slots + 2 * u * g.items;
        int late;
        if (hb == 0)
            gather_fwd(g, t, sums, &late, [&](int it, double2& p) {
                p = read_slot(slots, it, g);
                return true;
            });
        lds_barrier();
        if (threadIdx.x == 0)
            finish_fwd(g, sums, (double)x[u * g.cpg * g.HW], eps, u, kb == 0, mean, rstd, mean_lo,
                       bc);
        lds_barrier();
        for (int q = 0; q < depth; ++q) {
            const TeamChunk ck = team_chunk(g, u, block_chunk(g, kb, 2 * q + hb));
            f4 v[kVec];
            load_chunk(v, x, ck, t);
            apply_chunk<SILU, RES>(v, g, ck, gamma, beta, bc, y, t);
        }
        lds_barrier();  // sums and bc are free
    }
}

// ---- backward ----------------------------------------------------------------

// k_bwd_reduce's sums of a chunk for a thread of 256; with KEEP the dz
// replace the dy.  (A vector past the chunk's end has dy = 0 and adds zeros.)
struct BwdCoef {
    float mu, r, e, gm, bt;
};
template <bool SILU, bool KEEP>
__device__ __forceinline__ void add_bwd_vec(const f4& x, f4& dy, const BwdCoef& k, float (&sa)[2],
                                            float (&sb)[2]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float xh = fmaf(x[i] - k.mu, k.r, k.e);
        const float dz = SILU ? dsilu_fast(dy[i], fmaf(k.gm, xh, k.bt)) : dy[i];
        sa[i & 1] += dz;
        sb[i & 1] = fmaf(dz, xh, sb[i & 1]);
        if (KEEP) dy[i] = dz;
    }
}
template <bool SILU, bool KEEP>
__device__ __forceinline__ float2 chunk_bwd_sums(const f4 (&v)[kVec], f4 (&dy)[kVec],
                                                 const BwdCoef& k) {
    float sa[2] = {0.f, 0.f}, sb[2] = {0.f, 0.f};
#pragma unroll
    for (int q = 0; q < kVec; ++q) {
        add_bwd_vec<SILU, KEEP>(v[q], dy[q], k, sa, sb);
        if (q % 2 == 1)  // (or the vectors' work is interleaved and spills)
            __builtin_amdgcn_sched_barrier(0);
    }
    return make_float2(sa[0] + sa[1], sb[0] + sb[1]);
}

// finish_bwd_unit's sums by half-block 0 (thread t of it): groups of lanes, a
// plane each, into gsum, and the planes' own into psum (when `planes`).
// get(it, v) as in gather_fwd.
template <typename F>
__device__ __forceinline__ void gather_bwd(const Team& g, int t, int64_t u, bool planes,
                                           const float* __restrict__ gamma, double2* gsum,
                                           double2* psum, int* late, F get) {
    const int gs = bwd_plane_lanes(g.lanes), ngroups = kHalf / gs;
    const int grp = t / gs, rr = t & (gs - 1);
    double S1 = 0.0, S2 = 0.0;
    for (int j = grp; j - grp < g.cpg; j += ngroups) {
        const bool mine = j < g.cpg;
        double A = 0.0, B = 0.0;
        for (int q = rr; q - rr < g.lanes; q += gs) {
            double2 v;
            if (!get(j * g.lanes + min(q, g.lanes - 1), v)) *late = 1;
            if (mine && q < g.lanes) {
                A += v.x;
                B += v.y;
            }
        }
        for (int off = gs >> 1; off > 0; off >>= 1) {
            A += __shfl_xor(A, off);
            B += __shfl_xor(B, off);
        }
        if (mine && rr == 0) {
            const int64_t ch = (u * g.cpg + j) % g.C;
            if (planes) psum[j] = make_double2(A, B);
            const double gj = gamma ? (double)gamma[ch] : 1.0;
            S1 += gj * A;
            S2 += gj * B;
        }
    }
    if (rr == 0) gsum[grp] = make_double2(S1, S2);
}

// The planes' sums (the unit's first block): to plane_sums, or, with one
// sample, k_param_finish's additions.
__device__ __forceinline__ void give_planes(const Team& g, int64_t u, const double2* psum,
                                            double2* __restrict__ plane_sums,
                                            float* __restrict__ dgamma, float* __restrict__ dbeta) {
    for (int j = threadIdx.x; j < g.cpg; j += kTeamThreads) {
        const int64_t plane = u * g.cpg + j, ch = plane % g.C;
        const double2 s = psum[j];
        if (plane_sums) {
            plane_sums[plane] = s;
        } else {
            if (dbeta) dbeta[ch] = (float)((double)dbeta[ch] + s.x);
            if (dgamma) dgamma[ch] = (float)((double)dgamma[ch] + s.y);
        }
    }
}

// dx's two unit coefficients, into bc (thread 0).
__device__ __forceinline__ void finish_bwd(const Team& g, const double2* gsum, float r, float* bc) {
    const int ngroups = kHalf / bwd_plane_lanes(g.lanes);
    double s1 = 0.0, s2 = 0.0;
    for (int i = 0; i < ngroups; ++i) {
        s1 += gsum[i].x;
        s2 += gsum[i].y;
    }
    const double Md = (double)(g.cpg * g.HW);
    bc[0] = (float)(-(double)r * s1 / Md);
    bc[1] = (float)(-(double)r * s2 / Md);
}

// k_bwd_dx of a chunk that is held; DZ: d holds dz.
template <bool SILU, bool RES, bool DZ>
__device__ __forceinline__ void dx_chunk(const f4 (&v)[kVec], const f4 (&d)[kVec],
                                         const TeamChunk& ck, const BwdCoef& k, const float* bc,
                                         float* __restrict__ dx, int t) {
    const float B = bc[0], D = bc[1];
    const float A = k.gm * k.r;
#pragma unroll
    for (int q = 0; q < kVec; ++q) {
        f4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float xh = fmaf(v[q][i] - k.mu, k.r, k.e);
            const float dz = SILU && !DZ ? dsilu_fast(d[q][i], fmaf(k.gm, xh, k.bt)) : d[q][i];
            o[i] = fmaf(A, dz, fmaf(D, xh, B));
            if (RES) o[i] += d[q][i];
        }
        store_vec(o, dx, ck, t + q * kHalf);
        if (q % 2 == 1) __builtin_amdgcn_sched_barrier(0);
    }
}

__device__ __forceinline__ BwdCoef bwd_coef(const Team& g, int64_t u, const TeamChunk& c,
                                            const float* __restrict__ gamma,
                                            const float* __restrict__ beta,
                                            const float* __restrict__ mean,
                                            const float* __restrict__ rstd,
                                            const float* __restrict__ mean_lo) {
    const int64_t ch = c.plane % g.C;
    const float r = rstd[u];
    return BwdCoef{mean[u], r, mean_lo ? -mean_lo[u] * r : 0.0f, gamma ? gamma[ch] : 1.0f,
                   beta ? beta[ch] : 0.0f};
}

// One chunk (x and dy) per half-block, in registers.  RES: dx += dy, so dy is
// kept and dz formed again; else dz takes dy's place.
template <bool SILU, bool RES>
__global__ __launch_bounds__(kTeamThreads, 4) void k_team_bwd(
    const float* __restrict__ dy, const float* __restrict__ x, const float* __restrict__ gamma,
    const float* __restrict__ beta, const float* __restrict__ mean,
    const float* __restrict__ rstd, const float* __restrict__ mean_lo, float* __restrict__ dx,
    float* __restrict__ dgamma, float* __restrict__ dbeta, double2* __restrict__ plane_sums,
    TeamWs ws, Team g) {
    constexpr bool KEEP = SILU && !RES;
    __shared__ float2 wsum[2][4];
    __shared__ double2 gsum[kHalf];
    __shared__ double2 psum[kMaxCpg];  // the unit's plane sums (its first block)
    __shared__ float bc[2];
    __shared__ int late;
    const int hb = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8);
    const int t = threadIdx.x & (kHalf - 1), w = t >> 6;
    const int64_t u = blockIdx.x / (unsigned)g.blocks;
    const int kb = (int)(blockIdx.x - (unsigned)u * g.blocks);
    u64* __restrict__ slots = ws.slots + 2 * u * g.items;
    auto reduce = [&](float2 s, float2* dst) {  // block_sum2's wave part
        s.x = wave_sum(s.x);
        s.y = wave_sum(s.y);
        if ((t & 63) == 0) dst[w] = s;
    };
    auto wave_total = [](const float2* s) {  // and its sum over the waves
        float2 a = s[0];
#pragma unroll
        for (int i = 1; i < 4; ++i) {
            a.x += s[i].x;
            a.y += s[i].y;
        }
        return a;
    };

    const TeamChunk ck = team_chunk(g, u, block_chunk(g, kb, hb));
    const BwdCoef k = bwd_coef(g, u, ck, gamma, beta, mean, rstd, mean_lo);
    f4 v[kVec], d[kVec];
    load_chunk(v, x, ck, t);
    load_chunk(d, dy, ck, t);
    reduce(chunk_bwd_sums<SILU, KEEP>(v, d, k), wsum[hb]);
    lds_barrier();
    if ((int)threadIdx.x < g.ipb && kb * g.ipb + (int)threadIdx.x < g.items) {
        double A = 0.0, B = 0.0;
        for (int i = 0; i < g.nq; ++i) {
            const int m = threadIdx.x * g.nq + i;
            if (block_chunk(g, kb, m) < 0) continue;
            const float2 s = wave_total(wsum[m]);
            A += (double)s.x;
            B += (double)s.y;
        }
        publish(slots + 2 * (kb * g.ipb + threadIdx.x), A, B);
    }
    if (threadIdx.x == 0) late = g.leave;
    lds_barrier();
    if (hb == 0 && !g.leave) {
        const u64 t0 = __builtin_amdgcn_s_memrealtime();
        gather_bwd(g, t, u, kb == 0, gamma, gsum, psum, &late,
                   [&](int it, double2& v) { return poll(v, slots, it, g, ws, t0); });
    }
    lds_barrier();
    if (late) {
        if (threadIdx.x == 0) team_leave(ws, u, kb);
        return;  // whole block
    }
    if (kb == 0) give_planes(g, u, psum, plane_sums, dgamma, dbeta);
    if (threadIdx.x == 0) finish_bwd(g, gsum, k.r, bc);
    lds_barrier();
    dx_chunk<SILU, RES, KEEP>(v, d, ck, k, bc, dx, t);
}

// The units that blocks left.
template <bool SILU, bool RES>
__global__ __launch_bounds__(kTeamThreads) void k_team_bwd_rest(
    const float* __restrict__ dy, const float* __restrict__ x, const float* __restrict__ gamma,
    const float* __restrict__ beta, const float* __restrict__ mean,
    const float* __restrict__ rstd, const float* __restrict__ mean_lo, float* __restrict__ dx,
    float* __restrict__ dgamma, float* __restrict__ dbeta, double2* __restrict__ plane_sums,
    TeamWs ws, Team g, int64_t blocks) {
    __shared__ double2 gsum[kHalf];
    __shared__ double2 psum[kMaxCpg];
    __shared__ float bc[2];
    if (*ws.any == 0) return;
    const int hb = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8);
    const int t = threadIdx.x & (kHalf - 1);
    for (int64_t b = blockIdx.x; b < blocks; b += gridDim.x) {
        const int64_t u = b / g.blocks;
        const int kb = (int)(b - u * g.blocks);
        const unsigned left = ws.left[u];
        if (left == 0) continue;
        const u64* __restrict__ slots = ws.slots + 2 * u * g.items;
        const TeamChunk ck = team_chunk(g, u, block_chunk(g, kb, hb));
        const BwdCoef k = bwd_coef(g, u, ck, gamma, beta, mean, rstd, mean_lo);
        f4 v[kVec], d[kVec];
        load_chunk(v, x, ck, t);
        load_chunk(d, dy, ck, t);
        int late;
        if (hb == 0)
            gather_bwd(g, t, u, kb == 0, gamma, gsum, psum, &late, [&](int it, double2& p) {
                p = read_slot(slots, it, g);
                return true;
            });
        lds_barrier();
        // (once: a first block that did not leave has added its sums)
        if (kb == 0 && (left & kLeftFirst)) give_planes(g, u, psum, plane_sums, dgamma, dbeta);
        if (threadIdx.x == 0) finish_bwd(g, gsum, k.r, bc);
        lds_barrier();
        dx_chunk<SILU, RES, false>(v, d, ck, k, bc, dx, t);
        lds_barrier();  // the shared sums are free
    }
}

template <typename F>
void bsel(bool b, F&& f) {
    if (b)
        f(std::true_type{});
    else
        f(std::false_type{});
}

// CUs of the current device (a property of the device, asked once each).
int device_cus() {
    static std::atomic<int> cus[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    int n = cus[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return 0;
        cus[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

// Geometry for `depth` chunks per half-block: a block is one item of 2 depth
// chunks, or (backward) several planes of fewer.
Team team_of(const Plan& p, const Tuning& t, bool bwd, int depth) {
    Team g;
    g.C = p.C;
    g.G = p.G;
    g.HW = p.HW;
    g.cpg = (int)p.cpg;
    g.cpp = (int)p.cpp;
    g.P = (int)(p.cpg * p.cpp);
    const int n = 2 * depth;  // chunks of a block
    g.span = bwd ? g.cpp : g.P;
    g.nq = std::min(n, g.span);
    g.lanes = (g.span + g.nq - 1) / g.nq;
    g.items = g.P / g.span * g.lanes;
    g.ipb = n / g.nq;
    g.blocks = (g.items + g.ipb - 1) / g.ipb;
    g.limit = (u64)std::max<int64_t>(t.team_wait_us, 0) * 100;
    g.leave = t.team_wait_us == kTeamLeave;
    return g;
}

bool team_fits(const Plan& p, const Tuning& t, const Team& g) {
    return t.team_wait_us != kTeamOff && p.chunk == kTeamChunk && p.HW % 4 == 0 && p.cpg <= kMaxCpg &&
           p.cpg * p.cpp <= (int64_t)1 << 20 && p.units * p.cpg * p.cpp < (int64_t)1 << 30 &&
           g.blocks <= kMaxTeam * device_cus() / 256;
}

void launch_clear(const Plan& p, const Team& g, const TeamWs& w, hipStream_t s) {
    const int64_t words = 2 * p.units * g.items;
    k_team_clear<<<dim3((unsigned)((words + 255) / 256)), 256, 0, s>>>(w, words, p.units);
}

// Blocks of the launch for what was left (a block walks several there).
dim3 rest_grid(int64_t blocks) {
    return dim3((unsigned)std::min<int64_t>(blocks, 2 * device_cus()));
}

bool aligned(const void* p) { return ((uintptr_t)p & 15) == 0; }

// Outputs written over inputs stay with the two launches: the launch for what
// was left reads inputs of blocks that have written.
bool overlap(const Plan& p, const float* a, const float* b) {
    const int64_t n = p.planes * p.HW;
    return (uintptr_t)a < (uintptr_t)(b + n) && (uintptr_t)b < (uintptr_t)(a + n);
}

}  // namespace

// Chunks per half-block, 0: two launches.  Two, in registers (fewer slots to
// look at than with one); three, with LDS, only for units that need it (more
// than 512 chunks).
int team_fwd_depth(const Plan& p, const Tuning& t, const FwdArgs& a) {
    const int64_t chunks = p.units * p.cpg * p.cpp;
    if (a.res || !aligned(a.x) || !aligned(a.y) || overlap(p, a.x, a.y)) return 0;
    if (chunks < kTeamMinFwd) return 0;
    for (int depth = 2; depth <= 3; ++depth)
        if (team_fits(p, t, team_of(p, t, false, depth))) return depth;
    return 0;
}

// Units of at most 256 chunks (8 MB) backward: the size of a team.
bool team_bwd_fits(const Plan& p, const Tuning& t, const BwdArgs& a) {
    const bool res_silu = (a.flags & SOAR_GN_RESIDUAL) && (a.flags & SOAR_GN_SILU);
    return a.dx && !(a.flags & SOAR_GN_ACCUMULATE_DX) && aligned(a.x) && aligned(a.dy) &&
           aligned(a.dx) && !overlap(p, a.x, a.dx) && !overlap(p, a.dy, a.dx) &&
           p.units * p.cpg * p.cpp >= kTeamMinBwd &&
           !(res_silu && p.units * p.cpg * p.cpp > kTeamMaxResChunks) &&
           team_fits(p, t, team_of(p, t, true, 1));
}

hipError_t launch_team_forward(const Plan& p, const Tuning& t, const FwdArgs& a, const TeamWs& w,
                               int depth, hipStream_t s) {
    const Team g = team_of(p, t, false, depth);
    launch_clear(p, g, w, s);
    const int64_t blocks = p.units * g.blocks;
    const dim3 grid((unsigned)blocks);
    bsel((a.flags & SOAR_GN_SILU) != 0, [&](auto S) {
        bsel((a.flags & SOAR_GN_RESIDUAL) != 0, [&](auto R) {
            auto go = [&](auto NR, auto NL) {
                k_team_fwd<NR(), NL(), S(), R()><<<grid, kTeamThreads, 0, s>>>(
                    a.x, a.gamma, a.beta, a.y, a.mean, a.rstd, a.mean_lo, w, g, a.eps);
            };
            using Z = std::integral_constant<int, 0>;
            using I1 = std::integral_constant<int, 1>;
            using I2 = std::integral_constant<int, 2>;
            if (depth == 2)
                go(I2{}, Z{});
            else
                go(I2{}, I1{});
            k_team_fwd_rest<S(), R()><<<rest_grid(blocks), kTeamThreads, 0, s>>>(
                a.x, a.gamma, a.beta, a.y, a.mean, a.rstd, a.mean_lo, w, g, a.eps, blocks, depth);
        });
    });
    return hipGetLastError();
}

hipError_t launch_team_backward(const Plan& p, const Tuning& t, const BwdArgs& a, const TeamWs& w,
                                double2* plane_sums, hipStream_t s) {
    const Team g = team_of(p, t, true, 1);
    launch_clear(p, g, w, s);
    const int64_t blocks = p.units * g.blocks;
    const dim3 grid((unsigned)blocks);
    bsel((a.flags & SOAR_GN_SILU) != 0, [&](auto S) {
        bsel((a.flags & SOAR_GN_RESIDUAL) != 0, [&](auto R) {
            k_team_bwd<S(), R()><<<grid, kTeamThreads, 0, s>>>(
                a.dy, a.x, a.gamma, a.beta, a.mean, a.rstd, a.mean_lo, a.dx, a.dgamma, a.dbeta,
                plane_sums, w, g);
            k_team_bwd_rest<S(), R()><<<rest_grid(blocks), kTeamThreads, 0, s>>>(
                a.dy, a.x, a.gamma, a.beta, a.mean, a.rstd, a.mean_lo, a.dx, a.dgamma, a.dbeta,
                plane_sums, w, g, blocks);
        });
    });
    return hipGetLastError();
}

}  // namespace gn
}  // namespace soar
