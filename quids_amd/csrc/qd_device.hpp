// qd_device.hpp -- device-side building blocks shared by the step kernels:
// block scans, the canonical |m|^2 sum, and the candidate entry format.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

#include "qd_rules.hpp"

namespace qd {

constexpr int kWave = 64;

// Candidates after the first partition pass, as three arrays: hash, index
// in the candidate space (parents in order, then child_id:
// src/quids.hpp:666-694) and magnitude.  Generation writes only hash and
// magnitude, at the candidate's index.
struct Cands {
    u64 *h;
    u64 *c;
    double2 *m;
};

// One candidate in the partition passes: hash, candidate index, magnitude
// (32 bytes, two dwordx4 accesses, one scattered write per candidate).
struct __align__(16) Entry {
    u64 hash;
    u64 cand;
    double re, im;
};

// Raises *m to at least v.  Atomics on one address from every wavefront of
// a large grid serialise (about 11 ns each, measured), so the atomic is
// issued only when a plain read says it can raise the value; a stale read
// costs one atomic more, never a wrong result.
__device__ inline void raise_max(u32 *m, u32 v) {
    if (v > __hip_atomic_load(m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(m, v);
}

__device__ inline u64 wave_incl_scan(u64 v) {
    const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        u64 o = __shfl_up(v, d, kWave);
        if (lane >= d) v += o;
    }
    return v;
}

// Exclusive scan of one value per thread over the block; returns the
// exclusive prefix and the block total.  `tmp` holds blockDim/64 + 1 u64.
__device__ inline u64 block_excl_scan(u64 v, u64 *tmp, u64 &total) {
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave, nw = blockDim.x / kWave;
    const u64 inc = wave_incl_scan(v);
    if (lane == kWave - 1) tmp[wid] = inc;
    __syncthreads();
    if (threadIdx.x == 0) {
        u64 s = 0;
        for (int w = 0; w < nw; ++w) {
            const u64 t = tmp[w];
            tmp[w] = s;
            s += t;
        }
        tmp[nw] = s;
    }
    __syncthreads();
    const u64 r = tmp[wid] + inc - v;
    total = tmp[nw];
    __syncthreads();
    return r;
}

// An error word that may lie in pinned host memory (a modifier's: it raises
// one code only, so a store does).
__device__ inline void raise_error(u32 *err, u32 code) { *reinterpret_cast<volatile u32 *>(err) = code; }

// ---------------------------------------------------------------------------
// A step driven from the device (qd_k_lean.hpp): its sizes and layout, read
// by each kernel when it starts.
// ---------------------------------------------------------------------------
enum : u32 {
    LEAN_ERR = 1u,      // an invalid object, or a graph beyond the fast kernels' 64 nodes
    LEAN_EMPTY = 2u,    // no candidates
    LEAN_BIG = 4u,      // more candidates than there is room for
    LEAN_BUCKET = 8u,   // a bucket that the main dedup kernel hands back
    LEAN_SPILL = 32u,   // a bucket beyond its capacity (ERR_SPILL1's bit)
    LEAN_SELECT = 64u,  // more tied keys than one block takes, or a subnormal threshold
    LEAN_ROOM = 128u    // (the host's) a buffer does not fit the free memory
};
// Kernels that can stop the step, in launch order.  Each sets its own word,
// and a kernel looks only at the words of the kernels before it, so that
// every thread of it sees the same.
enum : int { LEAN_SCAN, LEAN_GENERATE, LEAN_LEVEL2, LEAN_DEDUP, LEAN_HIST, LEAN_FIRST, LEAN_FINISH, LEAN_EMIT };
struct LeanPlan {
    u64 C, items;      // candidates, work items
    u64 cap1, cap2;    // bucket capacities of the first and second radix pass
    u64 counters[8];   // the dedup's: [0] uniques, [5] and [6] buckets handed back
    u64 r1, r2;        // select: keys still to take after the first and second digit
    u64 ns;            // select: keys that tie after the second digit
    u64 K, bytes;      // survivors and their padded bytes
    u32 b1, b2;        // bits of the radix passes
    u32 d1;            // select: the first digit
    alignas(8) u32 ticket[3];  // next tiles of the look-back kernels; blocks of the generate that ended
    u32 stop[LEAN_EMIT];  // LEAN_* by kernel (the dedup's: counters 5 and 6)
};
// (the first two are cleared as one word when the order runs again)
static_assert(offsetof(LeanPlan, ticket) % sizeof(u64) == 0, "the tickets of the look-back kernels share a u64");
// What the last kernel reports to the host (pinned memory).
struct LeanReport {
    u64 U, K, bytes;
    double total;
    u32 stop, fits, b1, b2;
};
// The reasons to stop that the kernels before `stage` gave.
__device__ inline u32 lean_stopped(const LeanPlan *lp, int stage) {
    u32 w = 0;
    for (int i = 0; i < stage; ++i) w |= lp->stop[i];
    if (stage > LEAN_DEDUP && (lp->counters[5] | lp->counters[6])) w |= LEAN_BUCKET;
    return w;
}

}  // namespace qd
