#pragma once
// block scans: exclusive prefix of n loaded values
#include <hip/hip_runtime.h>

#include "qd_device.hpp"
#include "qd_rules.hpp"

namespace qd {

// ===========================================================================
// scans: exclusive prefix of n loaded values into out[0..n] (out[n] = total)
// ===========================================================================
constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;

struct LoadU32 {
    const u32 *p;
    __device__ u64 operator()(u64 i) const { return p[i]; }
};
struct LoadU64 {
    const u64 *p;
    __device__ u64 operator()(u64 i) const { return p[i]; }
};
struct LoadPopc {
    const u64 *p;
    __device__ u64 operator()(u64 i) const { return __popcll(p[i]); }
};

// ---------------------------------------------------------------------------
// decoupled look-back (the method of Merrill and Garland, "Single-pass
// Parallel Prefix Scan with Decoupled Look-back", 2016): the exclusive prefix
// of a tile's aggregate over the tiles before it.  desc[t] = status | epoch | value of VB bits: words of an
// earlier launch carry another epoch and read as not there yet, so a buffer
// is cleared when it is made and when the epochs wrap, not for every scan
// (VB = 62: no epochs, cleared for every scan).
// Tiles are handed out by an atomic ticket, so every tile before this one has
// started, and each publishes its aggregate before it waits for anything: the
// wait below always ends.  Status and value are one word, so no fence orders
// them.  Called by the 64 lanes of one wavefront.
// ---------------------------------------------------------------------------
constexpr u32 kEpochBits = 14;
constexpr u32 kShortVal = 62 - kEpochBits;  // value bits of counts and bytes in memory
constexpr u32 kWideVal = 62;                // and of children, which 31 decisions a parent may take beyond 2^48
constexpr u64 kDescAgg = 1ull << 62, kDescPre = 2ull << 62;

template <u32 VB>
__device__ inline u64 lookback(u64 *desc, u32 tile, u64 agg, u32 epoch) {
    constexpr u64 kDescVal = (1ull << VB) - 1;
    const u32 lane = threadIdx.x & (kWave - 1);
    const u64 ep = VB < kWideVal ? u64(epoch) << VB : 0;
    if (tile == 0) {
        if (lane == 0) __hip_atomic_store(desc, kDescPre | ep | agg, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return 0;
    }
    if (lane == 0) __hip_atomic_store(desc + tile, kDescAgg | ep | agg, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    u64 excl = 0;
    for (i64 top = i64(tile) - 1;; top -= kWave) {
        const i64 t = top - i64(lane);
        u64 v = kDescPre | ep;  // before the first tile: the empty prefix
        u64 have;
        do {
            if (t >= 0) v = __hip_atomic_load(desc + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            have = __ballot((v >> 62) != 0 && ((v ^ ep) & ~(3ull << 62) & ~kDescVal) == 0);
        } while (~have);
        const u64 pre = __ballot((v >> 62) == 2);
        const u32 stop = pre ? u32(__ffsll((unsigned long long)pre) - 1) : u32(kWave - 1);
        u64 s = lane <= stop ? (v & kDescVal) : 0;
#pragma unroll
        for (int d = kWave / 2; d > 0; d >>= 1) s += __shfl_xor(s, d, kWave);
        excl += s;
        if (pre) break;
    }
    if (lane == 0)
        __hip_atomic_store(desc + tile, kDescPre | ep | (excl + agg), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return excl;
}

// The next tile of a look-back kernel, for the whole block; first: the
// ticket's value before the launch.
__device__ inline u32 next_tile(u32 *ticket, u32 first, u32 *slot) {
    if (threadIdx.x == 0) *slot = atomicAdd(ticket, 1u) - first;
    __syncthreads();
    return *slot;
}

// One launch and one read of the values (a reduction, a scan of the block
// sums and a second read before it: three launches of 3-6 us each).
template <class Load, u32 VB>
__global__ __launch_bounds__(kScanThreads) void k_scan(Load ld, u64 n, u64 *out, u32 *ticket, u32 first, u64 *desc,
                                                       u32 epoch) {
    __shared__ u64 tmp[kScanThreads / kWave + 1];
    __shared__ u64 pre;
    __shared__ u32 slot;
    const u32 tile = next_tile(ticket, first, &slot);
    const u64 base = u64(tile) * kScanTile + u64(threadIdx.x) * kScanItems;
    u64 v[kScanItems];
    u64 s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        v[k] = base + k < n ? ld(base + k) : 0;
        s += v[k];
    }
    u64 total;
    u64 run = block_excl_scan(s, tmp, total);
    if (threadIdx.x < kWave) {
        const u64 e = lookback<VB>(desc, tile, total, epoch);
        if (threadIdx.x == 0) pre = e;
    }
    __syncthreads();
    run += pre;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        if (base + k < n) out[base + k] = run;
        run += v[k];
        if (base + k + 1 == n) out[n] = run;
    }
}

}  // namespace qd
