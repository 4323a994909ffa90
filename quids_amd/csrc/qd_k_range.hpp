#pragma once
// Hash-range passes of a step whose candidates exceed the scratch memory:
// the pool of surviving uniques carried from pass to pass.  A pass dedups
// the candidates of one range of top hash bits completely (equal hashes fall
// in the same range), so the step's uniques are the union of the passes'
// uniques, and the pool keeps the best max_num_object of them seen so far.
#include <hip/hip_runtime.h>

#include "qd_device.hpp"
#include "qd_k_dedup.hpp"
#include "qd_k_fastgen.hpp"
#include "qd_k_generate.hpp"
#include "qd_k_select.hpp"

namespace qd {

constexpr u32 kPoolThreads = 512;
constexpr u32 kPoolGrid = 512;  // blocks, at most

// Appends the slots holding a unique (UR != kNoRep) to the pool: hash (the
// slot key rotated back), representative, magnitude and, with UK, the top
// 32 |m|^2 bits, in slot order within a wavefront's run of slots (coalesced
// stores).  With UK, a unique whose top 24 |m|^2 bits are below t24 is left
// out: the pool already holds max_num_object keys at or above that prefix, so
// it can never be kept.  A block counts its run's first and reserves its
// places with one addition: one for every 4096 slots, to the same word, took
// 45 us of a group of 7.3e6 slots of which few are kept.
__global__ __launch_bounds__(kPoolThreads) void k_pool_append(const u64 *SK, const u64 *UR, const double2 *UM,
                                                              const u32 *UK, u32 t24, u64 nslots, u64 *Ph, u64 *Pr,
                                                              double2 *Pm, u32 *Pk, u64 *pcount) {
    constexpr u32 kWaves = kPoolThreads / kWave, kRows = 16;
    __shared__ u64 wcnt[kWaves];
    __shared__ u64 base;
    const u32 lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    const u64 nwave = u64(gridDim.x) * kWaves, w = u64(blockIdx.x) * kWaves + wid;
    const u64 per = (nslots + nwave * kWave - 1) / (nwave * kWave) * kWave;
    const u64 i0 = min(w * per, nslots), i1 = min(i0 + per, nslots);
    // which of a lane's kRows slots to keep (bit q: slot r + 64 q + lane), and
    // their keys.  The 4-byte key first: below t24, the slot, empty or not, is
    // left out without reading its representative; at or above t24 it is a
    // unique.  (All loads of the rows are issued before any is looked at.)
    auto rows = [&](u64 r, u32 (&key)[kRows]) {
        u32 keep = 0;
        u64 at[kRows];
#pragma unroll
        for (u32 q = 0; q < kRows; ++q) at[q] = min(r + q * kWave + lane, i1 - 1);
        if (UK) {
#pragma unroll
            for (u32 q = 0; q < kRows; ++q) key[q] = UK[at[q]];
        }
        if (UK && t24) {
#pragma unroll
            for (u32 q = 0; q < kRows; ++q) keep |= u32(key[q] >> 8 >= t24) << q;
        } else {
            u64 rep[kRows];
#pragma unroll
            for (u32 q = 0; q < kRows; ++q) rep[q] = UR[at[q]];
#pragma unroll
            for (u32 q = 0; q < kRows; ++q) keep |= u32(rep[q] != kNoRep) << q;
        }
#pragma unroll
        for (u32 q = 0; q < kRows; ++q)
            if (r + q * kWave + lane >= i1) keep &= ~(1u << q);
        return keep;
    };
    u64 cnt = 0;
    u32 key[kRows];
    for (u64 r = i0; r < i1; r += kRows * kWave) cnt += u32(__popc(rows(r, key)));
#pragma unroll
    for (int o = kWave / 2; o; o >>= 1) cnt += __shfl_xor(cnt, o, kWave);
    if (lane == 0) wcnt[wid] = cnt;
    __syncthreads();
    if (threadIdx.x == 0) {
        u64 sum = 0;
        for (u32 q = 0; q < kWaves; ++q) {
            const u64 v = wcnt[q];
            wcnt[q] = sum;
            sum += v;
        }
        base = sum ? atomicAdd(reinterpret_cast<unsigned long long *>(pcount), (unsigned long long)sum) : 0;
    }
    __syncthreads();
    if (!cnt) return;
    u64 at0 = base + wcnt[wid];
    for (u64 r = i0; r < i1; r += kRows * kWave) {
        const u32 keep = rows(r, key);
        if (__ballot(keep != 0) == 0) continue;
#pragma unroll
        for (u32 q = 0; q < kRows; ++q) {
            const bool kept = (keep >> q) & 1u;
            const u64 m = __ballot(kept);
            if (kept) {
                const u64 i = r + q * kWave + lane, at = at0 + __popcll(m & ((1ull << lane) - 1));
                Ph[at] = rotr12(SK[i]);
                Pr[at] = UR[i];
                Pm[at] = UM[i];
                if (UK) Pk[at] = key[q];
            }
            at0 += __popcll(m);
        }
    }
}

// Keeps the pool items whose bit is set in keep, in pool order (wprefix:
// exclusive popcount prefix of keep); Pk / Qk (the 32-bit keys) may be null.
__global__ __launch_bounds__(256) void k_pool_compact(const u64 *Ph, const u64 *Pr, const double2 *Pm, const u32 *Pk,
                                                      u64 n, const u64 *keep, const u64 *wprefix, u64 *Qh, u64 *Qr,
                                                      double2 *Qm, u32 *Qk) {
    for (u64 i = u64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += u64(gridDim.x) * blockDim.x) {
        const u64 w = keep[i >> 6];
        if (!((w >> (i & 63)) & 1)) continue;
        const u64 at = wprefix[i >> 6] + __popcll(w & ((1ull << (i & 63)) - 1));
        Qh[at] = Ph[i];
        Qr[at] = Pr[i];
        Qm[at] = Pm[i];
        if (Pk) Qk[at] = Pk[i];
    }
}

// Histogram of the top 12 bits of n 32-bit |m|^2 keys (the pool's).
__global__ __launch_bounds__(256) void k_ukey_hist0(const u32 *UK, u64 n, u64 *hist) {
    __shared__ u32 h[kHistBins];
    for (int i = threadIdx.x; i < kHistBins; i += blockDim.x) h[i] = 0;
    __syncthreads();
    for (u64 i = u64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += u64(gridDim.x) * blockDim.x)
        atomicAdd(&h[UK[i] >> 20], 1u);
    __syncthreads();
    for (int i = threadIdx.x; i < kHistBins; i += blockDim.x)
        if (h[i]) atomicAdd(reinterpret_cast<unsigned long long *>(hist + i), (unsigned long long)h[i]);
}

// Marks the representatives of the pool items in the candidate bitmap.
__global__ __launch_bounds__(256) void k_mark_reps(const u64 *Pr, u64 n, u64 *bitmap) {
    for (u64 i = u64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += u64(gridDim.x) * blockDim.x) mark(bitmap, Pr[i]);
}

// Places every pool item at the rank of its representative among the
// marked ones (ascending candidate order).
__global__ __launch_bounds__(256) void k_place_list(const u64 *Pr, const double2 *Pm, u64 n, const u64 *bitmap,
                                                    const u64 *wprefix, u64 *orep, double2 *omag) {
    for (u64 i = u64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += u64(gridDim.x) * blockDim.x) {
        const u64 rep = Pr[i];
        const u64 r = wprefix[rep >> 6] + __popcll(bitmap[rep >> 6] & ((1ull << (rep & 63)) - 1));
        orep[r] = rep;
        omag[r] = Pm[i];
    }
}

}  // namespace qd
