#pragma once
// The step driven from the device: for steps of up to some millions of
// candidates every size (candidates, buckets, uniques, survivors, bytes) is
// read by the next kernel from device memory (LeanPlan) instead of by the
// host, so that a step is one sequence of launches with one wait at its end.
//
// Why: such a step's kernels take 2-60 us each, and the path whose host
// reads every size back spends 35-60 launches and copies and seven waits on
// it, about 5 us of device idle time per launch and 15-20 us per wait
// (a 12-node split_merge step of 1.4e6 candidates: 91 launches, 0.51 ms of
// kernels in 0.73 ms; a 6-node step of 3e3: 42 launches, 0.15 ms in 0.25 ms).
// Driven from the device they take 15 and 11 launches and one or two waits.
// With that, shorter kernels and pooled state buffers, two 6-node iterations
// went from 1.25 to 0.42 ms, four truncated 9-node ones from 3.36 to 1.03 ms,
// a 12-node split_merge step of 2.9e6 candidates from 0.82 to 0.46 ms, an
// erase_create one of 6e6 from 0.95 to 0.62 ms.  Fixed grids cost little: a
// block with nothing to do exits within the launch overhead.  Larger steps
// (beyond kLeanMax) spend under 2 % on launches and waits and keep buffers
// sized for their own counts.
#include <hip/hip_runtime.h>

#include "qd_device.hpp"
#include "qd_k_dedup.hpp"
#include "qd_k_fastgen.hpp"
#include "qd_k_finalize.hpp"
#include "qd_k_generate.hpp"
#include "qd_k_scan.hpp"
#include "qd_k_select.hpp"

namespace qd {

// Clears the words of two areas (the plan and its arrays, the context's
// counters).
__global__ __launch_bounds__(256) void k_lean_clear(u64 *a, u64 na, u64 *b, u64 nb) {
    for (u64 i = u64(blockIdx.x) * blockDim.x + threadIdx.x; i < na + nb; i += u64(gridDim.x) * blockDim.x) {
        if (i < na) a[i] = 0;
        else b[i - na] = 0;
    }
}

// ---------------------------------------------------------------------------
// child offsets: exclusive prefixes of the parents' child counts (cb) and
// work items (wb, when wi is not null) in one pass, the first parent of every
// chunk of kLeanChunk candidates, and the layout of the step
// ---------------------------------------------------------------------------
constexpr u32 kLeanChunk = 1024;
constexpr u64 kLeanMax = 1ull << 24;  // candidates of a step driven from the device, at most
static_assert(LEAN_SPILL == ERR_SPILL1, "the work items' generate reports its spills in the plan");

// Buckets of C candidates: while one radix pass of at most 2^8 buckets is
// enough, buckets of at most 128 (their dedup blocks all run at once), then
// of at most 480 entries on average, in a capacity of at most 1000 (the
// dedup table holds 1024): 16 sigma and 256 entries beyond the mean, as sub-buckets
// whose hashes repeat spread more than distinct ones.
QD_HD void lean_layout(u64 C, u32 &b1, u32 &b2, u64 &cap1, u64 &cap2) {
    u32 L = 0;
    while (L < 8 && (C >> L) > 128) ++L;
    while (L < 20 && (C >> L) > 480) ++L;
    b1 = L < 8 ? L : 8;
    b2 = L - b1;
    auto slack = [](u64 mean) {  // 16 sqrt(mean), rounded up
        u64 r = 1;
        while (r * r < mean) r <<= 1;
        return 16 * r;
    };
    const u64 m1 = (C >> b1) + 1, m2 = (C >> L) + 1;
    cap1 = b2 ? m1 + slack(m1) + 4096 : 1000;
    cap2 = b2 ? (m2 + slack(m2) + 256 + 63) / 64 * 64 : 0;
    if (cap2 > 1000) cap2 = 1000;
}

// Reports of the scan to the host (pinned memory).
struct ScanReport {
    u64 C, items;
    u32 maxsz, err;
};

__global__ __launch_bounds__(kScanThreads) void k_lean_scan(const u32 *nc, const u32 *wi, u64 N, u32 ntile, u64 *cb,
                                                            u64 *wb, u64 *ctab, u64 ctab_n, u64 c_max, const u32 *maxsz,
                                                            const u32 *err, LeanPlan *lp, u64 *dc, u64 *dw,
                                                            ScanReport *rep) {
    __shared__ u64 tmp[kScanThreads / kWave + 1], tmp2[kScanThreads / kWave + 1];
    __shared__ u64 pre[2];
    __shared__ u32 slot;
    const u32 tile = next_tile(&lp->ticket[0], 0, &slot);
    const u64 base = u64(tile) * kScanTile + u64(threadIdx.x) * kScanItems;
    u32 v[kScanItems], w[kScanItems];
    u64 s = 0, sw = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        v[k] = base + k < N ? nc[base + k] : 0u;
        w[k] = wi && base + k < N ? wi[base + k] : 0u;
        s += v[k];
        sw += w[k];
    }
    u64 total, totalw;
    u64 run = block_excl_scan(s, tmp, total);
    u64 runw = block_excl_scan(sw, tmp2, totalw);
    // one wavefront looks back for each prefix
    if (threadIdx.x < kWave) {
        const u64 e = lookback<kWideVal>(dc, tile, total, 0);
        if (threadIdx.x == 0) pre[0] = e;
    } else if (threadIdx.x < 2 * kWave) {
        const u64 e = lookback<kWideVal>(dw, tile, totalw, 0);
        if (threadIdx.x == kWave) pre[1] = e;
    }
    __syncthreads();
    run += pre[0];
    runw += pre[1];
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const u64 p = base + k;
        if (p < N) {
            cb[p] = run;
            if (wi) wb[p] = runw;
            // chunks whose first candidate is one of this parent's
            for (u64 c = (run + kLeanChunk - 1) / kLeanChunk; c * kLeanChunk < run + v[k] && c < ctab_n; ++c) ctab[c] = p;
        }
        run += v[k];
        runw += w[k];
        if (p + 1 == N) {
            cb[N] = run;
            if (wi) wb[N] = runw;
            lp->C = run;
            lp->items = runw;
            u32 stop = 0;
            if (*err) stop |= LEAN_ERR;
            if (run == 0) stop |= LEAN_EMPTY;
            if (run > c_max) stop |= LEAN_BIG;
            lp->stop[LEAN_SCAN] = stop;
            lean_layout(run, lp->b1, lp->b2, lp->cap1, lp->cap2);
            // (the chunk after the last, where the last one's search ends)
            const u64 c = (run + kLeanChunk - 1) / kLeanChunk;
            if (c < ctab_n) ctab[c] = N - 1;
            rep->C = run;
            rep->items = runw;
            rep->maxsz = *maxsz;
            rep->err = *err;
        }
    }
}

// The host made room for the candidates that the scan found too many.
__global__ void k_lean_room(LeanPlan *lp) {
    if (threadIdx.x == 0) lp->stop[LEAN_SCAN] &= ~LEAN_BIG;
}

// Parent of candidate c: the last p with cb[p] <= c, searched between the
// first parents of c's chunk and of the next one.
__device__ inline u64 lean_parent(const u64 *cb, const u64 *ctab, u64 c) {
    u64 lo = ctab[c / kLeanChunk], hi = ctab[c / kLeanChunk + 1];
    while (lo < hi) {
        const u64 mid = (lo + hi + 1) >> 1;
        if (cb[mid] <= c) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// ---------------------------------------------------------------------------
// generate, one child per lane, fused with the first radix pass: blocks of
// 1024 children rank them per bucket in LDS, reserve one range per bucket and
// write the entries.  One lane walks one child from its parent's masks
// (flip_child / sm_child): about three times the instructions per child of
// the work items' shared walk, but a chain eight times shorter, which is what
// small steps wait for (3e4 children of 9-node split_merge parents: 13 us,
// 36 us with work items).
// ---------------------------------------------------------------------------
template <int KIND>
__global__ __launch_bounds__(1024) void k_lean_generate(Parents P, const PDesc *D, const u64 *cb, const u64 *ctab,
                                                        const u64 *tab, qd_rule rule, LeanPlan *lp, u64 *cnt1,
                                                        Entry *E1, u32 *slotof, u64 *off) {
    if (lean_stopped(lp, LEAN_GENERATE)) return;
    __shared__ u32 bcnt[256];
    __shared__ u64 bidx[256];
    __shared__ cplx ct[4];
    const u64 C = lp->C;
    const u32 b1 = lp->b1;
    const u64 cap1 = lp->cap1;
    if (KIND != QD_RULE_HADAMARD && threadIdx.x == 0) fill_factor_table(coef_of(rule), ct);
    bool spill = false;
    for (u64 c0 = u64(blockIdx.x) * kLeanChunk; c0 < C; c0 += u64(gridDim.x) * kLeanChunk) {
        if (threadIdx.x < 256) bcnt[threadIdx.x] = 0;
        __syncthreads();
        const u64 c = c0 + threadIdx.x;
        u64 h = 0;
        cplx m{0.0, 0.0};
        u32 d = 0, r = 0;
        if (c < C) {
            if (slotof) slotof[c] = ~0u;
            const u64 p = lean_parent(cb, ctab, c);
            const u32 j = u32(c - cb[p]);
            const double2 m0 = P.mag[p];
            m = cplx{m0.x, m0.y};
            if (KIND == QD_RULE_HADAMARD) {
                h = hadamard_child_hash(P.obj + P.begin[p], P.size[p], rule.bit, rule.coef, j, m);
            } else {
                const PDesc pd = D[p];
                if (KIND == QD_RULE_QCGD_SPLIT_MERGE) h = sm_child(pd, tab + sm_tab_base(P.begin[p]), j, ct, m);
                else h = flip_child(pd, j, ct, m);
            }
            d = b1 ? u32(h >> (64 - b1)) : 0u;
            r = atomicAdd(&bcnt[d], 1u);
        }
        __syncthreads();
        if (threadIdx.x < 256 && bcnt[threadIdx.x])
            bidx[threadIdx.x] =
                atomicAdd(reinterpret_cast<unsigned long long *>(cnt1 + threadIdx.x), (unsigned long long)bcnt[threadIdx.x]);
        __syncthreads();
        if (c < C) {
            const u64 at = bidx[d] + r;
            if (at < cap1) {
                Entry e;
                e.hash = h;
                e.cand = c;
                e.re = m.re;
                e.im = m.im;
                E1[u64(d) * cap1 + at] = e;
            } else {
                spill = true;
            }
        }
        __syncthreads();  // bcnt is cleared for the next chunk
    }
    if (spill) atomicOr(&lp->stop[LEAN_GENERATE], LEAN_SPILL);
    // one pass: the last block to end turns the buckets' counts into offsets
    // (a launch of its own cost 5 us).  The counts are read where the atomics
    // leave them; each block's have returned before it takes its ticket.
    if (!off) return;
    __shared__ u64 tmp[1024 / kWave + 1];
    if (threadIdx.x == 0) bcnt[0] = atomicAdd(&lp->ticket[2], 1u);
    __syncthreads();
    if (bcnt[0] != gridDim.x - 1) return;
    const u32 nb = 1u << b1;
    const u64 v = threadIdx.x < nb ? __hip_atomic_load(cnt1 + threadIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
    u64 total;
    const u64 run = block_excl_scan(v, tmp, total);
    if (threadIdx.x < nb) off[threadIdx.x] = run;
    if (threadIdx.x == 0) off[nb] = total;
}

// Bucket offsets (exclusive prefix of the buckets' counts): one block.
__global__ __launch_bounds__(1024) void k_lean_bscan(const u64 *cnt1, const u64 *cnt2, const LeanPlan *lp, u64 *off) {
    if (lean_stopped(lp, LEAN_DEDUP)) return;
    __shared__ u64 tmp[1024 / kWave + 1];
    const u64 *cnt = lp->b2 ? cnt2 : cnt1;
    const u32 nb = 1u << (lp->b1 + lp->b2);
    u64 carry = 0;
    for (u32 base = 0; base < nb; base += 4096) {
        const u32 i0 = base + 4 * threadIdx.x;
        u64 v[4], s = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            v[k] = i0 + k < nb ? cnt[i0 + k] : 0;
            s += v[k];
        }
        u64 total;
        u64 run = carry + block_excl_scan(s, tmp, total);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (i0 + k < nb) off[i0 + k] = run;
            run += v[k];
        }
        carry += total;
    }
    if (threadIdx.x == 0) off[nb] = carry;
}

// ---------------------------------------------------------------------------
// select
// ---------------------------------------------------------------------------
// The bin (of nbin, in descending order) in which the count from the top
// first reaches r, and the keys above it; every thread of the block gets
// them.  nbin is a multiple of the block size, at most 16 of it.
__device__ inline void pick_bin(const u64 *hist, u32 nbin, u64 r, u64 *tmp, u64 *res, u32 &bin, u64 &above) {
    const u32 per = nbin / blockDim.x;
    u64 s = 0;
    for (u32 k = 0; k < per; ++k) s += hist[nbin - 1 - (per * threadIdx.x + k)];
    u64 total;
    u64 run = block_excl_scan(s, tmp, total);
    for (u32 k = 0; k < per; ++k) {
        const u32 b = nbin - 1 - (per * threadIdx.x + k);
        const u64 v = hist[b];
        if (run < r && run + v >= r) {
            res[0] = b;
            res[1] = run;
        }
        run += v;
    }
    __syncthreads();
    bin = u32(res[0]);
    above = res[1];
    __syncthreads();
}

// The second 12-bit digit's histogram (of the slots on the first digit's
// threshold), and the map from representatives to slots, cleared.
__global__ __launch_bounds__(256) void k_lean_hist2(LeanPlan *lp, const u64 *nhist, const u32 *UK, u64 max_obj,
                                                    u64 *hist2, u32 *slotof) {
    if (lean_stopped(lp, LEAN_HIST)) return;
    __shared__ u32 h[kHistBins];
    __shared__ u64 tmp[256 / kWave + 1], res[2];
    const u64 C = lp->C, stride = u64(gridDim.x) * blockDim.x;
    const u64 t0 = u64(blockIdx.x) * blockDim.x + threadIdx.x;
    {
        uint4 *s4 = reinterpret_cast<uint4 *>(slotof);
        for (u64 i = t0; i < (C + 3) / 4; i += stride) s4[i] = make_uint4(~0u, ~0u, ~0u, ~0u);
    }
    if (lp->counters[0] <= max_obj) return;  // every unique survives
    if (blockIdx.x && u64(blockIdx.x) * blockDim.x * 4 >= C) return;
    u32 d1;
    u64 above;
    pick_bin(nhist, kNormBins, max_obj, tmp, res, d1, above);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        lp->d1 = d1;
        lp->r1 = max_obj - above;
        if (d1 == 0) lp->stop[LEAN_HIST] = LEAN_SELECT;  // a threshold among subnormal |m|^2: whole records
    }
    for (int i = threadIdx.x; i < kHistBins; i += blockDim.x) h[i] = 0;
    __syncthreads();
    for (u64 i = t0; i < (C + 3) / 4; i += stride) {
        const uint4 q = reinterpret_cast<const uint4 *>(UK)[i];
        const u32 v[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (u32 k = 0; k < 4; ++k)
            if (4 * i + k < C && (v[k] >> 20) == d1) atomicAdd(&h[(v[k] >> 8) & 0xFFF], 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kHistBins; i += blockDim.x)
        if (h[i]) atomicAdd(reinterpret_cast<unsigned long long *>(hist2 + i), (unsigned long long)h[i]);
}

constexpr u32 kSelRegs = 8;                   // items per thread of the finishing block
constexpr u32 kSelFinish = 1024 * kSelRegs;   // items it takes

// Survivors by slot: all uniques, or those above the 24-bit threshold; the
// ones on it are collected in S for the finishing block.
__global__ __launch_bounds__(256) void k_lean_first(LeanPlan *lp, const u64 *hist2, const u32 *UK, const u64 *UH,
                                                    u64 max_obj, SelItem *S, u32 *slotof) {
    if (lean_stopped(lp, LEAN_FIRST)) return;
    __shared__ u64 tmp[256 / kWave + 1], res[2];
    const u64 C = lp->C, stride = u64(gridDim.x) * blockDim.x;
    const u64 *UR = UH + C;
    const double2 *UM = reinterpret_cast<const double2 *>(UR + C);
    if (lp->counters[0] <= max_obj) {
        for (u64 i = u64(blockIdx.x) * blockDim.x + threadIdx.x; i < C; i += stride) {
            const u64 rep = UR[i];
            if (rep != kNoRep) slotof[rep] = u32(i);
        }
        return;
    }
    if (blockIdx.x && u64(blockIdx.x) * blockDim.x >= C) return;
    u32 d2;
    u64 above;
    pick_bin(hist2, kHistBins, lp->r1, tmp, res, d2, above);
    const u32 prefix24 = (lp->d1 << 12) | d2;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        lp->r2 = lp->r1 - above;
        if (hist2[d2] > kSelFinish) lp->stop[LEAN_FIRST] = LEAN_SELECT;
    }
    const SelKey plain{0u, 0u, 0ull};
    // uniform trip count per wave so that the appends see every lane
    for (u64 base = u64(blockIdx.x) * blockDim.x; base < C; base += stride) {
        const u64 i = base + threadIdx.x;
        const u32 t = i < C ? UK[i] >> 8 : 0u;
        if (t > prefix24) slotof[UR[i]] = u32(i);
        const bool take = i < C && t == prefix24;
        const u64 at = wave_append(take, &lp->ns);
        if (take && at < kSelFinish) {
            const double2 m = UM[i];
            const u64 hh = UH[i];
            S[at] = SelItem{sel_hi(m.x, m.y, hh, plain), ~hh, i};
        }
    }
}

// The r largest keys of the ns items of S (1 <= r <= ns <= kSelFinish),
// whose leading `pos` bits tie: one block, items in registers, a 12-bit
// digit per round through an LDS histogram; keep(slot) for each.  Returns
// false when equal keys are left at the end of the key.  In place of the
// rounds of four launches each (k_sl_*: nine rounds, 200 us in a 12-node
// split_merge step of 1.4e6 candidates): 13 us there, 2-3 us a round.
template <class Keep>
__device__ inline bool select_in_block(const SelItem *S, u32 ns, u64 r, u32 pos, u32 *h, u64 *tmp, u64 *res,
                                       Keep &&keep) {
    u64 hi[kSelRegs], lo[kSelRegs];
    u32 alive = 0;
#pragma unroll
    for (u32 k = 0; k < kSelRegs; ++k) {
        const u32 i = threadIdx.x + 1024 * k;
        hi[k] = lo[k] = 0;
        if (i < ns) {
            hi[k] = S[i].hi;
            lo[k] = S[i].lo;
            alive |= 1u << k;
        }
    }
    u64 tied = ns;
    for (;;) {
        if (r == tied) {  // all that are left
#pragma unroll
            for (u32 k = 0; k < kSelRegs; ++k)
                if ((alive >> k) & 1) keep(S[threadIdx.x + 1024 * k].slot);
            return true;
        }
        if (pos >= 128) return false;
        for (u32 i = threadIdx.x; i < kHistBins; i += 1024) h[i] = 0;
        __syncthreads();
#pragma unroll
        for (u32 k = 0; k < kSelRegs; ++k) {
            const bool a = (alive >> k) & 1;
            const u32 d = key_digit(hi[k], lo[k], pos);
            const u64 m = __ballot(a);
            if (!m) continue;
            // equal |m|^2 are common: a wavefront on one digit adds once
            const int lead = __ffsll((unsigned long long)m) - 1;
            const u32 d0 = __shfl(d, lead, kWave);
            if (__ballot(a && d != d0) == 0) {
                if (int(threadIdx.x & (kWave - 1)) == lead) atomicAdd(&h[d0], u32(__popcll(m)));
            } else if (a) {
                atomicAdd(&h[d], 1u);
            }
        }
        __syncthreads();
        u32 v[kHistBins / 1024];
        u64 s = 0;
#pragma unroll
        for (u32 k = 0; k < kHistBins / 1024; ++k) {
            v[k] = h[kHistBins - 1 - (kHistBins / 1024 * threadIdx.x + k)];
            s += v[k];
        }
        u64 total;
        u64 run = block_excl_scan(s, tmp, total);
#pragma unroll
        for (u32 k = 0; k < kHistBins / 1024; ++k) {
            if (run < r && run + v[k] >= r) {
                res[0] = kHistBins - 1 - (kHistBins / 1024 * threadIdx.x + k);
                res[1] = run;
                res[2] = v[k];
            }
            run += v[k];
        }
        __syncthreads();
        const u32 d = u32(res[0]);
        r -= res[1];
        tied = res[2];
#pragma unroll
        for (u32 k = 0; k < kSelRegs; ++k) {
            if (!((alive >> k) & 1)) continue;
            const u32 t = key_digit(hi[k], lo[k], pos);
            if (t == d) continue;
            alive &= ~(1u << k);
            if (t > d) keep(S[threadIdx.x + 1024 * k].slot);
        }
        pos += 12;
        __syncthreads();  // the histogram and the result are rewritten
    }
}

__global__ __launch_bounds__(1024) void k_lean_finish(LeanPlan *lp, const SelItem *S, u64 max_obj, const u64 *UH,
                                                      u32 *slotof) {
    if (lean_stopped(lp, LEAN_FINISH) || lp->counters[0] <= max_obj) return;
    __shared__ u32 h[kHistBins];
    __shared__ u64 tmp[1024 / kWave + 1], res[3];
    const u64 *UR = UH + lp->C;
    if (!select_in_block(S, u32(lp->ns), lp->r2, 24, h, tmp, res, [&](u64 slot) { slotof[UR[slot]] = u32(slot); }) &&
        threadIdx.x == 0)
        lp->stop[LEAN_FINISH] = LEAN_SELECT;
}

// The same block for the host-driven select: marks the r largest of the ns
// items as k_sl_split does, and reports like it (1 done, 2 equal keys).
__global__ __launch_bounds__(1024) void k_sel_finish(const SelItem *S, u32 ns, u64 r, u32 pos, const u64 *UR,
                                                     u64 *bitmap, u64 *sbm, u32 *state) {
    __shared__ u32 h[kHistBins];
    __shared__ u64 tmp[1024 / kWave + 1], res[3];
    const bool ok = select_in_block(S, ns, r, pos, h, tmp, res, [&](u64 slot) { select_item(true, slot, UR, bitmap, sbm); });
    if (threadIdx.x == 0) *state = ok ? 1u : 2u;
}

// ---------------------------------------------------------------------------
// order: the survivors in ascending representative order, with their
// parents, sizes, padded offsets and magnitudes, in one pass over the
// candidates.  A tile of 4096 candidates lists its survivors in order, sizes
// them, and two look-backs give its first rank and byte.  In place of a
// bitmap, its popcount scan, the placement, the child sizes and the scan of
// the sizes (eight launches): 24 us in place of 75 in a 12-node split_merge
// step of 1.4e6 candidates and 2e4 survivors.  Bound by a tile's chain of
// dependent reads (ticket, slots, parent search, size, look-backs), so a tile
// has 1024 threads: where every candidate survives, 256 of them took it in 16
// rounds (2^17 hadamard children 21 us, now 13).  Byte offsets are 64-bit, in
// the registers of the thread that sums a run of the list, which writes them
// (the same time as a 32-bit list in LDS, which 4096 survivors of 1 MiB pass).
// ---------------------------------------------------------------------------
constexpr u32 kEmitTile = 4096;
constexpr u32 kEmitThreads = 1024;

template <int KIND>
__global__ __launch_bounds__(kEmitThreads) void k_lean_emit(Parents P, const u64 *cb, const u64 *ctab,
                                                            const i32 *delta, LeanPlan *lp, const u32 *slotof,
                                                            const u64 *UH, u32 align, u64 capk, u64 *dk, u64 *db,
                                                            u64 *orep, u64 *opar, u32 *osize, u64 *obegin,
                                                            double2 *omag) {
    if (lean_stopped(lp, LEAN_EMIT)) return;
    constexpr u32 kPer = kEmitTile / kEmitThreads, kWaves = kEmitThreads / kWave, kRuns = kEmitTile / kWave;
    static_assert(kRuns == kWave, "one lane of the first wavefront per run of 64 candidates");
    // the tile's survivors, in order: dedup slot, candidate in the tile,
    // parent beyond the tile's first, size
    __shared__ u32 lslot[kEmitTile], lsize[kEmitTile], lpar[kEmitTile];
    __shared__ u16 loff[kEmitTile];
    __shared__ u32 roff[kRuns + 1];
    __shared__ u64 tmp[kWaves + 1], pre[2];
    __shared__ u32 slot;
    const u64 C = lp->C;
    const double2 *UM = reinterpret_cast<const double2 *>(UH + 2 * C);
    const u32 ntile = u32((C + kEmitTile - 1) / kEmitTile);
    const u32 lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    for (;;) {
        const u32 tile = next_tile(&lp->ticket[1], 0, &slot);
        if (tile >= ntile) return;
        const u64 c0 = u64(tile) * kEmitTile;
        u32 v[kPer];
        u64 m[kPer];
#pragma unroll
        for (u32 k = 0; k < kPer; ++k) {
            const u64 c = c0 + threadIdx.x + kEmitThreads * k;
            v[k] = c < C ? slotof[c] : ~0u;
        }
#pragma unroll
        for (u32 k = 0; k < kPer; ++k) {
            m[k] = __ballot(v[k] != ~0u);
            if (lane == 0) roff[k * kWaves + wid] = u32(__popcll(m[k]));
        }
        __syncthreads();
        if (wid == 0) {
            const u32 n = roff[lane];
            const u32 inc = u32(wave_incl_scan(n));
            roff[lane] = inc - n;
            if (lane == kWave - 1) roff[kRuns] = inc;
        }
        __syncthreads();
        const u32 cnt = roff[kRuns];
#pragma unroll
        for (u32 k = 0; k < kPer; ++k) {
            if (v[k] != ~0u) {
                const u32 q = roff[k * kWaves + wid] + u32(__popcll(m[k] & ((1ull << lane) - 1)));
                lslot[q] = v[k];
                loff[q] = u16(threadIdx.x + kEmitThreads * k);
            }
        }
        __syncthreads();
        const u64 p0 = ctab[c0 / kLeanChunk];
        for (u32 q = threadIdx.x; q < cnt; q += kEmitThreads) {
            const u64 c = c0 + loff[q];
            const u64 p = lean_parent(cb, ctab, c);
            u32 s = P.size[p];
            if (KIND == QD_RULE_QCGD_SPLIT_MERGE) {
                const i32 *dt = delta + sm_delta_base(P.begin[p]);
                for (u32 j = u32(c - cb[p]); j; j &= j - 1) s += u32(dt[__builtin_ctz(j)]);
            }
            lpar[q] = u32(p - p0);
            lsize[q] = s;
        }
        __syncthreads();
        // byte offsets within the tile: each thread a run of the list
        const u32 per = (cnt + kEmitThreads - 1) / kEmitThreads;
        const u32 q0 = min(threadIdx.x * per, cnt), q1 = min(q0 + per, cnt);
        u64 at[kPer], total;
        const u64 bytes = place_run(lsize + q0, q1 - q0, align, at);
        const u64 run = block_excl_scan(bytes, tmp, total);
        if (wid == 0) {
            const u64 e = lookback<kWideVal>(dk, tile, cnt, 0);
            if (lane == 0) pre[0] = e;
        } else if (wid == 1) {
            const u64 e = lookback<kWideVal>(db, tile, total, 0);
            if (lane == 0) pre[1] = e;
        }
        __syncthreads();
        const u64 r0 = pre[0], y0 = pre[1];
        for (u32 q = threadIdx.x; q < cnt; q += kEmitThreads) {
            const u64 r = r0 + q;
            if (r >= capk) continue;  // (the host then makes room and runs this kernel again)
            orep[r] = c0 + loff[q];
            opar[r] = p0 + lpar[q];
            osize[r] = lsize[q];
            omag[r] = UM[lslot[q]];
        }
#pragma unroll
        for (u32 k = 0; k < kPer; ++k)
            if (q0 + k < q1 && r0 + q0 + k < capk) obegin[r0 + q0 + k] = y0 + run + at[k];
        if (tile == ntile - 1 && threadIdx.x == 0) {
            lp->K = r0 + cnt;
            lp->bytes = y0 + total;
            if (r0 + cnt <= capk) obegin[r0 + cnt] = y0 + total;
        }
        __syncthreads();  // the lists are rewritten
    }
}

// ---------------------------------------------------------------------------
// normalize and report
// ---------------------------------------------------------------------------
// The canonical chunk sums (k_sum_chunks) of the K survivors' |m|^2.
__global__ __launch_bounds__(kSumThreads) void k_lean_sum(const LeanPlan *lp, u64 capk, u64 capb, const double2 *mag,
                                                          double *out) {
    if (!lean_fits(lp, capk, capb)) return;
    __shared__ double s[kSumThreads];
    const u64 n = lp->K, nchunk = (n + kSumChunk - 1) / kSumChunk;
    for (u64 ch = blockIdx.x; ch < nchunk; ch += gridDim.x) {
        const double t = sum_chunk(mag, nullptr, n, ch, s);
        if (threadIdx.x == 0) out[ch] = t;
        __syncthreads();  // s is rewritten
    }
}

// The total from the chunk sums (each block by itself: at most kSumChunk of
// them, else the host sums), the magnitudes divided by its root, and the
// report to the host.
__global__ __launch_bounds__(kSumThreads) void k_lean_scale(const LeanPlan *lp, u64 capk, u64 capb, const double *sums,
                                                            double2 *mag, LeanReport *rep) {
    __shared__ double s[kSumThreads];
    const bool fits = lean_fits(lp, capk, capb);
    const u64 n = fits ? lp->K : 0, nchunk = (n + kSumChunk - 1) / kSumChunk;
    double total = 0.0;
    if (nchunk == 1) total = sums[0];
    else if (nchunk && nchunk <= u64(kSumChunk)) total = sum_chunk(nullptr, sums, nchunk, 0, s);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        rep->U = lp->counters[0];
        rep->K = lp->K;
        rep->bytes = lp->bytes;
        rep->total = total;
        rep->stop = lean_stopped(lp, LEAN_EMIT);
        rep->fits = fits;
        rep->b1 = lp->b1;
        rep->b2 = lp->b2;
    }
    const double f = sqrt(total);
    if (f == 1 || nchunk > u64(kSumChunk)) return;
    for (u64 i = u64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += u64(gridDim.x) * blockDim.x) {
        double2 m = mag[i];
        m.x = m.x / f;
        m.y = m.y / f;
        mag[i] = m;
    }
}

}  // namespace qd
