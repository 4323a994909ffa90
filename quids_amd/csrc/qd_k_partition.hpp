#pragma once
// MSD radix partition of candidates on their hash
#include <hip/hip_runtime.h>

#include "qd_device.hpp"
#include "qd_rules.hpp"

namespace qd {

// ===========================================================================
// phase 4: radix partition
// ===========================================================================
constexpr int kTile1 = 4096;  // entries per workgroup in the first pass
constexpr int kLevel2Bins = 8192;  // up to 13 bits in the second pass

// First pass: from candidate order (index = candidate, hash and magnitude
// as written by generate) to 2^b1 buckets at exact offsets.
// CI, when not null, holds the candidate index of every input position
// (compacted inputs of the hash-range passes).
__global__ __launch_bounds__(256) void k_scatter1(const u64 *H0, const double2 *M0, u64 n, u32 b1, u64 *cursor,
                                                  Entry *out, const u64 *CI) {
    __shared__ u32 cnt[kHistBins];
    __shared__ u64 gbase[kHistBins];
    const int nbin = 1 << b1;
    for (int i = threadIdx.x; i < nbin; i += blockDim.x) cnt[i] = 0;
    __syncthreads();
    const u64 base = u64(blockIdx.x) * kTile1;
    constexpr int kPer = kTile1 / 256;
    u32 dr[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const u64 i = base + threadIdx.x + 256 * k;
        if (i < n) {
            const u32 d = b1 ? u32(H0[i] >> (64 - b1)) : 0u;
            const u32 r = atomicAdd(&cnt[d], 1u);
            dr[k] = (d << 16) | r;
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nbin; i += blockDim.x)
        if (cnt[i]) gbase[i] = atomicAdd(reinterpret_cast<unsigned long long *>(cursor + i), (unsigned long long)cnt[i]);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const u64 i = base + threadIdx.x + 256 * k;
        if (i < n) {
            const double2 m = M0[i];
            Entry e;
            e.hash = H0[i];
            e.cand = CI ? CI[i] : i;
            e.re = m.x;
            e.im = m.y;
            out[gbase[dr[k] >> 16] + (dr[k] & 0xFFFF)] = e;
        }
    }
}

// ---------------------------------------------------------------------------
// A run of entries split by a digit of their key.  A chunk of kSplitChunk
// entries is ordered by digit in LDS first, so that consecutive lanes write
// consecutive places of a bucket rather than one entry to each of up to 64
// buckets per store.
// ---------------------------------------------------------------------------
constexpr u32 kSplitThreads = 1024;
constexpr u32 kSplitBits = 10;      // of the digit, with two workgroups on a CU
constexpr u32 kSplitWideBits = 11;  // with one

// Chunks of 2048 entries: 79 KB, two workgroups fit a CU; of 4096: 156 KB.
template <u32 BITS>
struct SplitLds {
    static constexpr u32 PER = BITS > kSplitBits ? 4 : 2;  // entries of a chunk per thread
    static constexpr u32 CHUNK = kSplitThreads * PER, BINS = 1u << BITS, BPT = BINS / kSplitThreads;
    static_assert(BPT > 0, "every thread has buckets of its own");
    // the chunk's entries by field (8-byte words: an entry's place is random,
    // and a 32-byte store per lane to random places conflicts on the LDS
    // banks far more than four 8-byte ones)
    u64 key[CHUNK], cand[CHUNK];
    double re[CHUNK], im[CHUNK];
    u64 base[BINS];  // place of a bucket's next entry, less lst
    u32 cnt[BINS];   // entries of the chunk per bucket; zero between chunks
    u16 lst[BINS];   // first place of a bucket within the ordered chunk
    u32 tmp[kSplitThreads / kWave];
    __device__ Entry entry(u32 j) const {
        Entry x;
        x.hash = key[j];
        x.cand = cand[j];
        x.re = re[j];
        x.im = im[j];
        return x;
    }
};

// Calls store(d, place, entry index in the ordered chunk) for each of the n
// entries of src: the places of bucket d in a chunk are those that
// reserve(d, k, count), called by the thread whose k-th bucket it is (thread
// t's are t * BPT + k), returns the first of.  An entry that store refuses
// goes to refused(index).  All of L.cnt is zero on entry
// and on return; every thread of the workgroup calls it with the same n and
// nbin (at most 2^BITS).
template <u32 BITS, class Digit, class Reserve, class Store, class Refused>
__device__ inline void split_run(SplitLds<BITS> &L, const Entry *src, u64 n, u32 nbin, Digit digit, Reserve reserve,
                                 Store store, Refused refused) {
    constexpr u32 PER = SplitLds<BITS>::PER, CHUNK = SplitLds<BITS>::CHUNK, BPT = SplitLds<BITS>::BPT;
    const u32 t = threadIdx.x, lane = t & (kWave - 1), wid = t / kWave;
    Entry e[PER];
#pragma unroll
    for (u32 q = 0; q < PER; ++q)
        if (t + kSplitThreads * q < n) e[q] = src[t + kSplitThreads * q];
    for (u64 c0 = 0; c0 < n; c0 += CHUNK) {
        const u32 m = u32(min<u64>(CHUNK, n - c0));
        u32 dr[PER];
#pragma unroll
        for (u32 q = 0; q < PER; ++q)
            if (t + kSplitThreads * q < m) {
                const u32 d = digit(e[q].hash);
                dr[q] = (d << 16) | atomicAdd(&L.cnt[d], 1u);
            }
        __syncthreads();
        // the buckets' first places within the chunk
        u32 v[BPT], sum = 0;
#pragma unroll
        for (u32 k = 0; k < BPT; ++k) {
            v[k] = t * BPT + k < nbin ? L.cnt[t * BPT + k] : 0u;
            sum += v[k];
        }
        u32 inc = sum;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const u32 up = __shfl_up(inc, o, kWave);
            if (lane >= u32(o)) inc += up;
        }
        if (lane == kWave - 1) L.tmp[wid] = inc;
        __syncthreads();
        if (t * BPT < nbin) {
            u32 run = inc - sum;
            for (u32 w = 0; w < wid; ++w) run += L.tmp[w];
#pragma unroll
            for (u32 k = 0; k < BPT; ++k) {
                const u32 d = t * BPT + k;
                if (d < nbin) {
                    L.lst[d] = u16(run);
                    L.base[d] = reserve(d, k, v[k]) - run;
                    L.cnt[d] = 0;
                    run += v[k];
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (u32 q = 0; q < PER; ++q)
            if (t + kSplitThreads * q < m) {
                const u32 at = L.lst[dr[q] >> 16] + (dr[q] & 0xFFFF);
                L.key[at] = e[q].hash;
                L.cand[at] = e[q].cand;
                L.re[at] = e[q].re;
                L.im[at] = e[q].im;
            }
        // (the next chunk's entries are on their way while this one is written)
#pragma unroll
        for (u32 q = 0; q < PER; ++q) {
            const u64 i = c0 + CHUNK + t + kSplitThreads * q;
            if (i < n) e[q] = src[i];
        }
        __syncthreads();
        u32 over = 0;
#pragma unroll
        for (u32 q = 0; q < PER; ++q) {
            const u32 j = t + kSplitThreads * q;
            if (j < m) {
                const u32 d = digit(L.key[j]);
                if (!store(d, L.base[d] + j, j)) over |= 1u << q;
            }
        }
        // (apart from the stores above: an atomic among them made every chunk
        // wait for it, 24 % of the pass)
        while (over) {
            const u32 q = u32(__builtin_ctz(over));
            over &= over - 1;
            refused(t + kSplitThreads * q);
        }
    }
}

// Second pass, one workgroup per first-level bucket, splitting it by the
// next b2 hash bits in one read: sub-bucket d of bucket b owns cap2 slots at
// ((b << b2) + d) * cap2, and the final counts go to cnt2.  Entries beyond a
// sub-bucket's capacity go to the overflow list ovf (*ovf_n of them), where
// k_dedup_big finds them: a hash that hundreds of candidates share overflows
// a sub-bucket or two of hundreds of thousands, and repeating the pass for
// them cost a 12-node split_merge step of 3.2e8 candidates 10.7 ms.  A full
// list (or none) raises ERR_SPILL, and the step repeats this pass with exact
// counts.
// Bound by the memory's writes: ordered chunks make runs of 2 (2^11
// sub-buckets) to hundreds of entries of one store each.  At 2.7e8 entries
// of 2^8 x 2^11 sub-buckets 5.8 ms (3.0 TB/s; 6.7 ms with each lane writing
// its entries where they belong), at 6e6 of 2^8 x 2^6 87 us (4.4 TB/s; 112 us
// before).  For 2^11 sub-buckets a chunk of 4096 and one workgroup a CU beat
// 2^9 x 2^10 with chunks of 2048 and two (5.9 ms, and the first pass 0.35 ms
// slower).
constexpr u32 ERR_SPILL = 16u;
constexpr u64 kOvfCap = 1ull << 16;

// Input bucket b holds off1[b+1] - off1[b] entries, read from in at
// b * in_stride (fixed-capacity first pass) or at off1[b] (in_stride 0).
// Of the nbk1 buckets (2^b1, or a group of them: the caller offsets in and
// off1 to the group's first), workgroup g takes g, g + gridDim.x, ...; with
// parts, g / parts alone, and of it the piece g % parts (places then come from
// cnt2 itself, zero before: the caller clears it).
template <u32 BITS>
__global__ __launch_bounds__(kSplitThreads, BITS > kSplitBits ? 4 : 8) void k_level2_runs(const Entry *in, u64 in_stride, const u64 *off1,
                                                                  u64 nbk1, u32 b1, u32 b2, u64 cap2, Entry *out,
                                                                  u64 *cnt2, u32 *err, Entry *ovf, u64 *ovf_n,
                                                                  u32 parts, LeanPlan *lp) {
    if (lp) {  // a step driven from the device: off1 holds the buckets' counts
        if (lean_stopped(lp, LEAN_LEVEL2) || lp->b2 == 0) return;
        in_stride = lp->cap1;
        b1 = lp->b1;
        b2 = lp->b2;
        cap2 = lp->cap2;
        nbk1 = 1ull << b1;
        err = &lp->stop[LEAN_LEVEL2];
    }
    __shared__ SplitLds<BITS> L;
    constexpr u32 CHUNK = SplitLds<BITS>::CHUNK, BPT = SplitLds<BITS>::BPT;
    const u32 nb2 = 1u << b2, shift = 64 - b1 - b2;
    for (u32 i = threadIdx.x; i < nb2; i += kSplitThreads) L.cnt[i] = 0;
    __syncthreads();
    bool spill = false;
    auto digit = [&](u64 key) { return u32(key >> shift) & (nb2 - 1); };
    for (u32 w = blockIdx.x; w < u32(nbk1) * parts; w += gridDim.x) {
        const u32 b = w / parts, part = w % parts;
        const u64 beg = lp ? 0 : off1[b], all = (lp ? off1[b] : off1[b + 1]) - beg;
        const u64 piece = ((all + parts - 1) / parts + CHUNK - 1) / CHUNK * CHUNK;
        const u64 p0 = min(part * piece, all), p1 = min(p0 + piece, all);
        Entry *region = out + (u64(b) << b2) * cap2;
        u64 *c2 = cnt2 + (u64(b) << b2);
        u32 cur[BPT] = {};  // of this thread's sub-buckets
        split_run(
            L, in + (in_stride ? b * in_stride : beg) + p0, p1 - p0, nb2, digit,
            [&](u32 d, u32 k, u32 v) -> u64 {
                if (parts > 1) return v ? atomicAdd(reinterpret_cast<unsigned long long *>(c2 + d), (unsigned long long)v) : 0;
                cur[k] += v;
                return cur[k] - v;
            },
            [&](u32 d, u64 slot, u32 j) {
                if (slot >= cap2) return false;
                region[u64(d) * cap2 + slot] = L.entry(j);
                return true;
            },
            [&](u32 j) {
                const u64 at = ovf ? atomicAdd(reinterpret_cast<unsigned long long *>(ovf_n), 1ull) : kOvfCap;
                if (at < kOvfCap) ovf[at] = L.entry(j);
                else spill = true;
            });
        if (parts > 1) continue;
#pragma unroll
        for (u32 k = 0; k < BPT; ++k) {
            const u32 d = threadIdx.x * BPT + k;
            if (d < nb2) c2[d] = ovf ? cur[k] : min<u64>(cur[k], cap2);
        }
    }
    if (spill) atomicOr(err, lp ? LEAN_SPILL : ERR_SPILL);
}

// Each region's entries at its running places in the buckets: bucket d
// holds total[d] entries (every block scans the nbin totals, and the first
// writes the nbin + 1 offsets to off), region r's first place in it is
// bm[r * bstride + d] after the column scan.  clr: nclr words to clear (the
// counts of the pass that follows).
__global__ __launch_bounds__(kSplitThreads, 8) void k_region_place(const Entry *in, u64 capr, const u32 *rcount,
                                                                   u32 nreg, u32 shift, u32 nbin, const u32 *bm,
                                                                   u32 bstride, const u64 *total, u64 *off, Entry *out,
                                                                   u64 *clr, u64 nclr) {
    __shared__ SplitLds<kSplitBits> L;
    for (u64 i = u64(blockIdx.x) * kSplitThreads + threadIdx.x; i < nclr; i += u64(gridDim.x) * kSplitThreads)
        clr[i] = 0;
    u64 all;
    const u64 boff = block_excl_scan(threadIdx.x < nbin ? total[threadIdx.x] : 0, L.key, all);  // this thread's bucket's
    if (blockIdx.x == 0) {
        if (threadIdx.x < nbin) off[threadIdx.x] = boff;
        if (threadIdx.x == 0) off[nbin] = all;
    }
    if (threadIdx.x < nbin) L.cnt[threadIdx.x] = 0;
    __syncthreads();
    for (u32 r = blockIdx.x; r < nreg; r += gridDim.x) {
        u64 cur = threadIdx.x < nbin ? boff + bm[u64(r) * bstride + threadIdx.x] : 0;
        split_run(
            L, in + u64(r) * capr, rcount[r], nbin,
            [&](u64 key) { return nbin > 1 ? u32(key >> shift) & (nbin - 1) : 0u; },
            [&](u32, u32, u32 v) {
                cur += v;
                return cur - v;
            },
            [&](u32, u64 at, u32 j) {
                out[at] = L.entry(j);
                return true;
            },
            [](u32) {});
    }
}

// The pass for more than 2^kSplitWideBits sub-buckets (steps beyond 3.3e8
// candidates): ordering a chunk would give runs of an entry or less, so each
// lane writes its entries directly.  Arguments as k_level2_runs.
__global__ __launch_bounds__(1024) void k_level2_fixed(const Entry *in, u64 in_stride, const u64 *off1, u64 nbk1,
                                                       u32 b1, u32 b2, u64 cap2, Entry *out, u64 *cnt2, u32 *err,
                                                       Entry *ovf, u64 *ovf_n) {
    __shared__ u32 ccnt[kLevel2Bins];
    __shared__ u32 cur[kLevel2Bins];
    bool spill = false;
    for (u64 b = blockIdx.x; b < nbk1; b += gridDim.x) {
        const u64 beg = off1[b], end = off1[b + 1];
        const u64 ibase = in_stride ? b * in_stride : beg;  // entry i of [beg, end) is in[ibase + i - beg]
        const u32 nb2 = 1u << b2;
        const u32 shift = 64 - b1 - b2;
        Entry *region = out + (b << b2) * cap2;
        for (u32 i = threadIdx.x; i < nb2; i += blockDim.x) cur[i] = 0;
        // entries of the chunk being split, and the next chunk's, loaded while
        // this one is ranked and written: four 64-bit words per entry (key,
        // candidate, magnitude bits), in plain registers
        // (lanes past the bucket's end load its first entry and drop it)
        const u64 nent = end - beg;
        if (nent == 0) {  // uniform
            for (u32 i = threadIdx.x; i < nb2; i += blockDim.x) cnt2[(b << b2) + i] = 0;
            __syncthreads();
            continue;
        }
        const ulonglong2 *src = reinterpret_cast<const ulonglong2 *>(in + ibase);
        ulonglong2 *dst = reinterpret_cast<ulonglong2 *>(region);
        u64 w0[4], w1[4], w2[4], w3[4], n0[4], n1[4], n2[4], n3[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const u64 i = threadIdx.x + 1024 * k;
            const u64 ii = i < nent ? i : 0;
            const ulonglong2 lo = src[2 * ii], hi = src[2 * ii + 1];
            n0[k] = lo.x;
            n1[k] = lo.y;
            n2[k] = hi.x;
            n3[k] = hi.y;
        }
        for (u64 cbase = beg; cbase < end; cbase += 4096) {
            for (u32 i = threadIdx.x; i < nb2; i += blockDim.x) ccnt[i] = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                w0[k] = n0[k];
                w1[k] = n1[k];
                w2[k] = n2[k];
                w3[k] = n3[k];
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const u64 i = cbase + 4096 - beg + threadIdx.x + 1024 * k;
                const u64 ii = i < nent ? i : 0;
                const ulonglong2 lo = src[2 * ii], hi = src[2 * ii + 1];
                n0[k] = lo.x;
                n1[k] = lo.y;
                n2[k] = hi.x;
                n3[k] = hi.y;
            }
            u32 dr[4] = {0, 0, 0, 0};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const u64 i = cbase + threadIdx.x + 1024 * k;
                if (i < end) {
                    const u32 d = u32(w0[k] >> shift) & (nb2 - 1);
                    dr[k] = (d << 16) | atomicAdd(&ccnt[d], 1u);
                }
            }
            __syncthreads();
            u32 over = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const u64 i = cbase + threadIdx.x + 1024 * k;
                if (i < end) {
                    const u32 d = dr[k] >> 16;
                    const u64 slot = u64(cur[d]) + (dr[k] & 0xFFFF);
                    if (slot < cap2) {
                        const u64 at = u64(d) * cap2 + slot;
                        ulonglong2 lo, hi;
                        lo.x = w0[k];
                        lo.y = w1[k];
                        hi.x = w2[k];
                        hi.y = w3[k];
                        dst[2 * at] = lo;
                        dst[2 * at + 1] = hi;
                    } else {
                        over |= 1u << k;
                    }
                }
            }
            // (apart from the stores above: an atomic among them made every
            // chunk wait for it, 24 % of the pass; read again from in)
            while (over) {
                const u32 k = u32(__builtin_ctz(over));
                over &= over - 1;
                const u64 at = ovf ? atomicAdd(reinterpret_cast<unsigned long long *>(ovf_n), 1ull) : kOvfCap;
                if (at < kOvfCap) ovf[at] = in[ibase + (cbase - beg) + threadIdx.x + 1024 * k];
                else spill = true;
            }
            __syncthreads();
            for (u32 i = threadIdx.x; i < nb2; i += blockDim.x) cur[i] += ccnt[i];
        }
        __syncthreads();
        for (u32 i = threadIdx.x; i < nb2; i += blockDim.x) cnt2[(b << b2) + i] = ovf ? cur[i] : min<u64>(cur[i], cap2);
        __syncthreads();  // cur is cleared for the next bucket
    }
    if (spill) atomicOr(err, ERR_SPILL);
}

// The same split with exact offsets (a counting pass first): used when a
// sub-bucket spills its fixed capacity.  One workgroup per input bucket;
// positions in out and off2 are off1's minus obase (the offset of the
// group's first entry).
__global__ __launch_bounds__(1024) void k_level2_exact(const Entry *in, u64 in_stride, const u64 *off1, u64 obase,
                                                       u32 b1, u32 b2, Entry *out, u64 *off2) {
    __shared__ u32 cnt[kLevel2Bins];
    __shared__ u32 ccnt[kLevel2Bins];
    __shared__ u64 cur[kLevel2Bins];
    __shared__ u64 tmp[1024 / kWave + 1];
    const u64 b = blockIdx.x;
    const u64 beg = off1[b], end = off1[b + 1];
    const u64 ibase = in_stride ? b * in_stride : beg;
    const u32 nb2 = 1u << b2;
    const u32 shift = 64 - b1 - b2;
    for (u32 i = threadIdx.x; i < nb2; i += blockDim.x) cnt[i] = 0;
    __syncthreads();
    for (u64 i = beg + threadIdx.x; i < end; i += blockDim.x) atomicAdd(&cnt[u32(in[ibase + (i - beg)].hash >> shift) & (nb2 - 1)], 1u);
    __syncthreads();
    {
        constexpr int kPer = kLevel2Bins / 1024;
        u32 v[kPer];
        u64 s = 0;
        for (int k = 0; k < kPer; ++k) {
            const u32 d = threadIdx.x * kPer + k;
            v[k] = d < nb2 ? cnt[d] : 0;
            s += v[k];
        }
        u64 total;
        u64 run = block_excl_scan(s, tmp, total);
        for (int k = 0; k < kPer; ++k) {
            const u32 d = threadIdx.x * kPer + k;
            if (d < nb2) {
                cur[d] = beg - obase + run;
                off2[(b << b2) + d] = beg - obase + run;
            }
            run += v[k];
        }
    }
    __syncthreads();
    for (u64 cbase = beg; cbase < end; cbase += 4096) {
        for (u32 i = threadIdx.x; i < nb2; i += blockDim.x) ccnt[i] = 0;
        __syncthreads();
        u32 dr[4];
        for (int k = 0; k < 4; ++k) {
            const u64 i = cbase + threadIdx.x + 1024 * k;
            if (i < end) {
                const u32 d = u32(in[ibase + (i - beg)].hash >> shift) & (nb2 - 1);
                dr[k] = (d << 16) | atomicAdd(&ccnt[d], 1u);
            }
        }
        __syncthreads();
        for (int k = 0; k < 4; ++k) {
            const u64 i = cbase + threadIdx.x + 1024 * k;
            if (i < end) out[cur[dr[k] >> 16] + (dr[k] & 0xFFFF)] = in[ibase + (i - beg)];
        }
        __syncthreads();
        for (u32 i = threadIdx.x; i < nb2; i += blockDim.x) cur[i] += ccnt[i];
        __syncthreads();
    }
}


}  // namespace qd
