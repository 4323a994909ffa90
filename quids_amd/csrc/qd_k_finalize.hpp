#pragma once
// survivor placement, child sizes and bytes, normalisation sums, modifiers
#include <hip/hip_runtime.h>

#include "qd_device.hpp"
#include "qd_rules.hpp"
#include "qd_sizes.hpp"

namespace qd {

// ===========================================================================
// phase 7/8: order, sizes, populate
// ===========================================================================
// Survivors listed by their dedup output slot: rank = number of smaller
// representatives (popcount prefix of the representative bitmap).
// Survivors enumerated from the slot bitmap (one lane per 64-slot word, no
// bit set at or past U); each goes to the rank of its representative among
// the marked representatives.
__global__ __launch_bounds__(256) void k_place(const u64 *UR, const double2 *UM, const u64 *sbm, u64 U,
                                               const u64 *bitmap, const u64 *wprefix, u64 *orep, double2 *omag) {
    constexpr int kUnroll = 4;  // loads in flight per lane
    const u64 nw = (U + 63) / 64, stride = u64(gridDim.x) * blockDim.x;
    for (u64 w0 = u64(blockIdx.x) * blockDim.x + threadIdx.x; w0 < nw; w0 += kUnroll * stride) {
        u64 m[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const u64 w = w0 + u * stride;
            m[u] = w < nw ? sbm[w] : 0ull;
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            for (u64 mm = m[u]; mm; mm &= mm - 1) {
                const u64 i = (w0 + u * stride) * 64 + u64(__ffsll((unsigned long long)mm) - 1);
                const u64 rep = UR[i];
                const u64 word = bitmap[rep >> 6];
                const u32 bit = u32(rep & 63);
                const u64 r = wprefix[rep >> 6] + __popcll(word & ((1ull << bit) - 1));
                orep[r] = rep;
                omag[r] = UM[i];
            }
        }
    }
}

template <int KIND>
__global__ __launch_bounds__(256) void k_child_size(Parents P, const u64 *cb, qd_rule rule, const u64 *orep, u64 K,
                                                    u32 align, u32 *osize, u64 *padded, u64 *opar) {
    for (u64 k = u64(blockIdx.x) * blockDim.x + threadIdx.x; k < K; k += u64(gridDim.x) * blockDim.x) {
        const u64 c = orep[k];
        const u64 p = find_parent(cb, P.n, c);
        opar[k] = p;  // the populate kernels start from it
        const u32 j = u32(c - cb[p]);
        const u8 *o = P.obj + P.begin[p];
        u32 s;
        if (KIND == QD_RULE_QCGD_SPLIT_MERGE) {
            Graph g(o);
            s = sm_child_size(g, sm_first_hmlz(g), j);
        } else {
            s = P.size[p];
        }
        osize[k] = s;
        padded[k] = u64(s) + align_pad(s, align);
    }
}

// Whether the survivors of a step driven from the device have room in the
// output state (capk objects, capb bytes).
__device__ inline bool lean_fits(const LeanPlan *lp, u64 capk, u64 capb) {
    return !lean_stopped(lp, LEAN_EMIT) && lp->K <= capk && lp->bytes <= capb;
}

// Survivors' bytes.  A wavefront takes a batch of survivors: its lanes fetch
// their places, parents and decisions at once (one chain of dependent loads
// for the batch), then segments of lanes write them one after the other.
//  * erase_create / coin / hadamard: the child is the parent with some
//    particle (qubit) bytes flipped: copied in 8-byte words, the flips of a
//    word's bytes applied in registers (k_populate_flip);
//  * split_merge: one lane per parent node finds what becomes of it, lane
//    masks give the child's nodes and a segment scan places their names; the
//    lanes then copy the names word by word (k_populate_sm).
// Objects of other alignments, or beyond the lists, are written by a slower
// path of the same kernel.
// Copies the parent's words to the child with the flips of child_id applied
// (erase_create / coin: both particle bytes of every flipped node; hadamard:
// byte `bit` xor !child_id), on a segment of SEG lanes (SEG = 64, or 32 when
// two survivors share a wavefront; the segment's lanes are active together;
// a QCGD parent has at most SEG nodes).
template <int KIND, int SEG>
__device__ inline void populate_flip_seg(const u8 *o, u32 psz, u8 *d, u64 span, u32 j, const qd_rule &rule) {
    const u32 lane = threadIdx.x & (kWave - 1);
    const u32 sl = lane & (SEG - 1), sbase = lane & ~(SEG - 1);
    const u64 smask = SEG == kWave ? ~0ull : (((1ull << SEG) - 1) << sbase);
    u64 flipmask = 0;  // nodes whose particles flip (n <= SEG)
    u32 n = 0;
    if (KIND != QD_RULE_HADAMARD) {
        n = ld16(o);
        const bool l = sl < n && o[2 + sl], r = sl < n && o[2 + n + sl];
        const bool elig = sl < n && flip_eligible(KIND == QD_RULE_QCGD_COIN, l, r);
        const u64 em = (u64(__ballot(elig)) & smask) >> sbase;
        const u32 rank = __popcll(em & ((1ull << sl) - 1));
        flipmask = (u64(__ballot(elig && rank < 32 && ((j >> rank) & 1))) & smask) >> sbase;
    }
    for (u64 w = sl; w < (span + 3) / 4; w += SEG) {
        const u32 at = u32(4 * w);
        u32 v = 0;
        if (at + 4 <= psz) v = *reinterpret_cast<const u32 *>(o + at);
        else
            for (u32 q = 0; q < 4; ++q)
                if (at + q < psz) v |= u32(o[at + q]) << (8 * q);
        for (u32 q = 0; q < 4; ++q) {
            const u32 pos = at + q;
            bool flip = false;
            if (KIND == QD_RULE_HADAMARD) flip = pos == rule.bit && j == 0;
            else if (pos >= 2 && pos < 2 + 2 * n) {
                const u32 node = (pos - 2) < n ? pos - 2 : pos - 2 - n;
                flip = (flipmask >> node) & 1;
            }
            if (flip) {
                const u32 byte = (v >> (8 * q)) & 0xFF;
                const u32 nb = KIND == QD_RULE_HADAMARD ? (byte ^ 1u) : (byte ? 0u : 1u);
                v = (v & ~(0xFFu << (8 * q))) | (nb << (8 * q));
            }
        }
        if (at + 4 <= span) *reinterpret_cast<u32 *>(d + at) = v;
        else
            for (u32 q = 0; q < 4 && at + q < span; ++q) d[at + q] = u8(v >> (8 * q));
    }
}

// One survivor, with the lanes of its segment (SEG as above); objects that
// are not 4-byte aligned or have more nodes than the segment are written by
// the segment's first lane.
template <int KIND, int SEG>
__device__ inline void populate_flip_one(const Parents &P, const u64 *cb, const qd_rule &rule, const u64 *orep,
                                         const u64 *opar, u64 k, const u64 *obegin, u8 *oobj) {
    const u32 sl = threadIdx.x & (SEG - 1);
    const u64 c = orep[k];
    const u64 p = opar[k];
    const u32 j = u32(c - cb[p]);
    const u8 *o = P.obj + P.begin[p];
    const u32 psz = P.size[p];
    const u64 ob = obegin[k], oe = obegin[k + 1];
    const u64 span = oe - ob;  // child bytes + zero padding
    u8 *d = oobj + ob;
    const bool aligned = ((P.begin[p] | ob) & 3) == 0;
    const u32 n = KIND == QD_RULE_HADAMARD ? 0 : ld16(o);
    if (aligned && n <= u32(SEG)) {
        populate_flip_seg<KIND, SEG>(o, psz, d, span, j, rule);
    } else if (sl == 0) {
        if (KIND == QD_RULE_HADAMARD) hadamard_child_write(o, psz, rule.bit, j, d);
        else flip_child_write(o, psz, KIND == QD_RULE_QCGD_COIN, j, d);
        for (u64 q = psz; q < span; ++q) d[q] = 0;
    }
}

// The 8 bytes at offset `at` of a flip child from the parent's: the bytes of
// the particle bits (left bits at 2, right bits at 2 + n) of the nodes in
// `flip` are inverted; f0, f1: the low and high words of those bytes' bits,
// flip | flip << n.
__device__ inline u64 flip_word(u64 v, u32 at, u64 f0, u64 f1) {
    u32 bits;  // bit q: byte at + q flips
    if (at == 0) bits = u32(f0 << 2) & 0xFF;
    else {
        const u32 sh = at - 2;
        if (sh >= 128) return v;
        bits = u32(sh < 64 ? (f0 >> sh) | (sh ? f1 << (64 - sh) : 0ull) : f1 >> (sh - 64)) & 0xFF;
    }
    if (!bits) return v;
    u64 m = bits;  // bit q -> byte q
    m = (m | (m << 28)) & 0x0000000F0000000Full;
    m = (m | (m << 14)) & 0x0003000300030003ull;
    m = (m | (m << 7)) & 0x0101010101010101ull;
    constexpr u64 k7F = 0x7F7F7F7F7F7F7F7Full;
    const u64 nz = ((((v & k7F) + k7F) | v) >> 7) & 0x0101010101010101ull;  // 1 in nonzero bytes
    return (v & ~(m * 0xFF)) | (m & ~nz);
}

// Survivors a wavefront takes at a time: 64 when there are enough of them to
// fill the chip with wavefronts (4096), fewer otherwise.
__device__ inline u32 pop_batch(u64 K, u32 least) {
    u32 S = kWave;
    while (S > least && K / S < 4096) S >>= 1;
    return S;
}

// erase_create / coin / hadamard: single-wavefront blocks.  Bound by the
// memory's latency per survivor: with one survivor per wavefront, fetched
// through six dependent loads and stored in 4-byte words, 5.5e5 survivors of
// 808 bytes took 284 us (1.6 TB/s), and now 100 (4.4 TB/s).  D: the parents' descriptors, null in a
// step with graphs of more than 64 nodes (then, and for objects that are not
// 8-byte aligned, one survivor at a time).
template <int KIND>
__global__ __launch_bounds__(kWave) void k_populate_flip(Parents P, const PDesc *D, const u64 *cb, qd_rule rule,
                                                         const u64 *orep, const u64 *opar, u64 K, const u64 *obegin,
                                                         u8 *oobj, const LeanPlan *lp, u64 capb) {
    if (lp) {  // a step driven from the device: K objects of room, capb bytes
        if (!lean_fits(lp, K, capb)) return;
        K = lp->K;
    }
    struct Meta {
        u64 src, dst, f0, f1;
        u32 psz, words;
    };
    __shared__ Meta meta[kWave];
    const u32 lane = threadIdx.x;
    const u32 S = pop_batch(K, 8);
    for (u64 k0 = u64(blockIdx.x) * S; k0 < K; k0 += u64(gridDim.x) * S) {
        const u64 k = k0 + lane;
        const u32 nb = u32(min(u64(S), K - k0));
        u32 words = 0;
        bool slow = false;
        if (lane < nb) {
            const u64 c = orep[k], p = opar[k];
            const u64 ob = obegin[k], span = obegin[k + 1] - ob;
            const u64 pb = P.begin[p];
            u32 j = u32(c - cb[p]);
            Meta m;
            m.src = pb;
            m.dst = ob;
            m.psz = P.size[p];
            m.words = words = u32(span / 8);
            m.f0 = m.f1 = 0;
            slow = ((pb | ob | span) & 7) != 0;
            if (KIND == QD_RULE_HADAMARD) {
                m.f0 = j == 0 ? 1 : 0;
            } else if (D) {
                u64 f = 0;
                for (u64 dm = D[p].dmask; dm && j; dm &= dm - 1, j >>= 1)
                    if (j & 1) f |= dm & (0 - dm);
                const u32 n = D[p].n;
                m.f0 = f | (n < 64 ? f << n : 0ull);
                m.f1 = n < 64 ? (n ? f >> (64 - n) : 0ull) : f;
            } else {
                slow = true;
            }
            meta[lane] = m;
        }
        __syncthreads();
        if (__ballot(slow)) {  // uniform
            // two survivors in 32-lane segments when both parents have at
            // most 32 nodes, else one after the other on all lanes
            for (u32 q = 0; q < nb; q += 2) {
                u32 nq = 0;
                if (KIND != QD_RULE_HADAMARD && lane < 2 && q + lane < nb) nq = ld16(P.obj + P.begin[opar[k0 + q + lane]]);
                if (__ballot(nq > 32) == 0) {
                    if (q + lane / 32 < nb) populate_flip_one<KIND, 32>(P, cb, rule, orep, opar, k0 + q + lane / 32, obegin, oobj);
                } else {
                    for (u32 u = q; u < min(q + 2, nb); ++u)
                        populate_flip_one<KIND, kWave>(P, cb, rule, orep, opar, k0 + u, obegin, oobj);
                }
            }
            __syncthreads();  // meta is rewritten
            continue;
        }
        u32 mw = words;
        for (int off = kWave / 2; off > 0; off >>= 1) mw = max(mw, u32(__shfl_xor(int(mw), off, kWave)));
        u32 seg = 1;  // lanes per survivor: its words, at most 16
        while (seg < mw && seg < 16) seg <<= 1;
        const u32 sl = lane & (seg - 1), per = kWave / seg;
        for (u32 q = lane / seg; q < nb; q += per) {
            const Meta m = meta[q];
            const u8 *src = P.obj + m.src;
            u8 *dst = oobj + m.dst;
            constexpr u32 kUnroll = 4;  // loads in flight per lane
            for (u32 w0 = sl; w0 < m.words; w0 += kUnroll * seg) {
                u64 v[kUnroll];
#pragma unroll
                for (u32 u = 0; u < kUnroll; ++u) {
                    const u32 w = w0 + u * seg, at = 8 * w;
                    v[u] = 0;
                    if (w < m.words) {
                        if (at + 8 <= m.psz) v[u] = *reinterpret_cast<const u64 *>(src + at);
                        else if (at + 4 == m.psz) v[u] = *reinterpret_cast<const u32 *>(src + at);
                        else
                            for (u32 r = 0; r < 8 && at + r < m.psz; ++r) v[u] |= u64(src[at + r]) << (8 * r);
                    }
                }
#pragma unroll
                for (u32 u = 0; u < kUnroll; ++u) {
                    const u32 w = w0 + u * seg;
                    if (w >= m.words) continue;
                    if (KIND == QD_RULE_HADAMARD) {
                        if (m.f0 && w == rule.bit / 8) v[u] ^= 1ull << (8 * (rule.bit & 7));
                    } else {
                        v[u] = flip_word(v[u], 8 * w, m.f0, m.f1);
                    }
                    *reinterpret_cast<u64 *>(dst + 8 * w) = v[u];
                }
            }
        }
        __syncthreads();  // meta is rewritten
    }
}

// split_merge.  A segment of SEG lanes (as many as the batch's widest parent
// has nodes: 16, 32 or 64) writes one survivor at a time, lane i for the
// parent's node i.
constexpr u32 kPopNodes = 64;  // child nodes of a survivor in the lists
constexpr u32 kPopSubs = 384;   // sub_nodes of its names (beyond, one lane writes the child: with 128, a batch of
                                // 256 instances whose names had grown took 4.8 ms a step to write, now 0.5)

// A name tree of the child: an optional new root over the parent's sub_nodes
// [sb, sb + len) and [sb2, sb2 + len2).
struct PopName {
    u32 root;  // its type << 16 | hmlz (0: no new root; a root's type or hmlz is never 0)
    u64 hash;
    u32 sb, len, sb2, len2;
};

// LDS of one survivor.
struct PopSeg {
    u32 head[(4 + 4 * kPopNodes) / 4];  // the child's bytes before its names
    u16 src[kPopSubs];                  // parent's sub_node of each of the child's, or 0x8000 | new root
    u64 nhash[kPopNodes];               // the new roots
    u32 nroot[kPopNodes];
};

struct PopMeta {
    u64 src, dst;
    u32 j, span;
};

template <int SEG>
__device__ inline void populate_sm_seg(const Parents &P, const PopMeta &m, bool have, u8 *oobj, PopSeg &L) {
    const u32 lane = threadIdx.x & (kWave - 1), i = lane & (SEG - 1), sbase = lane & ~(SEG - 1);
    const u64 smask = SEG == kWave ? ~0ull : (((1ull << (SEG & 63)) - 1) << sbase);
    auto sballot = [&](bool x) -> u64 { return (u64(__ballot(x)) & smask) >> sbase; };
    const u8 *o = P.obj + m.src;
    u8 *d = oobj + m.dst;
    const u32 n = have ? ld16(o) : 0;
    const bool in = i < n;
    const bool l = in && o[2 + i], r = in && o[2 + n + i];
    const u8 *nb = o + 2 + 2 * n;
    const u32 b = in ? ld16(nb + 2 * i) : 0, e = in ? ld16(nb + 2 * i + 2) : 0, len = e - b;
    const u32 *subs = reinterpret_cast<const u32 *>(o + 4 + 4 * n);
    // (the root's type << 16 | hmlz)
    const u32 w0 = in ? subs[4 * b] : 0;
    const i32 type = i32(w0) >> 16;
    const i16 hmlz = i16(w0);
    u64 hash = 0;
    if (in) hash = u64(subs[4 * b + 2]) | (u64(subs[4 * b + 3]) << 32);
    const u64 lm = sballot(l), rm = sballot(r);
    const u64 below = (1ull << i) - 1;
    // the decisions (qcgd.hpp:623-668): the wrap-around merge first, then
    // one per split or merge in node order
    const bool split = l && r;
    const bool nl = in && i + 1 < n && ((lm >> (i + 1)) & 1), nr = in && i + 1 < n && ((rm >> (i + 1)) & 1);
    const bool merge = !split && l && nr && !nl;
    const u64 dm = sballot(split || merge);
    const bool fs = (lm & 1) && (rm & 1);
    const bool lmg = !fs && n > 1 && (rm & 1) && ((lm >> (n - 1)) & 1) && !((rm >> (n - 1)) & 1);
    const u32 dn = (lmg ? 1u : 0u) + u32(__popcll(dm & below));
    const bool take = (split || merge) && dn < 32 && ((m.j >> dn) & 1);
    const bool wrap = lmg && (m.j & 1);  // node n - 1 merged with node 0, placed first
    // (a split first node whose left half holds no most left zero: that half goes last)
    const bool late = __shfl(int(take && split && type >= 0 && i == 0 && i16(subs[4 * (b + 1)]) > 0), int(sbase), kWave) != 0;
    const u64 mt = sballot(take && merge);
    const bool gone = ((mt << 1) >> i & 1) || (wrap && (i == 0 || i + 1 == n));
    // the next node's name, for a merge
    const int nx = int(sbase + (i + 1 < n ? i + 1 : 0));
    const u32 b2 = u32(__shfl(int(b), nx, kWave)), len2 = u32(__shfl(int(len), nx, kWave)), w2 = u32(__shfl(int(w0), nx, kWave));
    const u64 hash2 = __shfl((unsigned long long)hash, nx, kWave);
    PopName A{0, 0, b, len, 0, 0}, B{0, 0, 0, 0, 0, 0};  // what this node becomes
    bool al = l, ar = r;
    const bool wrapper = wrap && i + 1 == n;
    u32 cnt = in && !gone ? 1 : 0;
    if (take && split) {
        if (type >= 0) {  // a pair's halves
            A = PopName{0, 0, b + 1, u32(type) - 1, 0, 0};
            B = PopName{0, 0, b + u32(type), len - u32(type), 0, 0};
        } else {
            A = PopName{(u32(u16(QCGD_DOT_L)) << 16) | u16(hmlz < 0 ? -1 : 1), hash_combine(hash, u64(i64(QCGD_DOT_L))), b, len, 0, 0};
            B = PopName{(u32(u16(QCGD_DOT_R)) << 16) | u16(1), hash_combine(hash, u64(i64(QCGD_DOT_R))), b, len, 0, 0};
        }
        al = true;
        ar = false;
        cnt = 2;
    } else if ((take && merge) || wrapper) {
        bool same = false;  // the halves of one node: it is whole again
        if (type == QCGD_DOT_L && (i32(w2) >> 16) == QCGD_DOT_R)
            same = subs[4 * (b + 1) + 2] == subs[4 * (b2 + 1) + 2] && subs[4 * (b + 1) + 3] == subs[4 * (b2 + 1) + 3];
        if (same) A = PopName{0, 0, b + 1, len - 1, 0, 0};
        else A = PopName{((len + 1) << 16) | u16((hmlz < 0 || i16(w2) < 0) ? -1 : 1), hash_combine(hash, hash2), b, len, b2, len2};
        al = ar = true;
        cnt = 1;
    }
    if (late && i == 0) {  // (its left half: B, placed last; its right half: A)
        const PopName t = A;
        A = B;
        B = t;
        al = false;
        ar = true;
    }
    const u32 la = cnt ? (A.root ? 1u : 0u) + A.len + A.len2 : 0u, lb = cnt == 2 ? (B.root ? 1u : 0u) + B.len : 0u;
    // places of the child's nodes and names: [wrapped merge] nodes in order
    // [late half]
    const bool own = cnt && !wrapper, two = cnt == 2 && !(late && i == 0);
    const u64 m1 = sballot(own), m2 = sballot(two);
    const u32 first = wrap ? 1u : 0u;
    const u32 nc = first + u32(__popcll(m1)) + u32(__popcll(m2)) + (late ? 1u : 0u);
    u32 pa = first + u32(__popcll(m1 & below)) + u32(__popcll(m2 & below));
    u32 sum = own ? la + (two ? lb : 0u) : 0u;
    u32 inc = sum;
#pragma unroll
    for (int dd = 1; dd < SEG; dd <<= 1) {
        const u32 t = __shfl_up(inc, dd, SEG);
        if (int(i) >= dd) inc += t;
    }
    const u32 wlen = wrap ? u32(__shfl(int(la), int(sbase + n - 1), kWave)) : 0u;  // (uniform over the segment)
    const u32 ownlen = u32(__shfl(int(inc), int(sbase + SEG - 1), kWave));
    const u32 llen = late ? u32(__shfl(int(lb), int(sbase), kWave)) : 0u;
    const u32 nsub = wlen + ownlen + llen;
    u32 oa = wlen + inc - sum, pbn = pa + 1, obn = oa + la;
    if (wrapper) pa = oa = 0;
    if (late && i == 0) {
        pbn = nc - 1;
        obn = wlen + ownlen;
    }
    const bool fits = have && nc <= kPopNodes && nsub <= kPopSubs;  // uniform over the segment
    if (fits) {
        u8 *hd = reinterpret_cast<u8 *>(L.head);
        auto put = [&](const PopName &x, u32 at, u32 off, bool nl_, bool nr_) {
            hd[2 + at] = nl_;
            hd[2 + nc + at] = nr_;
            st16(hd + 2 + 2 * nc + 2 * at, u16(off));
            if (x.root) {
                L.nroot[at] = x.root;
                L.nhash[at] = x.hash;
                L.src[off++] = u16(0x8000u | at);
            }
            for (u32 q = 0; q < x.len; ++q) L.src[off++] = u16(x.sb + q);
            for (u32 q = 0; q < x.len2; ++q) L.src[off++] = u16(x.sb2 + q);
        };
        if (cnt) put(A, pa, oa, al, ar);
        if (cnt == 2) put(B, pbn, obn, late && i == 0, !(late && i == 0));
        if (i == 0) {
            st16(hd, u16(nc));
            st16(hd + 2 + 4 * nc, u16(nsub));
        }
    }
    __syncthreads();  // (single-wavefront blocks: the lists are in place)
    if (fits) {
        u32 *dw = reinterpret_cast<u32 *>(d);
        const u32 hw = 1 + nc, cw = hw + 4 * nsub;
        for (u32 w = i; w < hw; w += SEG) dw[w] = L.head[w];
        constexpr u32 kUnroll = 4;  // loads in flight per lane
        for (u32 t0 = i; t0 < 4 * nsub; t0 += kUnroll * SEG) {
            u32 v[kUnroll];
#pragma unroll
            for (u32 u = 0; u < kUnroll; ++u) {
                const u32 t = t0 + u * SEG;
                v[u] = 0;
                if (t < 4 * nsub) {
                    const u32 s = L.src[t >> 2], q = t & 3;
                    if (!(s & 0x8000u)) v[u] = subs[4 * s + q];
                    else if (q == 0) v[u] = L.nroot[s & 0x7FFF];
                    else if (q >= 2) v[u] = u32(L.nhash[s & 0x7FFF] >> (32 * (q - 2)));
                }
            }
#pragma unroll
            for (u32 u = 0; u < kUnroll; ++u) {
                const u32 t = t0 + u * SEG;
                if (t < 4 * nsub) dw[hw + t] = v[u];
            }
        }
        if (4 * cw < m.span && i == 0)
            for (u32 q = 4 * cw; q < m.span; ++q) d[q] = 0;
    } else if (have && i == 0) {  // more nodes or sub_nodes than the lists hold
        Graph g(o);
        const u32 sz = sm_child_write(g, sm_first_hmlz(g), m.j, d);
        for (u32 q = sz; q < m.span; ++q) d[q] = 0;
    }
    __syncthreads();  // the lists are rewritten
}

// Single-wavefront blocks; bound by the memory's latency per survivor, as
// k_populate_flip.  One lane per survivor listing the child's nodes, and one
// per child node copying its name, took 2.2 ms for 2.1e6 survivors of 550
// bytes; this takes 0.9 (1.1 without the bound on the registers, which
// makes room for a fourth wavefront per SIMD; at six it spills, 1.5).
__global__ __launch_bounds__(kWave, 4) void k_populate_sm(Parents P, const u64 *cb, const u64 *orep, const u64 *opar,
                                                       u64 K, const u64 *obegin, u8 *oobj, const LeanPlan *lp,
                                                       u64 capb) {
    if (lp) {  // as in k_populate_flip
        if (!lean_fits(lp, K, capb)) return;
        K = lp->K;
    }
    __shared__ PopMeta meta[kWave];
    __shared__ PopSeg segs[kWave / 16];
    const u32 lane = threadIdx.x;
    const u32 S = pop_batch(K, 4);
    for (u64 k0 = u64(blockIdx.x) * S; k0 < K; k0 += u64(gridDim.x) * S) {
        const u32 nb = u32(min(u64(S), K - k0));
        u32 n = 0;
        bool slow = false;
        if (lane < nb) {
            const u64 k = k0 + lane, c = orep[k], p = opar[k];
            PopMeta m;
            m.src = P.begin[p];
            m.dst = obegin[k];
            m.span = u32(obegin[k + 1] - m.dst);
            m.j = u32(c - cb[p]);
            meta[lane] = m;
            n = ld16(P.obj + m.src);
            slow = ((m.src | m.dst) & 3) != 0 || n > u32(kWave);
            if (slow) {
                Graph g(P.obj + m.src);
                u8 *d = oobj + m.dst;
                const u32 sz = sm_child_write(g, sm_first_hmlz(g), m.j, d);
                for (u32 q = sz; q < m.span; ++q) d[q] = 0;
            }
        }
        const u64 skip = __ballot(slow);
        const bool wide = __ballot(!slow && n > 32), mid = __ballot(!slow && n > 16);
        __syncthreads();
        const u32 sg = wide ? 64u : mid ? 32u : 16u;
        for (u32 q0 = 0; q0 < nb; q0 += kWave / sg) {
            const u32 q = q0 + lane / sg;
            const bool have = q < nb && !((skip >> q) & 1);
            const PopMeta m = meta[q < nb ? q : 0];
            PopSeg &L = segs[lane / sg];
            if (wide) populate_sm_seg<64>(P, m, have, oobj, L);
            else if (mid) populate_sm_seg<32>(P, m, have, oobj, L);
            else populate_sm_seg<16>(P, m, have, oobj, L);
        }
        __syncthreads();  // meta is rewritten
    }
}

// ===========================================================================
// phase 9: canonical sum of |m|^2 and scaling
// ===========================================================================
constexpr int kSumThreads = 256;
constexpr int kSumChunk = 2048;

// Chunk `ch` of 2048 of the n values (|m|^2, or vals when mag is null), by
// one block: lane t sums t, t+256, ..., t+1792 in order, then a halving tree
// s[t] += s[t+stride], stride = 128 .. 1.  Every thread gets the sum.
__device__ inline double sum_chunk(const double2 *mag, const double *vals, u64 n, u64 ch, double *s) {
    const u64 base = ch * kSumChunk;
    double a = 0.0;
    for (int j = 0; j < kSumChunk / kSumThreads; ++j) {
        const u64 i = base + threadIdx.x + u64(kSumThreads) * j;
        if (i < n) {
            double v;
            if (mag) {
                const double2 m = mag[i];
                v = m.x * m.x + m.y * m.y;
            } else {
                v = vals[i];
            }
            a += v;
        }
    }
    s[threadIdx.x] = a;
    __syncthreads();
    for (int stride = kSumThreads / 2; stride > 0; stride >>= 1) {
        if (threadIdx.x < stride) s[threadIdx.x] = s[threadIdx.x] + s[threadIdx.x + stride];
        __syncthreads();
    }
    return s[0];
}

__global__ __launch_bounds__(kSumThreads) void k_sum_chunks(const double2 *mag, const double *vals, u64 n,
                                                            double *out) {
    __shared__ double s[kSumThreads];
    const double t = sum_chunk(mag, vals, n, blockIdx.x, s);
    if (threadIdx.x == 0) out[blockIdx.x] = t;
}

__global__ __launch_bounds__(256) void k_scale(double2 *mag, u64 n, double f) {
    for (u64 i = u64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += u64(gridDim.x) * blockDim.x) {
        double2 m = mag[i];
        m.x = m.x / f;
        m.y = m.y / f;
        mag[i] = m;
    }
}

// ===========================================================================
// modifiers
// ===========================================================================
__global__ __launch_bounds__(256) void k_modifier(u8 *obj, const u64 *begin, const u32 *size, double2 *mag, u64 n,
                                                  qd_modifier m, u32 *err) {
    for (u64 i = u64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += u64(gridDim.x) * blockDim.x) {
        u8 *o = obj + begin[i];
        const u32 sz = size[i];
        if (m.kind <= QD_MOD_ZGATE) {
            if (m.bit >= sz || (m.kind == QD_MOD_CNOT && m.control_bit >= sz)) {
                raise_error(err, ERR_BIT);
                continue;
            }
        } else if (!qcgd_valid(o, sz)) {
            raise_error(err, ERR_OBJECT);
            continue;
        }
        double2 mm = mag[i];
        cplx c{mm.x, mm.y};
        modifier_apply(m, o, sz, c);
        mag[i] = make_double2(c.re, c.im);
    }
}


// Plain streaming copy, 16 bytes per thread per iteration.
__global__ __launch_bounds__(256) void k_copy_probe(const uint4 *src, uint4 *dst, u64 n) {
    for (u64 i = u64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += u64(gridDim.x) * blockDim.x) dst[i] = src[i];
}

}  // namespace qd
