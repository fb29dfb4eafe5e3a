// Batched BFS/SSSP queries over one shared PMA graph: many sources answered by
// one launch per round, one PMA update per batch and one boundary sweep for
// all queries. No reference counterpart (the reference runs one query per
// process); each query follows the single-source semantics of the SSSP/BFS
// operators (hybrid_sssp.cu:28-194, hybrid_bfs.cu:26-167): a BFS query is an
// SSSP with unit weights, and the pair (distance, parent) is kept in one
// 64-bit word updated by a lexicographic atomicMin, so a query gives the same
// distances and parents alone and in a batch.
//
// Layout: queries are cut into G groups of QS slots (QS = 64, or the next
// power of two >= the query count when there are fewer than 64); a vertex
// holds G * QS words of state and one 64-bit mask per group for each of
// act / inv / ninv. A wave step covers 64 / QS items (edges, pairs) times QS
// queries: lane = item * QS + slot.
#ifndef SG_MULTI_H
#define SG_MULTI_H

#include "sg_operators.h"
#include "sg_pma.h"

namespace sg {

using api::hi32;
using api::kInf;
using api::kNone;
using api::lo32;
using api::pack;

constexpr uint32_t kMEdgeChunk = 512;  // edges a wave walks for one (vertex, group) item; the rest is spilled
constexpr int kMUnroll = 8;            // wave steps whose loads are in flight together

enum : uint8_t { kQWeighted = 0, kQUnit = 1, kQNone = 2 };

struct MultiState {
    unsigned long long *best;  // [nv][KP]: distance << 32 | parent; ~0 = unreached
    unsigned long long *act;   // [nv][G]: slots whose distance dropped (to push)
    unsigned long long *inv;   // [nv][G]: slots reset by this batch's deletions
    unsigned long long *ninv;  // [nv][G]: slots reset and not yet propagated to tree children
    uint32_t *invbit;          // [nv / 32]: v has a reset slot in some group
    uint32_t *coarse;          // coarse filter of invbit: one bit per 2^cshift vertices
    uint32_t cshift;
    const uint8_t *kind;       // [KP]: kQWeighted, kQUnit or kQNone (padding)
    uint32_t G, KP, QS, qs_log;
    uint32_t wmode;
    uint64_t wseed;
};

// Spilled piece of an adjacency list: walk [start, start + len) of u for the
// slots in mask of group grp.
struct MDesc {
    uint64_t start;
    uint64_t mask;
    uint32_t u, len, grp, pad;
};

struct QLane {
    uint32_t sub;    // item of the wave step
    uint32_t slot;   // query slot in the group
    uint32_t per;    // items per wave step (64 / QS)
    uint64_t smask;  // the QS bits of this lane's item in a ballot
};
__device__ __forceinline__ QLane qlane(const MultiState &ms) {
    QLane q;
    const uint32_t l = lane_id();
    q.sub = l >> ms.qs_log;
    q.slot = l & (ms.QS - 1);
    q.per = kWave >> ms.qs_log;
    const uint64_t ones = ms.QS == 64 ? ~0ull : ((1ull << ms.QS) - 1);
    q.smask = ones << (q.sub * ms.QS);
    return q;
}

__device__ __forceinline__ uint32_t qweight(const MultiState &ms, uint8_t kind, uint32_t u, uint32_t v) {
    return kind == kQUnit ? 1u : sg_weight(ms.wmode, ms.wseed, u, v);
}

// Relax slot (grp, slot) of v from u at distance du; true when v's distance
// dropped.
__device__ __forceinline__ bool mrelax(const MultiState &ms, uint32_t u, uint32_t v, uint32_t grp, uint32_t slot,
                                       uint32_t du, uint8_t kind) {
    const uint32_t cand = du + qweight(ms, kind, u, v);
    unsigned long long *p = &ms.best[(uint64_t)v * ms.KP + grp * ms.QS + slot];
    const unsigned long long nw = pack(cand, u);
    if (nw >= ld_peek(p)) return false;
    const unsigned long long old = atomicMin(p, nw);
    return cand < hi32(old);
}

// After a wave step: for every item whose ballot bits are set, OR them into
// the item's mask word and put its vertex on the frontier once per round.
__device__ __forceinline__ void mark_items(const MultiState &ms, const PassIO &io, OutStage &st, const QLane &q,
                                           unsigned long long *masks, uint32_t grp, uint32_t v, bool hit, uint32_t *stamp,
                                           uint32_t stamp_val) {
    const uint64_t b = __ballot(hit) & q.smask;
    bool app = false;
    if (q.slot == 0 && b) {
        atomicOr(&masks[(uint64_t)v * ms.G + grp], b >> (q.sub * ms.QS));
        app = atomicExch(&stamp[v], stamp_val) != stamp_val;
    }
    stage_push(app, v, st, io);
}

// Reset the slots of v whose parent is the walking source (child = true in
// the slot's lane): claim them in inv, queue them in ninv, flag v in the
// vertex bitmaps, reset the state words and put v on the frontier.
__device__ __forceinline__ void reset_children(const MultiState &ms, const PassIO &io, OutStage &st, const QLane &q,
                                               uint32_t grp, uint32_t v, bool child, uint32_t *stamp, uint32_t stamp_val) {
    const uint64_t b = __ballot(child) & q.smask;
    uint64_t fresh = 0;
    if (q.slot == 0 && b) {
        const uint64_t m = b >> (q.sub * ms.QS);
        fresh = m & ~atomicOr(&ms.inv[(uint64_t)v * ms.G + grp], m);
    }
    fresh = __shfl(fresh, (int)(q.sub * ms.QS), kWave);
    bool app = false;
    if (q.slot == 0 && fresh) {
        atomicOr(&ms.ninv[(uint64_t)v * ms.G + grp], fresh);
        atomicOr(&ms.invbit[v >> 5], 1u << (v & 31));
        coarse_mark(ms.coarse, ms.cshift, v);
        app = atomicExch(&stamp[v], stamp_val) != stamp_val;
    }
    if ((fresh >> q.slot) & 1u) ms.best[(uint64_t)v * ms.KP + grp * ms.QS + q.slot] = ~0ull;
    stage_push(app, v, st, io);
}

// Position of the r-th (0-based) set bit of m; r < popcount(m).
__device__ __forceinline__ uint32_t nth_set_bit(uint64_t m, uint32_t r) {
    uint32_t pos = 0;
#pragma unroll
    for (uint32_t width = 32; width >= 1; width >>= 1) {
        const uint32_t c = (uint32_t)__popcll(m & ((1ull << width) - 1));
        if (r >= c) {
            r -= c;
            m >>= width;
            pos += width;
        }
    }
    return pos;
}

// Entry v of u's list as a vertex. An entry that is none (no live list holds
// one) stands for u itself: weights are 1 at least, so the edge improves
// nothing, and no vertex is its own tree parent. (Applied where an id is used:
// right after its load it would wait for the ids fetched ahead.)
__device__ __forceinline__ uint32_t target_of(uint32_t v, uint32_t u) { return v != kGap ? v : u; }

// A wave takes the lists of up to 64 (vertex, group) items at a time: lane i
// holds item i's words, the lists are then walked one after the other, each
// item's ids and distances loaded while the one before it is walked.
struct MItem {
    uint32_t u, grp, len;
    uint64_t mask, start;
};

// Slot bits of rank bits (packed lanes).
__device__ __forceinline__ uint64_t rank_to_slots(uint64_t bits, uint64_t mask) {
    uint64_t s = 0;
    while (bits) {
        s |= 1ull << nth_set_bit(mask, (uint32_t)__builtin_ctzll(bits));
        bits &= bits - 1;
    }
    return s;
}

// What the edges of a step did, one edge per lane: hit = slots of v that
// dropped (kMode 0) or whose tree parent is the walked vertex (kMode 1).
template <int kMode>
__device__ __forceinline__ void mfinish(const MultiState &ms, const PassIO &io, OutStage &st, uint32_t *stamp,
                                        uint32_t stamp_val, uint32_t grp, uint32_t v, uint64_t hit) {
    bool app = false;
    if (hit) {
        if (kMode == 0) {
            atomicOr(&ms.act[(uint64_t)v * ms.G + grp], hit);
            app = atomicExch(&stamp[v], stamp_val) != stamp_val;
        } else {  // claim the slots once, queue them, reset their words
            const uint64_t fresh = hit & ~atomicOr(&ms.inv[(uint64_t)v * ms.G + grp], hit);
            if (fresh) {
                atomicOr(&ms.ninv[(uint64_t)v * ms.G + grp], fresh);
                atomicOr(&ms.invbit[v >> 5], 1u << (v & 31));
                coarse_mark(ms.coarse, ms.cshift, v);
                app = atomicExch(&stamp[v], stamp_val) != stamp_val;
                for (uint64_t f = fresh; f; f &= f - 1)
                    ms.best[(uint64_t)v * ms.KP + grp * ms.QS + (uint32_t)__builtin_ctzll(f)] = ~0ull;
            }
        }
    }
    stage_push(app, v, st, io);
}

// Walk one item for a sparse slot mask (at most kSparseSlots queries active at
// u): one lane per edge, the few active slots side by side, instead of QS
// lanes per edge of which most would idle.
constexpr int kSparseSlots = 4;
template <int kMode>
__device__ __forceinline__ void mwalk_sparse(const GraphView &g, const MultiState &ms, const PassIO &io, OutStage &st,
                                             uint32_t *stamp, uint32_t stamp_val, uint32_t u, uint32_t grp, uint64_t mask,
                                             uint64_t start, uint32_t len, uint32_t vv, uint32_t du, uint64_t units) {
    uint32_t sl[kSparseSlots], dus[kSparseSlots];
    bool unit[kSparseSlots], live[kSparseSlots];
    uint64_t m = mask;
#pragma unroll
    for (int a = 0; a < kSparseSlots; ++a) {  // the active slots and u's distances (wave-uniform)
        live[a] = m != 0;
        sl[a] = m ? (uint32_t)__builtin_ctzll(m) : 0u;
        m &= m - 1;
        unit[a] = (units >> sl[a]) & 1ull;
        dus[a] = (uint32_t)__builtin_amdgcn_readlane((int)du, (int)sl[a]);
    }
    const uint32_t lane = lane_id();
    for (uint32_t e0 = 0; e0 < len; e0 += kWave) {
        const bool in = e0 + lane < len;
        const uint32_t v = target_of(e0 == 0 ? vv : edge_at(g, start + min(e0 + lane, len - 1)), u);
        unsigned long long *const p = &ms.best[(uint64_t)v * ms.KP + grp * ms.QS];
        unsigned long long b[kSparseSlots];
#pragma unroll
        for (int a = 0; a < kSparseSlots; ++a) {
            b[a] = 0;
            if (live[a]) b[a] = kMode == 0 ? ld_peek(p + sl[a]) : ld_relaxed(p + sl[a]);
        }
        uint64_t hit = 0;
        if (kMode == 0) {
            const uint32_t w = sg_weight(ms.wmode, ms.wseed, u, v);
            uint32_t cand[kSparseSlots];
#pragma unroll
            for (int a = 0; a < kSparseSlots; ++a) {
                cand[a] = dus[a] + (unit[a] ? 1u : w);
                const unsigned long long nw = pack(cand[a], u);
                const bool ok = in && live[a] && nw < b[a];
                b[a] = 0;
                if (ok) b[a] = atomicMin(p + sl[a], nw);
            }
#pragma unroll
            for (int a = 0; a < kSparseSlots; ++a)
                if (live[a] && cand[a] < hi32(b[a])) hit |= 1ull << sl[a];
        } else {
#pragma unroll
            for (int a = 0; a < kSparseSlots; ++a)
                if (in && live[a] && lo32(b[a]) == u && hi32(b[a]) != kInf) hit |= 1ull << sl[a];
        }
        mfinish<kMode>(ms, io, st, stamp, stamp_val, grp, v, hit);
    }
}

// Relax (kMode 0: activations go to act) or reset the tree children (kMode 1:
// resets go to inv / ninv and the vertex bitmaps) along the lists of the
// wave's items, lane i holding item i; n items.
// 64 edges at a time: their ids and weights are loaded and computed one edge
// per lane, then kMUnroll edges (QS = 64; more with fewer lanes per edge) are
// tested and updated at once, the updates in flight together, and what the 64
// edges did is marked one edge per lane. With a weight in every lane and a
// wait for every edge's update, a dense round of 64 queries over 8 M edges
// took 2.1 ms, bound by instruction issue and those waits.
template <int kMode>
__device__ __forceinline__ void mwalk_items(const GraphView &g, const MultiState &ms, const PassIO &io, OutStage &st,
                                            uint32_t *stamp, uint32_t stamp_val, const MItem &it, uint32_t n,
                                            unsigned long long &edges) {
    const uint32_t lane = lane_id(), ql = min(lane, ms.QS - 1);
    const uint64_t slots = ms.QS == 64 ? ~0ull : (1ull << ms.QS) - 1;
    uint32_t kgrp = ~0u;  // the group units / used describe
    uint64_t units = 0, used = 0;
    // item i's first 64 ids and u's distance in slot `lane`; the mask was taken
    // before, and the distance is read past the caches: an improvement that
    // comes later sets its bit again
    auto ids = [&](uint32_t i) {
        const uint32_t len = (uint32_t)__builtin_amdgcn_readlane((int)it.len, (int)i);
        return len ? edge_at(g, read_lane_u64(it.start, (int)i) + min(lane, len - 1)) : 0u;
    };
    auto dist = [&](uint32_t i) {
        const uint32_t u = (uint32_t)__builtin_amdgcn_readlane((int)it.u, (int)i);
        const uint32_t grp = (uint32_t)__builtin_amdgcn_readlane((int)it.grp, (int)i);
        return kMode == 0 ? hi32(ld_relaxed(&ms.best[(uint64_t)u * ms.KP + grp * ms.QS + ql])) : 0u;
    };
    uint32_t vn = ids(0), dn = dist(0);
    for (uint32_t i = 0; i < n; ++i) {
        uint32_t vv = vn;
        const uint32_t du0 = dn;
        const uint32_t u = (uint32_t)__builtin_amdgcn_readlane((int)it.u, (int)i);
        const uint32_t grp = (uint32_t)__builtin_amdgcn_readlane((int)it.grp, (int)i);
        const uint32_t len = (uint32_t)__builtin_amdgcn_readlane((int)it.len, (int)i);
        const uint64_t start = read_lane_u64(it.start, (int)i);
        uint64_t mask = read_lane_u64(it.mask, (int)i);
        if (i + 1 < n) {
            vn = ids(i + 1);
            dn = dist(i + 1);
        }
        if (grp != kgrp) {
            const uint8_t kind = ms.kind[grp * ms.QS + ql];
            units = __ballot(kind == kQUnit);
            used = __ballot(kind != kQNone) & slots;
            kgrp = grp;
        }
        mask &= used;
        if (kMode == 0) mask &= __ballot(du0 != kInf);
        if (mask == 0 || len == 0) continue;
        edges += len;
        const uint32_t np = (uint32_t)__popcll(mask);
        if (ms.QS > kSparseSlots && np <= kSparseSlots) {
            mwalk_sparse<kMode>(g, ms, io, st, stamp, stamp_val, u, grp, mask, start, len, vv, du0, units);
            continue;
        }
        // W = 2^wlog lanes per edge: rank r of an edge's lanes takes the r-th
        // active slot (packed) or slot r
        const bool packed = ms.QS >= 16 && 2 * np <= ms.QS;
        const uint32_t wlog = packed ? (np <= 8 ? 3u : np <= 16 ? 4u : 5u) : ms.qs_log;
        const uint32_t r = lane & ((1u << wlog) - 1u);
        const bool live = packed ? r < np : ((mask >> r) & 1ull) != 0;
        const uint32_t slot = packed ? (live ? nth_set_bit(mask, r) : 0u) : r;
        const bool unit = (units >> slot) & 1ull;
        const uint32_t du = __shfl(du0, (int)slot, kWave);
        unsigned long long *const col = ms.best + grp * ms.QS + slot;
        const uint32_t per = kWave >> wlog, sub = lane >> wlog;
        const uint64_t ones = wlog == 6 ? ~0ull : (1ull << (1u << wlog)) - 1;
        for (uint32_t e0 = 0; e0 < len; e0 += kWave) {
            const uint32_t ne = min(len - e0, (uint32_t)kWave);
            vv = target_of(vv, u);
            const uint32_t wv = kMode == 0 ? sg_weight(ms.wmode, ms.wseed, u, vv) : 0u;
            const uint32_t vnext = e0 + kWave < len ? edge_at(g, start + min(e0 + kWave + lane, len - 1)) : 0u;
            uint64_t hit = 0;  // ranks of this lane's edge
            // edges past the last repeat it (lanes past ne hold its id): their
            // updates change nothing, their marks fall on the same vertex
            for (uint32_t s0 = 0; s0 < ne; s0 += per * kMUnroll) {
                uint64_t pk[kMUnroll];
                uint32_t cand[kMUnroll];
                unsigned long long *p[kMUnroll];
                bool ok[kMUnroll];
#pragma unroll
                for (int j = 0; j < kMUnroll; ++j) {
                    uint32_t v, w;
                    if (wlog == 6) {
                        v = (uint32_t)__builtin_amdgcn_readlane((int)vv, (int)(s0 + j));
                        w = (uint32_t)__builtin_amdgcn_readlane((int)wv, (int)(s0 + j));
                    } else {
                        const uint32_t e = min(s0 + j * per + sub, (uint32_t)kWave - 1);
                        v = __shfl(vv, (int)e, kWave);
                        w = kMode == 0 ? __shfl(wv, (int)e, kWave) : 0u;
                    }
                    cand[j] = du + (unit ? 1u : w);
                    p[j] = col + (uint64_t)v * ms.KP;
                }
#pragma unroll
                for (int j = 0; j < kMUnroll; ++j) pk[j] = kMode == 0 ? ld_peek(p[j]) : ld_relaxed(p[j]);
                if (kMode == 0) {
#pragma unroll
                    for (int j = 0; j < kMUnroll; ++j) {
                        const unsigned long long nw = pack(cand[j], u);
                        // (a step's positions past 63 must not win an update that edge 63 marks)
                        ok[j] = live && nw < pk[j] && (wlog == 6 || s0 + j * per + sub < (uint32_t)kWave);
                        if (ok[j]) pk[j] = atomicMin(p[j], nw);
                    }
                }
#pragma unroll
                for (int j = 0; j < kMUnroll; ++j) {
                    const bool h = kMode == 0 ? ok[j] && cand[j] < hi32(pk[j])
                                              : live && lo32(pk[j]) == u && hi32(pk[j]) != kInf;
                    const uint64_t b = __ballot(h);
                    if (wlog == 6) {
                        hit = lane == s0 + j ? b : hit;
                    } else if (b) {
                        const uint32_t at = lane - (s0 + j * per);  // the lane's edge among the step's
                        if (at < per) hit = (b >> (at << wlog)) & ones;
                    }
                }
            }
            if (packed) hit = rank_to_slots(hit, mask);
            mfinish<kMode>(ms, io, st, stamp, stamp_val, grp, vv, hit);
            vv = vnext;
        }
    }
}

// Owner of edge k among 64 staged lists: the largest j with excl[j] <= k.
__device__ __forceinline__ uint32_t staged_owner(const uint32_t *excl, uint32_t k) {
    uint32_t lo = 0;
#pragma unroll
    for (uint32_t step = kWave / 2; step > 0; step >>= 1)
        if (excl[lo + step] <= k) lo += step;
    return lo;
}

// LDS of the light path (per wave): 64 items of a wave batch.
constexpr uint32_t kMLightQS = 16;  // light path for one group of at most this many slots
struct MLight {
    uint32_t excl[kWave];
    uint32_t u[kWave];
    uint64_t start[kWave];
    uint32_t mask[kWave];
    uint32_t du[kWave * kMLightQS];
};

// Light path (one group, QS <= kMLightQS): a wave takes 64 frontier vertices
// at once, stages their lists (at most kMEdgeChunk edges each, the rest is
// spilled) and walks the concatenation, 64 / QS edges per wave step.
template <int kMode>
__device__ void mlight(const GraphView &g, const MultiState &ms, const PassIO &io, OutStage &st, MLight &sh,
                       MDesc *spill, uint32_t spill_cap, uint32_t *stamp, uint32_t n, uint64_t gw, uint64_t nw,
                       unsigned long long &edges, unsigned long long &verts) {
    unsigned long long *masks = kMode == 0 ? ms.act : ms.ninv;
    const QLane q = qlane(ms);
    const uint32_t lane = lane_id();
    const uint32_t stamp_val = io.round + 1;
    const uint8_t kind = ms.kind[q.slot];
    const uint32_t per = light_width(n, nw);  // small frontiers spread over all waves
    for (uint64_t b = gw * per; b < n; b += nw * per) {
        const uint64_t idx = b + lane;
        uint32_t u = 0, m = 0, len = 0, deg = 0;
        uint64_t start = 0;
        if (lane < per && idx < n) {
            u = io.in_list[idx];
            m = (uint32_t)atomicExch(&masks[u], 0ull);
            if (m) {
                deg = g.deg[u];
                start = list_start(g, u);
                len = min(deg, kMEdgeChunk);
                count_hot(g, u);
            }
        }
        verts += (uint32_t)__popcll(__ballot(m != 0));
        // lists past the wave's edge budget go to other waves whole, as
        // descriptors; of the others only the tail past kMEdgeChunk does
        const uint32_t pre = wave_incl_scan(len);
        if (len && pre > io.budget) len = 0;
        const uint32_t nch = deg > len ? (deg - len + kMEdgeChunk - 1) / kMEdgeChunk : 0u;
        const uint32_t incl = wave_incl_scan(nch);
        const uint32_t tot = __shfl(incl, kWave - 1, kWave);
        if (tot) {
            uint32_t base = 0;
            if (lane == 0) base = atomicAdd(io.heavy_cnt, tot);
            base = __shfl(base, 0, kWave) + incl - nch;
            for (uint32_t c = 0; c < nch; ++c) {
                const uint32_t lo = len + c * kMEdgeChunk;
                if (base + c < spill_cap) spill[base + c] = MDesc{start + lo, m, u, min(kMEdgeChunk, deg - lo), 0, 0};
                else atomicOr(io.stats + 3, 2ull);
            }
        }
        const uint32_t lincl = wave_incl_scan(len);
        const uint32_t total = __shfl(lincl, kWave - 1, kWave);
        sh.excl[lane] = lincl - len;
        sh.u[lane] = u;
        sh.start[lane] = start;
        sh.mask[lane] = m;
        if (kMode == 0) {
            for (uint32_t s2 = 0; s2 < ms.QS; ++s2)
                sh.du[lane * ms.QS + s2] = ((m >> s2) & 1u) ? hi32(ld_relaxed(&ms.best[(uint64_t)u * ms.KP + s2])) : kInf;
        }
        __builtin_amdgcn_wave_barrier();
        if (total == 0) continue;
        edges += total;
        for (uint32_t k0 = 0; k0 < total; k0 += q.per * kMUnroll) {
            uint32_t vv[kMUnroll], src[kMUnroll], dv[kMUnroll];
            bool on[kMUnroll];
#pragma unroll
            for (int j = 0; j < kMUnroll; ++j) {
                const uint32_t k = k0 + j * q.per + q.sub;
                const bool ok = k < total;
                const uint32_t o = staged_owner(sh.excl, ok ? k : 0u);
                src[j] = sh.u[o];
                on[j] = ok && ((sh.mask[o] >> q.slot) & 1u) && kind != kQNone;
                dv[j] = kMode == 0 ? sh.du[o * ms.QS + q.slot] : 0u;
                vv[j] = ok ? edge_at(g, sh.start[o] + (k - sh.excl[o])) : kGap;
            }
            if (kMode == 0) {
                uint64_t pk[kMUnroll];
                uint32_t cand[kMUnroll];
#pragma unroll
                for (int j = 0; j < kMUnroll; ++j) {
                    const bool ok = on[j] && vv[j] != kGap && dv[j] != kInf;
                    cand[j] = ok ? dv[j] + qweight(ms, kind, src[j], vv[j]) : kInf;
                    pk[j] = ok ? ld_peek(&ms.best[(uint64_t)vv[j] * ms.KP + q.slot]) : 0ull;
                }
#pragma unroll
                for (int j = 0; j < kMUnroll; ++j) {
                    bool hit = false;
                    const unsigned long long nwv = pack(cand[j], src[j]);
                    if (cand[j] != kInf && nwv < pk[j]) {
                        const unsigned long long old = atomicMin(&ms.best[(uint64_t)vv[j] * ms.KP + q.slot], nwv);
                        hit = cand[j] < hi32(old);
                    }
                    mark_items(ms, io, st, q, ms.act, 0, vv[j], hit, stamp, stamp_val);
                }
            } else {
                uint64_t pk[kMUnroll];
#pragma unroll
                for (int j = 0; j < kMUnroll; ++j)
                    pk[j] = (on[j] && vv[j] != kGap) ? ld_relaxed(&ms.best[(uint64_t)vv[j] * ms.KP + q.slot]) : 0ull;
#pragma unroll
                for (int j = 0; j < kMUnroll; ++j) {
                    const uint32_t v = vv[j];
                    const bool child = on[j] && v != kGap && lo32(pk[j]) == src[j] && hi32(pk[j]) != kInf;
                    reset_children(ms, io, st, q, 0, v, child, stamp, stamp_val);
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// One convergence (kMode 0) or invalidation (kMode 1) round: items are
// (frontier vertex, group); the mask of the item is taken (and cleared) from
// act or ninv; lists longer than kMEdgeChunk leave their tail to the next
// round as descriptors; then the descriptors the previous round spilled.
template <int kMode>
__global__ void __launch_bounds__(kBlock) k_mround(GraphView g, MultiState ms, PassIO io, MDesc *spill, const MDesc *sin,
                                                   uint32_t spill_cap, uint32_t *stamp) {
    __shared__ uint32_t s_out[kWavesPerBlock][kOutStage];
    __shared__ unsigned long long s_red[kWavesPerBlock], s_red2[kWavesPerBlock];
    __shared__ MLight s_light[kWavesPerBlock];
    __shared__ uint32_t s_n[kWavesPerBlock + 1];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (io.zero_cnt) *io.zero_cnt = 0;
        if (io.heavy_zero) *io.heavy_zero = 0;
        if (io.log) {
            const uint32_t i = 2 * ((io.round + kRoundLog - 1) % kRoundLog);
            io.log[i] = *io.in_cnt;
            io.log[i + 1] = io.hin_cnt ? *io.hin_cnt : 0u;
        }
    }
    unsigned long long *masks = kMode == 0 ? ms.act : ms.ninv;
    const uint32_t n = min(*io.in_cnt, io.in_cap);
    const uint32_t nh = sin ? min(*io.hin_cnt, spill_cap) : 0u;
    const uint32_t w = threadIdx.x / kWave, lane = lane_id();
    const uint64_t gw = (uint64_t)blockIdx.x * kWavesPerBlock + w, nw = (uint64_t)gridDim.x * kWavesPerBlock;
    OutStage st{s_out[w], 0};
    unsigned long long edges = 0, verts = 0;
    const bool light = ms.G == 1 && ms.QS <= kMLightQS;
    if (light) mlight<kMode>(g, ms, io, st, s_light[w], spill, spill_cap, stamp, n, gw, nw, edges, verts);
    // (frontier vertex, group) items, then the previous round's spilled
    // descriptors, in one loop: a wave takes up to 64 of them at a time, dealt
    // out in turn (neighbours in the frontier are alike: a run of hubs would
    // be one wave's work)
    const uint64_t items = light ? 0 : (uint64_t)n * ms.G;
    for (uint64_t i0 = gw; i0 < items + nh; i0 += nw * kWave) {
        const uint64_t i = i0 + lane * nw;
        MItem it{0, 0, 0, 0, 0};
        uint32_t nch = 0, deg = 0;
        if (i < items) {
            it.u = io.in_list[i / ms.G];
            it.grp = (uint32_t)(i % ms.G);
            it.mask = atomicExch(&masks[(uint64_t)it.u * ms.G + it.grp], 0ull);
            if (it.mask) {
                it.start = list_start(g, it.u);
                count_hot(g, it.u);
                deg = g.deg[it.u];
                it.len = min(deg, kMEdgeChunk);
                nch = (deg - it.len + kMEdgeChunk - 1) / kMEdgeChunk;
            }
        } else if (i < items + nh) {
            const MDesc d = sin[i - items];
            it = MItem{d.u, d.grp, d.len, d.mask, d.start};
        }
        verts += (uint32_t)__popcll(__ballot(i < items && it.mask != 0));
        const uint32_t incl = wave_incl_scan(nch);
        const uint32_t tot = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
        if (tot) {  // the tails of long lists go to the next round
            uint32_t base = 0;
            if (lane == 0) base = atomicAdd(io.heavy_cnt, tot);
            base = (uint32_t)__builtin_amdgcn_readlane((int)base, 0);
            for (uint64_t m = __ballot(nch != 0); m; m &= m - 1) {  // lane by lane, its chunks side by side
                const int l = __builtin_ctzll(m);
                const uint32_t c1 = (uint32_t)__builtin_amdgcn_readlane((int)incl, l);
                const uint32_t cn = (uint32_t)__builtin_amdgcn_readlane((int)nch, l), at = base + c1 - cn;
                const MDesc d{read_lane_u64(it.start, l) + kMEdgeChunk, read_lane_u64(it.mask, l),
                              (uint32_t)__builtin_amdgcn_readlane((int)it.u, l),
                              (uint32_t)__builtin_amdgcn_readlane((int)deg, l) - kMEdgeChunk,
                              (uint32_t)__builtin_amdgcn_readlane((int)it.grp, l), 0};
                for (uint32_t c = lane; c < cn; c += kWave) {
                    const uint32_t lo = c * kMEdgeChunk;
                    if (at + c < spill_cap) spill[at + c] = MDesc{d.start + lo, d.mask, d.u, min(kMEdgeChunk, d.len - lo), d.grp, 0};
                    else atomicOr(io.stats + 3, 2ull);
                }
            }
        }
        mwalk_items<kMode>(g, ms, io, st, stamp, io.round + 1, it,
                           (uint32_t)min_u64(kWave, (items + nh - i0 + nw - 1) / nw), edges);
    }
    block_flush<kWavesPerBlock>(st, io, s_n);
    // one atomic per counter and block
    if (lane == 0) {
        s_red[w] = edges;
        s_red2[w] = verts;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long a = 0, b = 0;
        for (int i = 0; i < kWavesPerBlock; ++i) {
            a += s_red[i];
            b += s_red2[i];
        }
        if (a) atomicAdd(io.stats + 0, a);
        if (b) atomicAdd(io.stats + 1, b);
    }
}

// Pairs (u, v) processed per wave step (one per item, QS slots each):
// kMode 0 relaxes all slots of inserted edges that survive the batch;
// kMode 1 resets the slots of v whose parent is u for deleted edges.
template <int kMode>
__global__ void __launch_bounds__(kBlock) k_mpairs(MultiState ms, BatchView bv, BatchRanges br, PassIO io,
                                                   uint32_t *stamp, uint32_t stamp_val) {
    __shared__ uint32_t s_out[kWavesPerBlock][kOutStage];
    const uint32_t w = threadIdx.x / kWave;
    const QLane q = qlane(ms);
    OutStage st{s_out[w], 0};
    const uint64_t n = kMode == 0 ? bv.nins : bv.ndel;
    const uint64_t gw = (uint64_t)blockIdx.x * kWavesPerBlock + w, nw = (uint64_t)gridDim.x * kWavesPerBlock;
    for (uint64_t b0 = gw * q.per; b0 < n; b0 += nw * q.per) {
        const uint64_t i = b0 + q.sub;
        bool ok = i < n;
        uint32_t u = 0, v = 0;
        if (ok) {
            if (kMode == 0) {
                u = bv.ins_key[i];
                v = bv.ins_val[i];
                ok = u != kGap;
                if (ok) {
                    const uint32_t db = br.del_b[u], de = br.del_e[u];
                    ok = db == de || !in_sorted_u64(bv.del_key, db, de, ((uint64_t)u << 32) | v);
                }
            } else {
                const uint64_t k = bv.del_key[i];
                ok = k != ~0ull;
                u = (uint32_t)(k >> 32);
                v = (uint32_t)k;
            }
        }
        for (uint32_t grp = 0; grp < ms.G; ++grp) {
            const uint32_t qi = grp * ms.QS + q.slot;
            const uint8_t kind = ms.kind[qi];
            const bool on = ok && kind != kQNone;
            if (kMode == 1) {
                const uint64_t cur = on ? ld_relaxed(&ms.best[(uint64_t)v * ms.KP + qi]) : 0ull;
                const bool child = on && lo32(cur) == u && hi32(cur) != kInf;
                reset_children(ms, io, st, q, grp, v, child, stamp, stamp_val);
            } else {
                const uint32_t du = on ? hi32(ld_relaxed(&ms.best[(uint64_t)u * ms.KP + qi])) : kInf;
                const bool hit = on && du != kInf && mrelax(ms, u, v, grp, q.slot, du, kind);
                mark_items(ms, io, st, q, ms.act, grp, v, hit, stamp, stamp_val);
            }
        }
    }
    stage_flush(st, io);
}

constexpr int kSweepSlots = 4;
// Edge-centric sweep for the batch: every live edge (u, v) whose target has a
// reset slot relaxes v's reset slots from u (the sweep hits). Same wave tiles
// as k_sweep_edges: the tile's hits are compacted in place in the wave's LDS
// (owner into own[k], target into the dead base words) and relaxed one hit
// per lane, over the reset slots of the target only.
__global__ void __launch_bounds__(kSweepBlock) k_msweep(GraphView g, const unsigned long long *dpre, SweepTiles tiles,
                                                        MultiState ms, PassIO io, uint32_t *stamp, uint32_t stamp_val) {
    __shared__ SweepWave s_wave[kSweepWaves];
    __shared__ uint32_t s_filter[kFilterWords];
    const unsigned long long E = dpre[g.nv];
    const unsigned long long ntiles = (g.nv + E + kSweepTile - 1) / kSweepTile;
    const uint32_t w = threadIdx.x / kWave, lane = lane_id();
    SweepWave &sh = s_wave[w];
    OutStage st{sh.out, 0, kSweepOutStage};
    uint32_t n_edges = 0;
    const uint32_t cs = ms.cshift;
    load_filter(s_filter, ms.coarse, coarse_words(g.nv, cs));
    TilePipe tp(TileWalk(0, min_u64(ntiles, tiles.cap - 1), kSweepWaves), g, dpre, tiles);
    while (tp.more) {
        uint32_t vv[kSweepPerLane];
        const uint32_t v0 = tp.h.v0;
        sweep_tile(g, dpre, tp.h, tp.pre, g.col, 0, 0, g.nv, sh, vv, n_edges);
        tp.advance(g, dpre, tiles);
        bool pass[kSweepPerLane];
#pragma unroll
        for (int j = 0; j < kSweepPerLane; ++j) pass[j] = coarse_test(s_filter, cs, vv[j] != kGap ? vv[j] : 0u) && vv[j] != kGap;
        uint32_t word[kSweepPerLane];
#pragma unroll
        for (int j = 0; j < kSweepPerLane; ++j) word[j] = pass[j] ? ms.invbit[vv[j] >> 5] : 0u;
        uint32_t nh = 0;  // wave-uniform
        uint32_t *const hv = reinterpret_cast<uint32_t *>(sh.base);
#pragma unroll
        for (int j = 0; j < kSweepPerLane; ++j) {
            const bool h = pass[j] && ((word[j] >> (vv[j] & 31)) & 1u);
            const uint64_t m = __ballot(h);
            if (m) {
                const uint32_t o = sh.own[j * kWave + lane];
                __builtin_amdgcn_wave_barrier();
                if (h) {
                    const uint32_t k = nh + (uint32_t)__popcll(m & lanemask_lt());
                    sh.own[k] = (uint16_t)o;
                    hv[k] = vv[j];
                }
                nh += (uint32_t)__popcll(m);
            }
        }
        __builtin_amdgcn_wave_barrier();
        // one lane per hit: relax exactly the reset slots of its target (usually
        // a few of the group's QS), then flag the improved ones and queue v once
        for (uint32_t i0 = 0; i0 < nh; i0 += kWave) {
            const uint32_t i = i0 + lane;
            bool app = false;
            uint32_t v = 0;
            if (i < nh) {
                v = hv[i];
                const uint32_t u = v0 + sh.own[i];
                const uint32_t wt = sg_weight(ms.wmode, ms.wseed, u, v);
                bool any = false;
                for (uint32_t grp = 0; grp < ms.G; ++grp) {
                    uint64_t m = ms.inv[(uint64_t)v * ms.G + grp];
                    uint64_t better = 0;
                    unsigned long long *const bu = &ms.best[(uint64_t)u * ms.KP + grp * ms.QS];
                    unsigned long long *const bv = &ms.best[(uint64_t)v * ms.KP + grp * ms.QS];
                    while (m) {  // kSweepSlots slots at a time, their loads and updates in flight together
                        uint32_t sl[kSweepSlots], cand[kSweepSlots];
                        uint8_t kind[kSweepSlots];
                        unsigned long long du[kSweepSlots], cur[kSweepSlots];
#pragma unroll
                        for (int a = 0; a < kSweepSlots; ++a) {  // past the last: the last again
                            sl[a] = m ? (uint32_t)__builtin_ctzll(m) : sl[a ? a - 1 : 0];
                            m &= m - 1;
                        }
#pragma unroll
                        for (int a = 0; a < kSweepSlots; ++a) {
                            kind[a] = ms.kind[grp * ms.QS + sl[a]];
                            du[a] = ld_relaxed(bu + sl[a]);
                            cur[a] = ld_peek(bv + sl[a]);
                        }
#pragma unroll
                        for (int a = 0; a < kSweepSlots; ++a) {
                            const uint32_t d = hi32(du[a]);
                            const bool on = kind[a] != kQNone && d != kInf && (a == 0 || sl[a] != sl[a - 1]);
                            cand[a] = d + (kind[a] == kQUnit ? 1u : wt);
                            const unsigned long long nw = pack(cand[a], u);
                            const bool ok = on && nw < cur[a];
                            cur[a] = 0;
                            if (ok) cur[a] = atomicMin(bv + sl[a], nw);
                        }
#pragma unroll
                        for (int a = 0; a < kSweepSlots; ++a)
                            if (cand[a] < hi32(cur[a])) better |= 1ull << sl[a];
                    }
                    if (better) {
                        atomicOr(&ms.act[(uint64_t)v * ms.G + grp], better);
                        any = true;
                    }
                }
                app = any && atomicExch(&stamp[v], stamp_val) != stamp_val;
            }
            stage_push(app, v, st, io);
        }
        __builtin_amdgcn_wave_barrier();
    }
    stage_flush(st, io);
}

// Clear the masks of the vertices with a reset slot (one thread per bitmap word).
// The vertex bitmap and its coarse filter are cleared on the way.
__global__ void k_mclear_inv(uint32_t nv, uint32_t G, uint32_t *invbit, uint32_t *coarse, uint32_t cshift,
                             unsigned long long *inv) {
    const uint32_t nw = (nv + 31) / 32;
    for (uint64_t wd = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; wd < nw; wd += (uint64_t)gridDim.x * blockDim.x) {
        uint32_t bits = invbit[wd];
        if (bits) invbit[wd] = 0;
        if ((wd & ((1ull << cshift) - 1)) == 0) coarse[wd >> cshift] = 0;
        while (bits) {
            const uint32_t b = __builtin_ctz(bits);
            bits &= bits - 1;
            const uint64_t v = wd * 32 + b;
            for (uint32_t grp = 0; grp < G; ++grp) inv[v * G + grp] = 0ull;
        }
    }
}

// Initial state: every slot unreached, each query's source at distance 0 and
// active; the sources form the first frontier (each vertex once).
__global__ void k_minit_sources(MultiState ms, const uint32_t *src, uint32_t nq, uint32_t *stamp, uint32_t stamp_val,
                                uint32_t *list, uint32_t *cnt, uint32_t cap, unsigned long long *overflow) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < nq; i += gridDim.x * blockDim.x) {
        const uint32_t s = src[i], grp = i / ms.QS, slot = i % ms.QS;
        ms.best[(uint64_t)s * ms.KP + i] = pack(0, kNone);
        atomicOr(&ms.act[(uint64_t)s * ms.G + grp], 1ull << slot);
        if (atomicExch(&stamp[s], stamp_val) != stamp_val) {
            const uint32_t pos = atomicAdd(cnt, 1u);
            if (pos < cap) list[pos] = s;
            else atomicOr(overflow, 1ull);
        }
    }
}

// ---- continuous batching: queries join and leave fixed slots between round batches ----
// New slots: every vertex's word unreached, no pending or reset bits.
__global__ void k_slot_reset(MultiState ms, uint32_t nv, const uint32_t *slots, uint32_t n) {
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nv; v += (uint64_t)gridDim.x * blockDim.x) {
        for (uint32_t i = 0; i < n; ++i) {
            const uint32_t s = slots[i], grp = s / ms.QS;
            const unsigned long long keep = ~(1ull << (s % ms.QS));
            ms.best[v * ms.KP + s] = ~0ull;
            if (ms.act[v * ms.G + grp] & ~keep) ms.act[v * ms.G + grp] &= keep;
        }
    }
}
// Each new query's source at distance 0 and active, appended once to the
// frontier the next round reads (stamp_val = that round).
__global__ void k_slot_seed(MultiState ms, const uint32_t *slots, const uint32_t *src, uint32_t n, uint32_t *stamp,
                            uint32_t stamp_val, uint32_t *list, uint32_t *cnt, uint32_t cap, unsigned long long *overflow) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const uint32_t s = src[i], q = slots[i], grp = q / ms.QS, slot = q % ms.QS;
        ms.best[(uint64_t)s * ms.KP + q] = pack(0, kNone);
        atomicOr(&ms.act[(uint64_t)s * ms.G + grp], 1ull << slot);
        if (atomicExch(&stamp[s], stamp_val) != stamp_val) {
            const uint32_t pos = atomicAdd(cnt, 1u);
            if (pos < cap) list[pos] = s;
            else atomicOr(overflow, 1ull);
        }
    }
}
// Slots with work still pending (per group): the masks of the frontier the
// next round reads and of the descriptors the last round spilled.
__global__ void __launch_bounds__(kBlock) k_slot_pending(MultiState ms, const uint32_t *list, const uint32_t *cnt,
                                                         uint32_t cap, const MDesc *spill, const uint32_t *scnt,
                                                         uint32_t scap, unsigned long long *out) {
    const uint32_t n = min(*cnt, cap), ns = min(*scnt, scap);
    for (uint32_t grp = 0; grp < ms.G; ++grp) {
        unsigned long long m = 0;
        for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
            m |= ms.act[(uint64_t)list[i] * ms.G + grp];
        for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < ns; i += (uint64_t)gridDim.x * blockDim.x)
            if (spill[i].grp == grp) m |= spill[i].mask;
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) m |= __shfl_xor(m, d, kWave);
        if (lane_id() == 0 && m) atomicOr(&out[grp], m);
    }
}

// Column q of the state: distance (what = 0) or parent (what = 1).
__global__ void k_mextract(uint32_t nv, const unsigned long long *best, uint32_t KP, uint32_t q, uint32_t *out, int what) {
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nv; v += (uint64_t)gridDim.x * blockDim.x) {
        const unsigned long long b = best[v * KP + q];
        out[v] = what ? lo32(b) : hi32(b);
    }
}

}  // namespace sg

#endif
