// Pull rounds over the in-edge store (a second PMA of the same graph with
// every edge reversed, kept up to date by the same batches).
//
// A PageRank round R takes the residual of every frontier vertex u (value[u]
// += x, push p[u] = alpha * x / outdeg(u)) and delivers p[u] to every
// out-neighbour. The push form walks u's out-list with one f32 atomic add per
// edge; on R-MAT graphs the frontier is a few hub vertices that own most of
// the edges for tens of rounds, so those rounds are atomic-bound. The pull
// form walks all in-lists instead: r[v] += sum of p[u] over in-neighbours u
// in the frontier. Every destination is owned by one wave (or, for a list cut
// by a tile boundary, finished by a second pass), so no global atomic is
// issued per edge. The form is picked per round from the frontier's out-edge
// count (direction-optimising, as Beamer's BFS), on the device, so rounds stay
// queued ahead of the host.
//
// Reference: the pull functor shape of include/framework/variants/pull_functor.h:22-369
// and sync_pull_dd.cuh:1-357 (dead code there: its schedule calls do not match
// cta_scheduler_hybrid.cuh:63), and PageRank's operator (samples/hybrid_pr/hybrid_pr.cu:66-136).
#ifndef SG_PULL_H
#define SG_PULL_H

#include "sg_pma.h"

namespace sg {

// ---- PageRank rounds with an in-edge store ----------------------------------------
// A round is two kernels. k_pr_step does the round in the form its frontier
// asks for:
//   pull   (the frontier's out-edges pass the threshold) the in-lists are
//          walked; a destination whose new residual passes epsilon is taken
//          on the spot: its value, the push of the next round and the next
//          round's counts are written by the lane that finished it, so a
//          dense round makes no frontier list and the next one has no take
//          pass;
//   push   the out-lists of the frontier are walked (light tier), long ones
//          are cut into chunks;
//   take   the frontier is a list and the round would pull: its pushes are
//          taken, and the next round pulls them.
// k_pr_tail finishes it: the destinations cut by tile boundaries (pull) or the
// chunks (push), and clears the pushes the round consumed.
// A frontier is either a list with untaken residuals (after a push) or a push
// array pv (after a pull or a take): pv[rank] = push of the source of that
// rank, 0 for sources not in the frontier. Two push arrays alternate; the one
// a round writes is all zero when it starts.
//
// Appending a dense round's destinations to a frontier list would cost more
// than its edges: one counter serves all waves, and atomics on one address
// take ~12 ns each whoever issues them (a frontier of 4 M vertices, 128 a
// flush: ~0.4 ms). Here a block adds its counts once.
constexpr int kPrWaves = 16;              // one block per CU: all of its LDS serves one table of hot pushes
constexpr int kPrBlock = kPrWaves * kWave;
// The pushes of the first ranks are kept in LDS. In-lists record sources by
// out-degree rank, so they serve the in-edges that come most often (of an
// R-MAT graph of 2^22 vertices: about half); an LDS read of 64 random words
// takes a few cycles where a gather moves a 128-byte line from L2 per word.
// Measured on a pull of 65 M in-edges: 1 Ki entries 330 us, 26 Ki 270 us. A
// table costs its load in every block: at most an entry per kPrHotEdges
// in-edges of a block.
constexpr uint32_t kPrHotPlan = 31 * 1024, kPrHotSlots = 26 * 1024;
constexpr uint64_t kPrHotEdges = 4;

// ---- the pull plan: the store's in-edges as a pull reads them -----------------------
// Built after every batch and read by every pull until the next one. The
// live in-edges, without gaps and in list order (edge k), in tiles of
// kPullTile edges, ids packed at `bits` bits each: a tile is 16 * bits words,
// so every tile starts on a 64-byte boundary. Instead of offsets and degrees
// a pull reads one bit per edge (the first of its list) and the tile's first
// list; nothing it loads depends on another load, so the next tile is in
// flight while one is summed.
constexpr uint32_t kPullTile = 512;
constexpr int kPullPerLane = kPullTile / kWave;

struct PullTileMeta {
    uint32_t first;  // list (index in dst) of the tile's first edge
    uint32_t flags;  // kPullCont, kPullOn
};
constexpr uint32_t kPullCont = 1;  // the first list began in an earlier tile
constexpr uint32_t kPullOn = 2;    // the last list goes on in the next tile

struct PullPlan {
    const uint32_t *ids;        // tiles [0, split)
    const uint32_t *tail;       // tiles [split, ntiles): pinned host memory
    const uint32_t *heads;      // bit k: edge k is the first of its list
    const uint32_t *dst;        // vertices with in-edges, ascending (64 spare words)
    const PullTileMeta *meta;   // [ntiles]
    uint64_t ntiles, split, ne;
    uint32_t bits;
};
__host__ __device__ constexpr uint64_t pull_tile_words(uint32_t bits) { return (uint64_t)kPullTile / 32 * bits; }

// Lists and edges per kScanSpan vertices; clears the nh words of heads.
__global__ void __launch_bounds__(kScanBlock) k_plan_sums(uint32_t nv, const uint32_t *deg, unsigned long long *bsum,
                                                          unsigned long long *bcnt, uint32_t *heads, uint64_t nh) {
    for (uint64_t i = (uint64_t)blockIdx.x * kScanBlock + threadIdx.x; i < nh; i += (uint64_t)gridDim.x * kScanBlock) heads[i] = 0;
    __shared__ unsigned long long s_w[2][kScanBlock / kWave];
    const uint64_t base = (uint64_t)blockIdx.x * kScanSpan;
    unsigned long long x = 0, c = 0;
#pragma unroll 4
    for (uint32_t i = 0; i < kScanIters; ++i) {
        const uint64_t v = base + (uint64_t)i * kScanBlock + threadIdx.x;
        const uint32_t d = v < nv ? deg[v] : 0u;
        x += d;
        c += d != 0;
    }
    unsigned long long tx, tc;
    block_excl_scan(x, s_w[0], tx);
    block_excl_scan(c, s_w[1], tc);
    if (threadIdx.x == 0) {
        bsum[blockIdx.x] = tx;
        bcnt[blockIdx.x] = tc;
    }
}
// start[r], dst[r] of every list r, its head bit, start[lists] = ne, *nlists
// (bsum / bcnt: k_plan_sums). heads is zero before.
__global__ void __launch_bounds__(kScanBlock) k_plan_lists(uint32_t nv, const uint32_t *deg, const unsigned long long *bsum,
                                                           const unsigned long long *bcnt, unsigned long long *start,
                                                           uint32_t *dst, uint32_t *heads, uint32_t *nlists) {
    __shared__ unsigned long long s_w[6][kScanBlock / kWave];
    const uint64_t base = (uint64_t)blockIdx.x * kScanSpan;
    unsigned long long e0 = block_before(bsum, gridDim.x, s_w[4]), r0 = block_before(bcnt, gridDim.x, s_w[5]);
    for (uint32_t i = 0; i < kScanIters; ++i) {
        const uint64_t v = base + (uint64_t)i * kScanBlock + threadIdx.x;
        const uint32_t d = v < nv ? deg[v] : 0u;
        unsigned long long te, tr;
        const unsigned long long a = e0 + block_excl_scan(d, s_w[i & 1], te);
        const unsigned long long r = r0 + block_excl_scan(d != 0, s_w[2 + (i & 1)], tr);
        e0 += te;
        r0 += tr;
        if (d) {
            start[r] = a;
            dst[r] = (uint32_t)v;
            atomicOr(&heads[a >> 5], 1u << (a & 31));
        }
        if (v + 1 == nv) {
            start[r + (d != 0)] = a + d;
            *nlists = (uint32_t)(r + (d != 0));
        }
    }
}
// One thread per tile: the list of its first edge by binary search.
__global__ void k_plan_meta(uint64_t ntiles, uint64_t ne, const unsigned long long *start, const uint32_t *nlists,
                            const uint32_t *heads, PullTileMeta *meta) {
    const uint32_t n = *nlists;
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < ntiles; t += (uint64_t)gridDim.x * blockDim.x) {
        const unsigned long long e = t * kPullTile, e1 = e + kPullTile;
        uint32_t lo = 0, hi = n - 1;  // largest r with start[r] <= e
        while (lo < hi) {
            const uint32_t m = lo + (hi - lo + 1) / 2;
            if (start[m] <= e) lo = m; else hi = m - 1;
        }
        PullTileMeta x{lo, start[lo] < e ? kPullCont : 0u};
        if (e1 < ne && !((heads[e1 >> 5] >> (e1 & 31)) & 1u)) x.flags |= kPullOn;
        meta[t] = x;
    }
}

// Head bits of positions [64 * j, 64 * j + 64) of tile t (wave-uniform).
__device__ __forceinline__ uint64_t pull_heads(const uint32_t *heads, uint64_t t, int j) {
    const uint64_t w = t * (kPullTile / 32) + 2 * j;
    return ((uint64_t)heads[w + 1] << 32) | heads[w];
}

// Packed ids of tiles [t0, t1) from the store's slots, one wave per tile:
// tile t at out + (t - t0) * pull_tile_words(bits). Every word is stored
// whole (positions past the last edge are 0).
__global__ void __launch_bounds__(kBlock) k_plan_ids(GraphView g, PullPlan pl, const unsigned long long *start, uint64_t t0,
                                                     uint64_t t1, uint32_t *out) {
    __shared__ unsigned long long s_base[kWavesPerBlock][kPullTile + 1];
    __shared__ uint32_t s_id[kWavesPerBlock][kPullTile + 4];
    const uint32_t w = threadIdx.x / kWave, lane = lane_id();
    unsigned long long *const base = s_base[w];
    uint32_t *const id = s_id[w];
    const uint32_t b = pl.bits, words = (uint32_t)pull_tile_words(b);
    for (uint64_t t = t0 + (uint64_t)blockIdx.x * kWavesPerBlock + w; t < t1; t += (uint64_t)gridDim.x * kWavesPerBlock) {
        const PullTileMeta m = pl.meta[t];
        const unsigned long long e0 = t * kPullTile;
        const uint32_t ne = (uint32_t)min_u64(kPullTile, pl.ne - e0);
        uint64_t h[kPullPerLane];
        uint32_t total = 0;
#pragma unroll
        for (int j = 0; j < kPullPerLane; ++j) {
            h[j] = pull_heads(pl.heads, t, j);
            total += (uint32_t)__popcll(h[j]);
        }
        const uint32_t own0 = m.flags & kPullCont ? 0u : 1u;  // heads at or before a position, less this = its list
        const uint32_t nlists = total + 1 - own0;
        for (uint32_t i = lane; i < nlists; i += kWave)  // slot of edge k in list i: base[i] + k
            base[i] = g.off[pl.dst[m.first + i]] - start[m.first + i];
        wave_lds_sync();
        uint32_t before = 0, x[kPullPerLane];
#pragma unroll
        for (int j = 0; j < kPullPerLane; ++j) {
            const uint32_t q = j * kWave + lane;
            const uint32_t own = before + (uint32_t)__popcll(h[j] & (lanemask_lt() | (1ull << lane))) - own0;
            x[j] = q < ne ? g.col[base[own] + e0 + q] : 0u;
            before += (uint32_t)__popcll(h[j]);
        }
#pragma unroll
        for (int j = 0; j < kPullPerLane; ++j) id[j * kWave + lane] = x[j];
        wave_lds_sync();
        uint32_t *const dstw = out + (t - t0) * words;
        for (uint32_t wd = lane; wd < words; wd += kWave) {
            uint32_t word = 0, q = wd * 32 / b;  // the first id that overlaps the word
            for (int bit = (int)(q * b) - (int)(wd * 32); bit < 32; bit += (int)b, ++q)
                word |= bit >= 0 ? id[q] << bit : id[q] >> -bit;
            dstw[wd] = word;
        }
        wave_lds_sync();
    }
}

// ---- a round --------------------------------------------------------------------------
enum : int {
    kPrAuto = 0,   // by the frontier's out-edges
    kPrPull = 1,   // pull and take (one segment of a streamed pull)
    kPrAccum = 2,  // pull, residuals only (nothing taken: another pass follows)
};
// The activity threshold of a pass: none is passed when nothing is to be taken.
__device__ __forceinline__ float pr_eps(const api::PageRank &op, int mode) {
    return mode == kPrAccum ? __builtin_huge_valf() : (float)op.m_error;
}

// ---- fewer rounds: the slow part of the residual taken in one step ------------------
// A round that takes d and delivers alpha * d / outdeg leaves
//     residual = (1 - alpha) - (I - A) value
// whatever d is, so a round may take more of a residual than is there. Plain
// rounds (d = r) shrink the residual by alpha a round at best: its part along
// the graph's dominant eigenvector, eigenvalue l, shrinks by l only (R-MAT:
// 0.84), everything else much faster (0.2 to 0.4). Taking d = r / (1 - l) once
// removes that part and leaves the rest a few times larger, which two or three
// plain rounds make good. l is what the sums of the residuals taken in
// successive rounds show. Rounds of a static solve of R-MAT graphs of 2^14 to
// 2^18 vertices: 91 dense ones without, 17 with; of a snapshot: 41 and 11; the
// error against 64 bits is a fifth (solve) and the same (snapshot).
// A snapshot's seed already takes a step, with the l of the last one that did
// what it should on this engine's graph (a batch hardly changes l; without it
// a snapshot takes 16 dense rounds). It is a guess like the round count that
// sizes the batches: it decides how many rounds are run, not where they end.
//
// A step is taken when two successive ratios agree (the dominant part leads),
// kPrStepWait rounds after the last one (their plain rounds shrink what the
// step enlarged), and only while each step finds half of the residual the one
// before it found: so there are finitely many, and plain rounds between them
// converge as ever. One that left more than plain rounds would have (a graph
// with more than one slow part: a tree, a star) is the last: such graphs take
// 10 to 20 rounds more than without.
constexpr uint32_t kPrStepWait = 5;
constexpr double kPrStepAgree = 0.3;   // ratios may differ by this share of 1 - l
constexpr double kPrStepLeast = 0.3;   // below this l plain rounds are as fast
constexpr double kPrStepKeep = 0.5;    // an l above this is kept for the next snapshot's seed
// Sums over the residuals that one round took (of their magnitudes: mag).
struct PrSums {
    double sum, mag;
};
// What a round hands the next (all zero before the first).
struct PrPace {
    double sum;      // of the frontier before this one
    double ratio;    // of that one's sum to the one's before
    double found;    // magnitude at the last step (0: none yet; -1: the seed's, not known yet)
    double bound;    // what plain rounds would have left of it by now
    double l;        // the last step's l
    uint32_t since;  // rounds since then, or since the first
    uint32_t off;    // no more steps
    uint32_t pull;   // the frontier was taken in a step: only a pull finds what the step left behind
    uint32_t pad;
};

struct PrState {
    api::PageRank op;
    float *value, *res;             // committed ranks, residuals
    const float *pv_in;             // pushes of this round's frontier by rank
    float *pv_out;                  // the next round's
    float *accg;                    // partial sums of in-lists cut by tile boundaries (zero between rounds)
    const uint32_t *relabel, *unlabel;  // rank of a vertex, vertex of a rank
    const uint32_t *deg;            // out-degrees
    const uint32_t *cnt_in;         // sources in pv_in
    uint32_t *cnt_out, *cnt_zero;   // sources in pv_out; a later round's counter to clear (or null)
    uint32_t *stamp;
    uint32_t hot;  // pushes of the first ranks kept in LDS (a multiple of 4, at least 4)
    // Tiles in pinned host memory (PullPlan::split): host_waves64 / 64 of the
    // waves take those, the others the tiles in HBM, so that both run at once
    // instead of every wave stalling on the host link in turn.
    uint32_t host_waves64;
    // sums of this round's frontier, of the next (added to), of a later one (to
    // clear); pace of this round and the next. null: plain rounds.
    const PrSums *sums_in;
    PrSums *sums_out, *sums_zero;
    const PrPace *pace_in;
    PrPace *pace_out;
    double *kept;            // l for the next snapshot's seed (0: none)
    const uint32_t *in_deg;  // in-degrees
};

// What a thread took: sources and their out-edges.
struct PrTaken {
    uint32_t n = 0;
    unsigned long long edges = 0;
    float sum = 0.0f, mag = 0.0f;
};

// A destination's words.
struct PrDest {
    float res, value;
    uint32_t deg, rank;
};
__device__ __forceinline__ PrDest pr_dest(const PrState &p, uint32_t v) {
    return PrDest{p.res[v], p.value[v], p.deg[v], p.relabel[v]};
}
// CombineValueBuffer (hybrid_pr.cu:66-85) on a residual already known: commit
// it and record the push of the next round. step: the multiple of r to take.
__device__ __forceinline__ void pr_take(const PrState &p, uint32_t v, float r, const PrDest &d, float step, PrTaken &tk) {
    float x = step * r;
    float push = d.deg ? (float)(p.op.m_alpha * (double)x / (double)d.deg) : 0.0f;
    if (push == 0.0f) x = r;  // dangling: mass dropped, nothing comes back
    p.value[v] = d.value + x;
    p.res[v] = r - x;
    if (push == 0.0f) return;
    p.pv_out[d.rank] = push;
    ++tk.n;
    tk.edges += d.deg;
    tk.sum += r;
    tk.mag += fabsf(r);
}
// total: what v's in-edges delivered this round. cut: the list goes on in
// another tile; k_pr_tail finishes v from the partial sums.
__device__ __forceinline__ void pr_finish(const PrState &p, uint32_t v, float total, bool cut, const PrDest &d, float eps,
                                          float step, PrTaken &tk) {
    if (cut) {
        if (total != 0.0f) unsafeAtomicAdd(&p.accg[v], total);
        return;
    }
    const float r = total != 0.0f ? d.res + total : d.res;
    if (fabsf(r) > eps) pr_take(p, v, r, d, step, tk);
    else if (total != 0.0f) p.res[v] = r;
}

// One atomic per counter and block (kWaves waves, all threads).
template <int kWaves>
__device__ __forceinline__ void pr_count(const PrTaken &tk, const PrState &p, const PassIO &io,
                                         unsigned long long (*red)[4]) {
    const unsigned long long n = wave_sum_u64(tk.n), e = wave_sum_u64(tk.edges);
    const float s = wave_sum_f32(tk.sum), m = wave_sum_f32(tk.mag);
    const uint32_t w = threadIdx.x / kWave;
    if (lane_id() == 0) {
        red[w][0] = n;
        red[w][1] = e;
        red[w][2] = (unsigned long long)__double_as_longlong((double)s);
        red[w][3] = (unsigned long long)__double_as_longlong((double)m);
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        unsigned long long t = 0;
        for (int i = 0; i < kWaves; ++i) t += red[i][threadIdx.x];
        if (t) {
            if (threadIdx.x == 0) atomicAdd(p.cnt_out, (uint32_t)t);
            else atomicAdd(io.ecnt_out, t);
        }
    } else if (threadIdx.x < 4 && p.sums_out) {
        double t = 0.0;
        for (int i = 0; i < kWaves; ++i) t += __longlong_as_double((long long)red[i][threadIdx.x]);
        if (t != 0.0) unsafeAtomicAdd(threadIdx.x == 2 ? &p.sums_out->sum : &p.sums_out->mag, t);
    }
}

// Vertex functors of a push round: the frontier as a list (take the residual
// now), or as taken pushes by rank.
struct VPrList {
    static constexpr bool kDense = false;
    static constexpr bool kItems = false;
    api::PageRank op;
    float *value, *res;
    __device__ bool operator()(uint32_t u, uint32_t deg, uint32_t &push, bool &self) const {
        self = false;
        const auto p = op.CombineValueBuffer(u, &value[u], &res[u], deg);
        push = __float_as_uint(p.value);
        return p.scheduled;
    }
};
struct VPrRanks {
    static constexpr bool kDense = false;
    static constexpr bool kItems = true;
    const float *pv;
    const uint32_t *unlabel;
    __device__ bool item(uint32_t rank, uint32_t &u, uint32_t &push) const {
        const float x = pv[rank];
        if (x == 0.0f) return false;
        u = unlabel[rank];
        push = __float_as_uint(x);
        return true;
    }
};

// What the round does (uniform over the grid; both kernels read the same words).
struct PrRound {
    uint32_t n_list, n_pv;
    bool idle, dense, pull;
    float step = 1.0f;  // the multiple of their residuals that destinations of a pull take
    double keep = -1.0;  // a new kept l (negative: none)
    PrPace next{};
    __device__ __forceinline__ PrRound(const PrState &p, const PassIO &io, int mode) {
        n_list = mode == kPrAuto ? min(*io.in_cnt, io.in_cap) : 0u;
        n_pv = mode == kPrAuto ? *p.cnt_in : 1u;
        idle = n_list == 0 && n_pv == 0;
        dense = mode != kPrAuto || *io.ecnt_in > io.dense_thr;
        const bool paced = mode == kPrAuto && p.pace_in;
        if (paced && p.pace_in->pull) dense = true;
        pull = dense && n_pv != 0;
        if (paced && !idle) pace(p, *p.pace_in, *p.sums_in);
    }
    // Frontiers that a push made have no sums: their ratios are 0 and agree with none.
    __device__ __forceinline__ void pace(const PrState &p, const PrPace &a, const PrSums &f) {
        next = a;
        next.pull = 0;
        next.since = a.since + 1;
        next.sum = f.sum;
        next.ratio = a.sum != 0.0 ? f.sum / a.sum : 0.0;
        next.bound = a.bound * a.l;
        if (a.found < 0.0) next.found = next.bound = f.mag;
        if (!pull || a.off || next.since < kPrStepWait) return;
        if (a.found > 0.0) {
            if (f.mag > next.bound) {
                next.off = 1;
                if (*p.kept == a.l) keep = 0.0;
                return;
            }
            if (a.l > kPrStepKeep) keep = a.l;
        }
        const double l = next.ratio;  // an eigenvalue is at most alpha
        if (!(l > kPrStepLeast && l < 0.5 * (1.0 + p.op.m_alpha)) || !(fabs(l - a.ratio) < kPrStepAgree * (1.0 - l))) return;
        if (a.found > 0.0 && !(f.mag <= 0.5 * a.found)) return;
        step = (float)(1.0 / (1.0 - l));
        next.found = next.bound = f.mag;
        next.l = l;
        next.since = 0;
        next.pull = 1;
    }
};

// Tiles of a pull as the kernel walks them. Sums of a tile's lists (acc) take
// the place of its packed words.
struct alignas(16) PullWave {
    uint32_t words[kPullTile + 4];
};

// A tile whose loads are in flight.
struct PullRaw {
    lds_u32x4 w0, w1;  // packed words [4 * lane, + 4) and [256 + 4 * lane, + 4)
    uint32_t heads;    // head bits of positions [8 * lane, 8 * lane + 8)
    uint32_t dst;      // vertex of list first + lane
    PullTileMeta meta;
};
__device__ __forceinline__ PullRaw pull_load(const PullPlan &pl, uint64_t t, const PullTileMeta &m) {
    const uint32_t lane = lane_id();
    const uint32_t words = (uint32_t)pull_tile_words(pl.bits);
    const uint32_t *const src = t < pl.split ? pl.ids + t * words : pl.tail + (t - pl.split) * words;
    PullRaw r;
    // lanes past the tile's words load its last group again (not used)
    // read once per pull: non-temporal, so that the pushes keep the L2 (pull of
    // 195 M in-edges: 857 us, 895 us without)
    r.w0 = __builtin_nontemporal_load(reinterpret_cast<const lds_u32x4 *>(src + min(4 * lane, words - 4)));
    r.w1 = __builtin_nontemporal_load(reinterpret_cast<const lds_u32x4 *>(src + min(4 * (kWave + lane), words - 4)));
    r.heads = reinterpret_cast<const uint8_t *>(pl.heads)[t * kWave + lane];
    r.dst = pl.dst[m.first + lane];
    r.meta = m;
    return r;
}

// Pull over the plan's tiles: per destination, the sum of the pushes of its
// in-neighbours in the frontier.
// Ids are unpacked for positions 64 * j + lane, so that a sorted list's
// gathers fall on few lines; the pushes then change to the lane's own 8
// consecutive positions through LDS, where runs of one list are summed in
// registers and across lanes by a segmented scan: one LDS store per list.
// (Adding every push to its destination in LDS serialises on the long lists:
// 64 lanes on one address.)
__device__ __forceinline__ void pull_tiles(const PullPlan &pl, const PrState &p, TileWalk walk, const float *hot,
                                           uint32_t nhot, float eps, float step, PullWave &sh, PrTaken &tk) {
    const uint32_t lane = lane_id(), b = pl.bits;
    const uint32_t mask = b == 32 ? ~0u : (1u << b) - 1u, shift = (lane * b) & 31u;
    const uint32_t *const lw = sh.words + ((lane * b) >> 5);  // position 64 * j + lane starts 2 * b * j words on
    float *const acc = reinterpret_cast<float *>(sh.words);
    if (walk.tile() >= walk.tend) return;
    uint64_t t = walk.tile();
    PullRaw cur = pull_load(pl, t, pl.meta[t]);
    uint64_t t1 = walk.ahead(1);
    PullTileMeta m1 = pl.meta[t1 < walk.tend ? t1 : t];
    for (;;) {
        const bool more = t1 < walk.tend;
        // ids
        reinterpret_cast<lds_u32x4 *>(sh.words)[lane] = cur.w0;
        reinterpret_cast<lds_u32x4 *>(sh.words)[kWave + lane] = cur.w1;
        wave_lds_sync();
        uint32_t id[kPullPerLane];
#pragma unroll
        for (int j = 0; j < kPullPerLane; ++j) {
            const uint32_t lo = lw[2 * b * j], hi = lw[2 * b * j + 1];
            id[j] = __builtin_amdgcn_alignbit(hi, lo, shift) & mask;
        }
        wave_lds_sync();
        // pushes: from the table, or gathered (lanes served by the table read word 0)
        float c[kPullPerLane];
#pragma unroll
        for (int j = 0; j < kPullPerLane; ++j) c[j] = p.pv_in[id[j] < nhot ? 0u : id[j]];
        // lists of the tile
        const uint32_t hb = cur.heads, cnt = (uint32_t)__popc(hb);
        const uint32_t incl = wave_incl_scan(cnt);
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
        const bool cont = cur.meta.flags & kPullCont;
        const uint32_t nl = total + (cont ? 1u : 0u);
        const uint32_t v = lane < nl ? cur.dst : 0u;
        const PrDest d = pr_dest(p, v);
        // the next tile's loads, in flight from here on
        PullRaw nxt = cur;
        const uint64_t t2 = walk.ahead(2);
        if (more) {
            nxt = pull_load(pl, t1, m1);
            m1 = pl.meta[t2 < walk.tend ? t2 : t1];
        }
#pragma unroll
        for (int j = 0; j < kPullPerLane; ++j) {
            const float x = hot[min(id[j], nhot - 1)];
            c[j] = id[j] < nhot ? x : c[j];
        }
        const uint64_t left = pl.ne - t * kPullTile;
        if (left < kPullTile) {
#pragma unroll
            for (int j = 0; j < kPullPerLane; ++j)
                if (j * kWave + lane >= left) c[j] = 0.0f;
        }
        if (nl == 1) {
            float s = 0.0f;
#pragma unroll
            for (int j = 0; j < kPullPerLane; ++j) s += c[j];
            s = wave_sum_f32(s);
            if (lane == 0) pr_finish(p, v, s, cur.meta.flags != 0, d, eps, step, tk);
        } else {
#pragma unroll
            for (int j = 0; j < kPullPerLane; ++j) acc[j * kWave + lane] = c[j];
            wave_lds_sync();
            const lds_f32x4 x0 = reinterpret_cast<const lds_f32x4 *>(acc)[2 * lane];
            const lds_f32x4 x1 = reinterpret_cast<const lds_f32x4 *>(acc)[2 * lane + 1];
            wave_lds_sync();
            const float x[kPullPerLane] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
            // list (in the tile) of the position before the lane's first; -1 at a
            // tile that starts with a head
            int at = (int)(incl - cnt) - (cont ? 0 : 1);
            const int at0 = at;
            float run = 0.0f, first = 0.0f;  // open list; what the lane adds to the list that was open before it
#pragma unroll
            for (int j = 0; j < kPullPerLane; ++j) {
                if ((hb >> j) & 1u) {
                    if (at == at0) first = run;
                    else acc[at] = run;
                    ++at;
                    run = 0.0f;
                }
                run += x[j];
            }
            const float upto = wave_seg_scan(run, cnt);
            const float carry = __uint_as_float(wave_shr1(__float_as_uint(upto)));
            if (cnt && at0 >= 0) acc[at0] = first + carry;
            if (lane == kWave - 1) acc[at] = upto;
            wave_lds_sync();
            for (uint32_t i = lane; i < nl; i += kWave) {
                const bool cut = (i == 0 && cont) || (i + 1 == nl && (cur.meta.flags & kPullOn));
                if (i == lane) {
                    pr_finish(p, v, acc[i], cut, d, eps, step, tk);
                } else {
                    const uint32_t u = pl.dst[cur.meta.first + i];
                    pr_finish(p, u, acc[i], cut, pr_dest(p, u), eps, step, tk);
                }
            }
        }
        wave_lds_sync();
        if (!more) return;
        cur = nxt;
        t = t1;
        t1 = t2;
        walk.k += walk.step;
    }
}

// The same over the store's slots (merge-path tiles), for a store without a
// plan: one streamed segment of it (slots at colp[slot - slot_lo],
// destinations [dst_lo, dst_hi)), or a device budget that has no room for it.
__device__ __forceinline__ void pull_slots(const GraphView &rg, const unsigned long long *dpre, const SweepTiles &tiles,
                                           const TileWalk &walk, const uint32_t *colp, uint64_t slot_lo, uint32_t dst_lo,
                                           uint32_t dst_hi, const PrState &p, const float *hot, uint32_t nhot, float eps, float step,
                                           SweepTileLds &sh, uint32_t &n_edges, PrTaken &tk) {
    const uint32_t lane = lane_id();
    float *const acc = reinterpret_cast<float *>(sh.base);  // base[] is dead once a tile's edges are loaded
    TilePipe tp(walk, rg, dpre, tiles);
    while (tp.more) {
        uint32_t vv[kSweepPerLane];
        const TileHead h = tp.h;
        sweep_tile(rg, dpre, h, tp.pre, colp, slot_lo, dst_lo, dst_hi, sh, vv, n_edges);
        tp.advance(rg, dpre, tiles);
        float c[kSweepPerLane];
#pragma unroll
        for (int j = 0; j < kSweepPerLane; ++j) c[j] = vv[j] >= nhot && vv[j] != kGap ? p.pv_in[vv[j]] : 0.0f;
#pragma unroll
        for (int j = 0; j < kSweepPerLane; ++j)
            if (vv[j] < nhot) c[j] = hot[vv[j]];
        wave_lds_sync();
        for (uint32_t i = lane; i < h.span; i += kWave) acc[i] = 0.0f;
        wave_lds_sync();
#pragma unroll
        for (int j = 0; j < kSweepPerLane; ++j)
            if (c[j] != 0.0f) atomicAdd(&acc[sh.own[j * kWave + lane]], c[j]);
        wave_lds_sync();
        for (uint32_t i = lane; i < h.span; i += kWave) {
            const uint32_t v = h.v0 + i;
            if (v < dst_lo || v >= dst_hi) continue;
            const bool cut = i == 0 || i + 1 == h.span;  // the list may go on in a neighbouring tile
            pr_finish(p, v, acc[i], cut, pr_dest(p, v), eps, step, tk);
        }
        wave_lds_sync();
    }
}

template <bool kPlan>
struct PrShared {
    static constexpr uint32_t kHot = kPlan ? kPrHotPlan : kPrHotSlots;
    union {
        struct {
            std::conditional_t<kPlan, PullWave, SweepTileLds> tile[kPrWaves];
            alignas(16) float hot[kHot];
        };
        LightWave light[kPrWaves];
    };
    unsigned long long red[kPrWaves][4];
    uint32_t n[kPrWaves + 1];
};
static_assert(sizeof(PrShared<true>) <= 160 * 1024 && sizeof(PrShared<false>) <= 160 * 1024, "one block's LDS");

// Slots of an in-edge store (pull_slots).
struct PullSlots {
    GraphView rg;
    const unsigned long long *dpre;
    SweepTiles tiles;
    const uint32_t *colp;
    uint64_t slot_lo;
    uint32_t dst_lo, dst_hi;
    uint64_t t_begin, t_end;
};

// The round over the forward view g and the in-edge store (kPlan: its plan,
// else its slots). Bound: HBM reads of the ids and of the push lines that miss
// L2.
template <bool kPlan>
__global__ void __launch_bounds__(kPrBlock) k_pr_step(GraphView g, PullPlan pl, PullSlots sl, PrState p, PassIO io, int mode) {
    __shared__ PrShared<kPlan> sh;
    const uint32_t w = threadIdx.x / kWave;
    const PrRound rd(p, io, mode);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (io.zero_cnt) *io.zero_cnt = 0;
        if (io.heavy_zero) *io.heavy_zero = 0;
        if (io.ecnt_zero) *io.ecnt_zero = 0;
        if (p.cnt_zero) *p.cnt_zero = 0;
        if (mode == kPrAuto && p.pace_out) {
            *p.sums_zero = PrSums{};
            *p.pace_out = rd.next;
            if (rd.keep >= 0.0) *p.kept = rd.keep;
        }
        if (io.log) {  // what round R - 1 produced, and whether round R pulls
            io.log[2 * ((io.round + kRoundLog - 1) % kRoundLog)] = rd.n_list + rd.n_pv;
            io.log[2 * (io.round % kRoundLog) + 1] = rd.pull ? 1u : 0u;
        }
        if (kPlan && rd.pull) atomicAdd(io.stats + 0, (unsigned long long)pl.ne);
    }
    if (rd.idle) return;
    PrTaken tk;
    if (rd.pull) {
        const uint32_t nhot = min(p.hot, sh.kHot);  // 16-byte groups: the push arrays have a spare group
        for (uint32_t i = 4 * threadIdx.x; i < nhot; i += 4 * kPrBlock)
            *reinterpret_cast<float4 *>(&sh.hot[i]) = *reinterpret_cast<const float4 *>(&p.pv_in[i]);
        __syncthreads();
        const float eps = pr_eps(p.op, mode);
        if constexpr (kPlan) {
            TileWalk walk(0, pl.ntiles, kPrWaves);
            const uint32_t nh = max(1u, walk.step * p.host_waves64 / 64);
            if (pl.split > 0 && pl.split < pl.ntiles && nh < walk.step) {
                if (walk.k < nh) {
                    walk.t0 = pl.split;
                    walk.step = nh;
                } else {
                    walk.tend = pl.split;
                    walk.k -= nh;
                    walk.step -= nh;
                }
            }
            pull_tiles(pl, p, walk, sh.hot, nhot, eps, rd.step, sh.tile[w], tk);
        } else {
            const unsigned long long ntiles = (sl.rg.nv + sl.dpre[sl.rg.nv] + kSweepTile - 1) / kSweepTile;
            const TileWalk walk(sl.t_begin, min_u64(min_u64(sl.t_end, ntiles), sl.tiles.cap - 1), kPrWaves);
            uint32_t n_edges = 0;
            pull_slots(sl.rg, sl.dpre, sl.tiles, walk, sl.colp, sl.slot_lo, sl.dst_lo, sl.dst_hi, p, sh.hot, nhot, eps,
                       rd.step, sh.tile[w], n_edges, tk);
            const unsigned long long ne = wave_sum_u64(n_edges);
            if (lane_id() == 0 && ne) atomicAdd(io.stats + 0, ne);
        }
        if (mode != kPrAccum) pr_count<kPrWaves>(tk, p, io, sh.red);
        return;
    }
    const uint64_t gwave = (uint64_t)w * gridDim.x + blockIdx.x, nwaves = (uint64_t)gridDim.x * kPrWaves;
    if (rd.dense) {  // take the listed frontier; the next round pulls
        for (uint64_t i = gwave * kWave + lane_id(); i < rd.n_list; i += nwaves * kWave) {
            const uint32_t u = io.in_list[i];  // listed once: no other lane holds u
            const PrDest d = pr_dest(p, u);
            if (d.res != 0.0f) pr_take(p, u, d.res, d, 1.0f, tk);
        }
        pr_count<kPrWaves>(tk, p, io, sh.red);
        return;
    }
    OutStage st{sh.light[w].out, 0};
    WaveStats ws;
    const ERelax<api::PageRank> efn{p.op, p.res, p.stamp, io.round + 1, 0, 0};
    if (rd.n_pv)
        light_body(g, io, VPrRanks{p.pv_in, p.unlabel}, efn, g.nv, gwave, nwaves, sh.light[w], st, ws);
    else
        light_body(g, io, VPrList{p.op, p.value, p.res}, efn, rd.n_list, gwave, nwaves, sh.light[w], st, ws);
    block_flush<kPrWaves>(st, io, sh.n);
    stage_count_flush(st, io);
    block_stats<kPrWaves>(ws, sh.red, io.stats);
}

// Second pass of the round.
//   pull: the destinations whose lists tiles cut, each at one tile, take their
//   partial sums and are finished;
//   push: the chunks that k_pr_step cut;
//   both: the pushes the round consumed are cleared for the round after next.
template <bool kPlan>
__global__ void __launch_bounds__(kPrBlock) k_pr_tail(GraphView g, PullPlan pl, const unsigned long long *dpre,
                                                      SweepTiles tiles, PrState p, PassIO io, int mode) {
    const PrRound rd(p, io, mode);
    if (rd.idle) return;
    __shared__ uint32_t s_out[kPrWaves][kOutStage];
    __shared__ unsigned long long s_red[kPrWaves][4];
    __shared__ uint32_t s_n[kPrWaves + 1];
    const uint32_t w = threadIdx.x / kWave;
    const uint64_t first = (uint64_t)blockIdx.x * kPrBlock + threadIdx.x, stride = (uint64_t)gridDim.x * kPrBlock;
    if (rd.n_pv) {
        float *const pv = const_cast<float *>(p.pv_in);
        for (uint64_t i = first; i < g.nv; i += stride) pv[i] = 0.0f;
    }
    if (rd.pull) {
        if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(io.stats + 4, 1ull);  // a pull round
        const float eps = pr_eps(p.op, mode);
        PrTaken tk;
        auto finish = [&](uint32_t v) {
            const float total = p.accg[v];
            if (total != 0.0f) p.accg[v] = 0.0f;
            pr_finish(p, v, total, false, pr_dest(p, v), eps, rd.step, tk);
        };
        if constexpr (kPlan) {
            for (uint64_t t = first + 1; t < pl.ntiles; t += stride) {
                const PullTileMeta m = pl.meta[t], b = pl.meta[t - 1];
                // at the first tile that the list goes on into
                if ((m.flags & kPullCont) && !((b.flags & kPullCont) && b.first == m.first)) finish(pl.dst[m.first]);
            }
        } else {
            // every tile's first destination (the vertices whose lists can cross a
            // tile boundary); tile ntiles is the sentinel, vertex nv - 1
            const unsigned long long E = dpre[g.nv];
            const unsigned long long nt =
                min_u64(((unsigned long long)g.nv + E + kSweepTile - 1) / kSweepTile, tiles.cap - 1);
            for (uint64_t t = first; t <= nt; t += stride) {
                const uint32_t v = tiles.v[t];
                if (t == 0 || tiles.v[t - 1] != v) finish(v);
            }
        }
        if (mode != kPrAccum) pr_count<kPrWaves>(tk, p, io, s_red);
        return;
    }
    if (rd.dense) return;
    OutStage st{s_out[w], 0};
    WaveStats ws;
    PassIO hio = io;
    hio.hin = io.heavy;
    const uint32_t nh = min(*io.heavy_cnt, io.heavy_cap);
    const ERelax<api::PageRank> efn{p.op, p.res, p.stamp, io.round + 1, 0, 0};
    heavy_body(g, hio, efn, nh, (uint64_t)w * gridDim.x + blockIdx.x, (uint64_t)gridDim.x * kPrWaves, st, ws);
    block_flush<kPrWaves>(st, io, s_n);
    stage_count_flush(st, io);
    block_stats<kPrWaves>(ws, s_red, io.stats);
}

// Every vertex whose residual passes epsilon (kBothSigns: in either direction)
// is taken into the push array of the first round (RebuildWorklist,
// driver.cuh:654-674).
template <bool kBothSigns>
__global__ void __launch_bounds__(kPrBlock) k_pr_seed(uint32_t nv, PrState p, PassIO io) {
    __shared__ unsigned long long s_red[kPrWaves][4];
    PrTaken tk;
    const double l = kBothSigns && p.pace_out ? *p.kept : 0.0;
    const float step = (float)(1.0 / (1.0 - l));
    if (l > 0.0 && blockIdx.x == 0 && threadIdx.x == 0) {
        PrPace a{};
        a.l = l;
        a.found = -1.0;
        a.pull = 1;
        *p.pace_out = a;
    }
    for (uint64_t i = (uint64_t)blockIdx.x * kPrBlock + threadIdx.x; i < nv; i += (uint64_t)gridDim.x * kPrBlock) {
        const uint32_t v = (uint32_t)i;
        const float r = p.res[v];
        if (p.op.IsActiveNode(v, r, 0.0f) || (kBothSigns && p.op.IsActiveNode_INC(v, r, 0.0f)))
            // no pull comes to a vertex without in-edges: nothing of it may be left
            pr_take(p, v, r, pr_dest(p, v), p.in_deg[v] ? step : 1.0f, tk);
    }
    pr_count<kPrWaves>(tk, p, io, s_red);
}

// Cancel / compensate of a PageRank snapshot as pushes for a pull pass: each
// touched source records the push its CombineValueBufferAmend makes (type -1
// over the old out-degree before the commit, +1 over the new one after it).
// The pull over the in-edge store as it stands then delivers it along exactly
// the lists the push form walks (old in-lists before the store's update, new
// ones after), one read of the store instead of the hub out-lists twice.
__global__ void k_pr_amend_take(const uint32_t *list, const uint32_t *cnt, uint32_t cap, PrState p, int type, float *pv) {
    const uint32_t n = min(*cnt, cap);
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const uint32_t u = list[i];
        const auto x = p.op.CombineValueBufferAmend(u, type, &p.value[u], &p.res[u], p.deg[u]);
        if (x.scheduled) pv[p.relabel[u]] = x.value;
    }
}

// ---- pull rounds of traversal programs -------------------------------------------
// The same direction choice for min-type programs (SSSP, BFS, CC and a
// caller's operator with a MergeBuffer method). In a dense round R the round
// kernel commits every frontier vertex and records its push tagged with R
// (VCombinePull::take) instead of walking its out-list; k_trav_pull then walks
// every in-list: per destination, the offers of the in-neighbours tagged R are
// accumulated in LDS with the operator's AccumulateBuffer (from
// GetIdentityElement) and folded into the destination's buffer with
// MergeBuffer. The fold is atomic, so a destination whose in-list is split by
// a tile boundary needs no fix-up pass: each tile folds its part. Every offer
// a push round makes along u -> v is made here along the same edge, and both
// folds keep the minimum, so both directions reach the same buffers and
// schedule the same vertices.
// The pushes a dense round takes: bit u of the round's frontier bitmap and the
// push bits pv[u]. A pull pass tests the bitmap for every in-edge - one bit
// per vertex, small enough to stay in the caches (16 MiB at 2^27 vertices) -
// and reads pv only for the in-neighbours in the frontier. Two bitmaps
// alternate between rounds; round R's is cleared before round R (it last
// served round R - 2).
struct PullTake {
    uint32_t *bits;  // [ceil(nv / 32)] this round's frontier
    uint32_t *pv;    // [nv] push bits of the frontier's vertices
    __device__ void take(uint32_t u, uint32_t push) const {
        pv[u] = push;
        atomicOr(&bits[u >> 5], 1u << (u & 31));
    }
};

__device__ __forceinline__ bool pull_dense(const PassIO &io, int force) {
    return force || (io.dense_thr && io.ecnt_in && *io.ecnt_in > io.dense_thr);
}

template <class Op>
struct VCombinePull {
    static constexpr bool kDense = true;
    static constexpr bool kItems = false;
    Op op;
    typename Op::value_t *value;
    typename Op::buffer_t *buffer;
    PullTake t;
    __device__ bool operator()(uint32_t u, uint32_t deg, uint32_t &push, bool &self) const {
        self = false;
        auto p = op.CombineValueBuffer(u, &value[u], &buffer[u], deg);
        push = to_bits<typename Op::push_t>(p.value);
        return p.scheduled;
    }
    __device__ void take(uint32_t u, uint32_t push) const { t.take(u, push); }
};

template <class Op>
struct PullTrav {
    Op op;
    const uint32_t *bits;          // this round's frontier bitmap
    const uint32_t *pv;            // pushes of the frontier's vertices
    typename Op::buffer_t *buffer;
    uint32_t *stamp;               // round stamps (frontier de-duplication)
    uint32_t round;                // R
    uint32_t wmode;
    uint64_t wseed;
};

// One wave per tile of the in-edge store; colp/slot_lo as in PullSlots.
template <class Op>
__global__ void __launch_bounds__(kSweepBlock) k_trav_pull(GraphView rg, const unsigned long long *dpre, SweepTiles tiles,
                                                           const uint32_t *colp, uint64_t slot_lo, PullTrav<Op> p,
                                                           PassIO io, int force) {
    using buf_t = typename Op::buffer_t;
    if (!pull_dense(io, force)) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(io.stats + 4, 1ull);  // a pull round
    __shared__ SweepWave s_wave[kSweepWaves];
    __shared__ buf_t s_acc[kSweepWaves][kSweepTile + 1];
    __shared__ unsigned long long s_red[kSweepWaves];
    const unsigned long long E = dpre[rg.nv];
    const unsigned long long ntiles = (rg.nv + E + kSweepTile - 1) / kSweepTile;
    const uint32_t w = threadIdx.x / kWave, lane = lane_id();
    SweepWave &sh = s_wave[w];
    buf_t *const acc = s_acc[w];
    const buf_t ident = p.op.GetIdentityElement();
    OutStage st{sh.out, 0, kSweepOutStage};
    uint32_t n_edges = 0;
    unsigned long long n_done = 0;
    TilePipe tp(TileWalk(0, min_u64(ntiles, tiles.cap - 1), kSweepWaves), rg, dpre, tiles);
    while (tp.more) {
        uint32_t vv[kSweepPerLane];
        const TileHead h = tp.h;
        sweep_tile(rg, dpre, h, tp.pre, colp, slot_lo, 0u, rg.nv, sh, vv, n_edges);
        tp.advance(rg, dpre, tiles);
        uint32_t bw[kSweepPerLane];
#pragma unroll
        for (int j = 0; j < kSweepPerLane; ++j) bw[j] = vv[j] != kGap ? p.bits[vv[j] >> 5] : 0u;
        uint32_t pw[kSweepPerLane];
#pragma unroll
        for (int j = 0; j < kSweepPerLane; ++j) {
            bw[j] = (bw[j] >> (vv[j] & 31)) & 1u;
            pw[j] = bw[j] ? p.pv[vv[j]] : 0u;
        }
        for (uint32_t i = lane; i < h.span; i += kWave) acc[i] = ident;
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < kSweepPerLane; ++j) {
            if (bw[j]) {
                const uint32_t own = sh.own[j * kWave + lane];
                const uint32_t u = vv[j], v = h.v0 + own;
                const uint32_t wt = Op::kWeighted ? sg_weight(p.wmode, p.wseed, u, v) : 0u;
                p.op.AccumulateBuffer(u, v, wt, &acc[own], from_bits<typename Op::push_t>(pw[j]));
            }
        }
        __builtin_amdgcn_wave_barrier();
        for (uint32_t i0 = 0; i0 < h.span; i0 += kWave) {
            const uint32_t i = i0 + lane;
            const uint32_t v = h.v0 + i;
            bool act = false;
            if (i < h.span) {
                const buf_t a = acc[i];
                if (a != ident) {
                    act = p.op.MergeBuffer(v, &p.buffer[v], a) && atomicExch(&p.stamp[v], p.round + 1) != p.round + 1;
                    ++n_done;
                }
            }
            stage_push(act, v, st, io);
        }
        __builtin_amdgcn_wave_barrier();
    }
    stage_flush(st, io);
    stage_count_flush(st, io);
    block_count<kSweepWaves>((unsigned long long)n_edges, s_red, io.stats + 0);
    __syncthreads();
    block_count<kSweepWaves>(n_done, s_red, io.stats + 1);
}

// ---- read copies of a host-resident in-edge store ----------------------------------
// Lanes [l0, l0 + n) of the wave hold (in v) the ids of indices i0 .. i0 + n - 1
// of an array of b-bit ids packed back to back (b <= 31 here, so the words
// they cover fit one per lane; the array is zeroed before the fill). Each
// lane assembles one word from the up to 32 / b + 2 ids that overlap it;
// whole words are stored, the two end words - shared with the neighbouring
// runs - are ORed in. Every lane of the wave calls it (the ids move by
// shuffles).
__device__ __forceinline__ void pack_run(uint32_t *arr, unsigned long long i0, uint32_t l0, uint32_t n, uint32_t v,
                                         uint32_t b) {
    if (n == 0) return;
    const uint32_t lane = lane_id();
    const unsigned long long bit0 = i0 * b, bit1 = (i0 + n) * b;
    const unsigned long long w0 = bit0 >> 5, w1 = (bit1 - 1) >> 5;
    const unsigned long long w = w0 + lane;
    const unsigned long long wb = w << 5;
    unsigned long long q = wb / b;  // first id overlapping word w
    if (q < i0) q = i0;
    uint32_t word = 0;
    const uint32_t nt = 32 / b + 2;
    for (uint32_t t = 0; t < nt; ++t, ++q) {
        const long long rel = (long long)(q - i0);
        const uint32_t src = l0 + (uint32_t)(rel < (long long)n ? rel : (long long)n - 1);
        const uint32_t x = __shfl(v, (int)src, kWave);
        if (w <= w1 && q < i0 + n && q * b < wb + 32) {
            const long long sh = (long long)(q * b) - (long long)wb;
            word |= sh >= 0 ? (x << (uint32_t)sh) : (x >> (uint32_t)(-sh));
        }
    }
    if (w <= w1) {
        if (w == w0 || w == w1) atomicOr(&arr[w], word);
        else arr[w] = word;
    }
}

// Store the ids of lanes [l0, l0 + n) at indices i0 .. of a copy: packed at
// b bits, or plain words (b = 32).
__device__ __forceinline__ void copy_run(uint32_t *arr, unsigned long long i0, uint32_t l0, uint32_t n, uint32_t v,
                                         uint32_t b) {
    if (b == 32) {
        const uint32_t lane = lane_id();
        if (lane >= l0 && lane < l0 + n) arr[i0 + (lane - l0)] = v;
    } else {
        pack_run(arr, i0, l0, n, v, b);
    }
}

// HBM copy of the store's leading live edges, read from the store in host
// memory through the tile sweep (live slots only, coalesced): copy id k = live
// edge k (merge-path order) for k < mlive. g must carry no copy itself, and a
// packed array must be zero. The tiles of a wave are in edge order, so it
// stops at its first tile past mlive.
__global__ void __launch_bounds__(kSweepBlock) k_mirror_fill(GraphView g, const unsigned long long *dpre, SweepTiles tiles,
                                                             uint32_t *mirror, uint64_t mlive, uint32_t b) {
    __shared__ SweepWave s_wave[kSweepWaves];
    const unsigned long long E = dpre[g.nv];
    const unsigned long long ntiles = min_u64((g.nv + E + kSweepTile - 1) / kSweepTile, tiles.cap - 1);
    const uint32_t w = threadIdx.x / kWave;
    SweepWave &sh = s_wave[w];
    uint32_t n_edges = 0;
    TilePipe tp(TileWalk(0, ntiles, kSweepWaves), g, dpre, tiles);
    while (tp.more) {
        const TileHead h = tp.h;
        if (h.e0 >= mlive) break;
        uint32_t vv[kSweepPerLane];
        sweep_tile(g, dpre, h, tp.pre, g.col, 0, 0u, g.nv, sh, vv, n_edges);
        tp.advance(g, dpre, tiles);
#pragma unroll
        for (int j = 0; j < kSweepPerLane; ++j) {
            // positions [j * 64, j * 64 + n) of the tile: edges k0 .. k0 + n - 1
            const uint32_t pj = j * kWave;
            const unsigned long long k0 = h.e0 + pj;
            const uint32_t n = h.ne > pj && k0 < mlive ? (uint32_t)min_u64(min(h.ne - pj, (uint32_t)kWave), mlive - k0) : 0u;
            if (n) copy_run(mirror, k0, 0, n, vv[j], b);
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// ---- traversal recompute from the in-lists of invalidated vertices -------------
// After deletions, every invalidated vertex v must see the best value any
// in-neighbour u offers: PushValue(best(u)) + w(u, v) (for CC the label of u).
// The forward form sweeps every live edge and relaxes those whose target is
// invalidated (the reference re-pushes from every vertex:
// RelaxCTADB_all_vertices, sync_push_dd.cuh:1470-1557); with an in-edge store
// only the in-lists of the invalidated vertices are read. A round kernel walks
// those lists (in-store view, the invalidated vertices as items) with this
// functor; whatever improves v appends v itself.
template <class Op>
struct EPullSeed {
    static constexpr bool kAppendSource = true;
    static constexpr int kUpdates = kIlp;
    Op op;
    typename Op::buffer_t *buffer;
    uint32_t *stamp;
    uint32_t stamp_val;
    uint32_t wmode;
    uint64_t wseed;
    const uint32_t *unlabel;  // vertex of each in-list id (null: ids are vertices)
    __device__ uint32_t vertex(uint32_t x) const { return unlabel ? unlabel[x] : x; }
    __device__ uint64_t load(uint32_t x) const { return ld_peek(&buffer[vertex(x)]); }
    // v: the invalidated vertices whose in-lists are walked; x: in-list entries
    template <int N>
    __device__ __forceinline__ void apply_n(const uint32_t (&v)[N], const uint32_t (&x)[N], const uint32_t (&)[N],
                                            const uint64_t (&bu)[N], bool (&enq)[N]) const {
        uint32_t u[N], w[N];
#pragma unroll
        for (int j = 0; j < N; ++j) {
            u[j] = x[j] != kGap ? vertex(x[j]) : 0u;
            w[j] = Op::kWeighted ? sg_weight(wmode, wseed, u[j], v[j]) : 0u;
            enq[j] = x[j] != kGap && op.MayImprove(u[j], w[j], op.PushValue(bu[j]), ld_peek(&buffer[v[j]]));
        }
#pragma unroll
        for (int j = 0; j < N; ++j)
            if (enq[j])
                enq[j] = op.AccumulateBuffer(u[j], v[j], w[j], &buffer[v[j]], op.PushValue(bu[j])) &&
                         atomicExch(&stamp[v[j]], stamp_val) != stamp_val;
    }
};

// The vertices of a bitmap as a list (one thread per word; one atomic per wave).
__global__ void __launch_bounds__(kBlock) k_bits_to_list(uint32_t nv, const uint32_t *bits, uint32_t *list, uint32_t *cnt,
                                                         uint32_t cap, unsigned long long *overflow) {
    const uint32_t nw = (nv + 31) / 32;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t base = (uint64_t)blockIdx.x * blockDim.x; base < nw; base += stride) {
        const uint64_t wd = base + threadIdx.x;
        uint32_t b = wd < nw ? bits[wd] : 0u;
        if (wd + 1 == nw && (nv & 31)) b &= (1u << (nv & 31)) - 1;
        const uint32_t c = __popc(b);
        const uint32_t incl = wave_incl_scan(c);
        const uint32_t total = __shfl(incl, kWave - 1, kWave);
        if (total == 0) continue;
        uint32_t at = 0;
        if (lane_id() == 0) at = atomicAdd(cnt, total);
        at = __shfl(at, 0, kWave) + incl - c;
        while (b) {
            const uint32_t v = (uint32_t)wd * 32 + __builtin_ctz(b);
            b &= b - 1;
            if (at < cap) list[at] = v;
            else atomicOr(overflow, 1ull);
            ++at;
        }
    }
}

// Out-edges of a frontier list (the first round's direction choice).
__global__ void __launch_bounds__(kBlock) k_list_degsum(const uint32_t *list, const uint32_t *cnt, uint32_t cap,
                                                        const uint32_t *deg, unsigned long long *out) {
    const uint32_t n = min(*cnt, cap);
    unsigned long long s = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        s += deg[list[i]];
    s = wave_sum_u64(s);
    if (lane_id() == 0 && s) atomicAdd(out, s);
}

}  // namespace sg

#endif
