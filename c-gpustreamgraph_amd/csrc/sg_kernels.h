// Device building blocks of the engine: wave64 primitives, the frontier
// expansion kernels (light + heavy tiers) and the per-vertex / per-edge
// functors that specialise them for each phase.
//
// Reference counterparts:
//   frontier append          groute::dev::Queue::append (groute/device/queue.cuh:84-88):
//                            there one atomicAdd per item; here one per wave (ballot).
//   neighbour scheduling     CTAWorkSchedulerNew::schedule (groute/device/cta_scheduler_hybrid.cuh:59-245):
//                            there block-owner election for huge lists + warp loops;
//                            here a wave stages 64 lists in LDS and walks their union,
//                            and lists longer than kHeavyDeg become fixed-size chunks
//                            taken by any wave (second kernel).
//   relax                    RelaxCTADB (framework/variants/sync_push_dd.cuh:180-268) +
//                            PushFunctorDB (framework/variants/push_functor.h:252-321)
#ifndef SG_KERNELS_H
#define SG_KERNELS_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "sg_operators.h"
#include "../host/sg_rng.h"

namespace sg {

constexpr uint32_t kGap = 0xFFFFFFFFu;       // empty PMA slot (csr_graph.cuh:416, memset -1)
constexpr int kWave = 64;
constexpr int kBlock = 256;                  // threads per block of the expansion kernels
constexpr int kWavesPerBlock = kBlock / kWave;
constexpr uint32_t kHeavyDeg = 2048;         // lists longer than this go to the heavy tier
constexpr uint32_t kChunk = 1024;            // edges per heavy descriptor

// A kChunk-edge piece of an adjacency list: (start << kLenBits | len - 1),
// source, push value bits.
constexpr uint32_t kLenBits = 11;
struct HeavyDesc {
    uint64_t start_len;
    uint32_t u;
    uint32_t push;
};

// Graph as seen by kernels: PMA CSR with per-vertex gaps.
struct GraphView {
    uint32_t nv;
    const uint64_t *off;  // [nv + 1], off[nv] = capacity
    const uint32_t *deg;  // [nv]
    const uint32_t *col;  // [capacity], kGap in unused slots (HBM, or pinned host memory)
    // HBM edge cache (null when unused): copies of the lists of hot vertices.
    // A list start s >= cap addresses ccol[s - cap].
    const uint32_t *ccol;
    const uint64_t *coff;  // [nv] start of v's copy in ccol, ~0 = not cached
    uint64_t cap;
    uint8_t *hot;          // [nv] activations this snapshot (null when unused)
    // HBM copy of the live edges [0, mlive) of a col in pinned host memory, in
    // live-edge order (edge k of the merge path, vertex by vertex: no gaps),
    // ids packed at mbits bits each (packed_at), read by the tile sweeps; list
    // walks and updates use col. mlive = 0: none.
    const uint32_t *mirror;
    uint64_t mlive;
    uint32_t mbits;  // bits per packed id (32: plain words)
};

// Id i of an array of b-bit ids packed back to back from bit 0 (b in [1, 32];
// the array holds one spare word past its last id).
__device__ __forceinline__ uint32_t packed_at(const uint32_t *p, unsigned long long i, uint32_t b) {
    const unsigned long long bit = i * b;
    const unsigned long long w = bit >> 5;
    const uint64_t x = ((uint64_t)p[w + 1] << 32) | p[w];
    const uint32_t v = (uint32_t)(x >> (bit & 31u));
    return b == 32 ? v : v & ((1u << b) - 1u);
}

// Where a relax walk reads u's list: its cached copy when there is one.
__device__ __forceinline__ uint64_t list_start(const GraphView &g, uint32_t u) {
    if (g.coff) {
        const uint64_t c = g.coff[u];
        if (c != ~0ull) return g.cap + c;
    }
    return g.off[u];
}
__device__ __forceinline__ uint32_t edge_at(const GraphView &g, uint64_t s) {
    const uint32_t *const p = s < g.cap ? g.col + s : g.ccol + (s - g.cap);
    return *p;
}
// Activation count of the cache's hotness window (non-atomic and saturating,
// like the reference's hotness[0]++ in RelaxCTADB, sync_push_dd.cuh:196-230).
__device__ __forceinline__ void count_hot(const GraphView &g, uint32_t u) {
    if (g.hot) {
        const uint8_t h = g.hot[u];
        if (h < 255) g.hot[u] = h + 1;
    }
}

// Where a pass reads its work items and appends the vertices it activates.
struct PassIO {
    const uint32_t *in_list;  // explicit list, or null for the range [range_lo, range_lo + range_n)
    const uint32_t *in_cnt;   // device count of in_list
    uint32_t in_cap;          // capacity of in_list
    uint32_t range_lo, range_n;
    uint32_t *out_list;       // next frontier
    uint32_t *out_cnt;
    uint32_t out_cap;
    uint32_t *zero_cnt;       // frontier counter this pass clears for a later round (or null)
    HeavyDesc *heavy;         // descriptors this pass spills (processed by the next pass)
    uint32_t *heavy_cnt;
    const HeavyDesc *hin;     // descriptors spilled by the previous pass (or null)
    const uint32_t *hin_cnt;
    uint32_t *heavy_zero;     // descriptor counter this pass clears for a later round (or null)
    uint32_t heavy_cap;
    uint32_t budget;          // light-tier edges per 64-item batch of a wave
    uint32_t heavy_deg;       // lists longer than this always go to the heavy tier
    unsigned long long *stats;  // [0] edges (light), [1] vertices, [2] edges (heavy), [3] overflow
    uint32_t *log;            // round log (or null): round R records the counts its inputs had
    uint32_t round;           // R, for the log
    // Direction choice (PageRank with an in-edge store): ecnt_in holds the
    // out-edges of this round's frontier; above dense_thr the round is dense
    // and the vertex functor only takes the frontier's pushes (a pull pass
    // over the in-edges delivers them). Appended vertices add their out-degree
    // (fdeg) to ecnt_out. All null / 0 when the engine has no such choice.
    const unsigned long long *ecnt_in;
    unsigned long long *ecnt_out;
    unsigned long long *ecnt_zero;  // edge counter this pass clears for a later round (or null)
    const uint32_t *fdeg;
    unsigned long long dense_thr;
};
constexpr uint32_t kRoundLog = 256;  // entries of the round log ring

// ---- wave64 primitives -----------------------------------------------------
__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }
__device__ __forceinline__ uint64_t lanemask_lt() {
    const uint32_t l = lane_id();
    return l ? (~0ull >> (64 - l)) : 0ull;
}
// Lane moves on the VALU (DPP): lane i takes x of another lane of its row of 16
// (row_shr) or of an earlier row's last lane (row_bcast); lanes without a
// source, or outside kRowMask's rows, take `old`. A shuffle goes through the
// LDS crossbar instead. Every lane of the wave must be active.
template <int kCtrl, int kRowMask>
__device__ __forceinline__ uint32_t dpp_mov(uint32_t old, uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)x, kCtrl, kRowMask, 0xf, false);
}
constexpr int kDppRowShr = 0x110, kDppWaveShr1 = 0x138, kDppBcast15 = 0x142, kDppBcast31 = 0x143;
// x of the previous lane (lane 0: 0)
__device__ __forceinline__ uint32_t wave_shr1(uint32_t x) { return dpp_mov<kDppWaveShr1, 0xf>(0u, x); }
// Six steps of an inclusive scan: step(shift lanes within a row, then across rows).
#define SG_DPP_SCAN(STEP)      \
    STEP(kDppRowShr + 1, 0xf)  \
    STEP(kDppRowShr + 2, 0xf)  \
    STEP(kDppRowShr + 4, 0xf)  \
    STEP(kDppRowShr + 8, 0xf)  \
    STEP(kDppBcast15, 0xa)     \
    STEP(kDppBcast31, 0xc)
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x) {
#define SG_STEP(C, M) x += dpp_mov<C, M>(0u, x);
    SG_DPP_SCAN(SG_STEP)
#undef SG_STEP
    return x;
}
__device__ __forceinline__ unsigned long long wave_incl_scan(unsigned long long x) {
#define SG_STEP(C, M)                                                                                   \
    x += ((unsigned long long)dpp_mov<C, M>(0u, (uint32_t)(x >> 32)) << 32) | dpp_mov<C, M>(0u, (uint32_t)x);
    SG_DPP_SCAN(SG_STEP)
#undef SG_STEP
    return x;
}
__device__ __forceinline__ uint32_t wave_max_scan(uint32_t x) {
#define SG_STEP(C, M) x = max(x, dpp_mov<C, M>(0u, x));
    SG_DPP_SCAN(SG_STEP)
#undef SG_STEP
    return x;
}
// Inclusive segmented sum: lanes with head != 0 start a segment.
__device__ __forceinline__ float wave_seg_scan(float x, uint32_t head) {
#define SG_STEP(C, M)                                                    \
    {                                                                    \
        const float y = __uint_as_float(dpp_mov<C, M>(0u, __float_as_uint(x))); \
        const uint32_t h = dpp_mov<C, M>(0u, head);                      \
        x = head ? x : x + y;                                            \
        head |= h;                                                       \
    }
    SG_DPP_SCAN(SG_STEP)
#undef SG_STEP
    return x;
}
// Sum over the wave (in every lane).
__device__ __forceinline__ float wave_sum_f32(float x) {
#define SG_STEP(C, M) x += __uint_as_float(dpp_mov<C, M>(0u, __float_as_uint(x)));
    SG_DPP_SCAN(SG_STEP)
#undef SG_STEP
    return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(x), kWave - 1));
}
// LDS of one wave: what its lanes stored before is read by the loads after
// (the hardware keeps a wave's LDS operations in order; the compiler must too).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// Wave-aggregated append: one atomicAdd per wave. Every active lane of the
// wave must call it (pred may differ per lane).
__device__ __forceinline__ void wave_append(bool pred, uint32_t item, uint32_t *list, uint32_t *cnt,
                                            uint32_t cap, unsigned long long *overflow) {
    const uint64_t m = __ballot(pred);
    if (m == 0) return;
    const uint32_t leader = (uint32_t)__ffsll((unsigned long long)m) - 1;
    uint32_t base = 0;
    if (lane_id() == leader) base = atomicAdd(cnt, (uint32_t)__popcll(m));
    base = __shfl(base, (int)leader, kWave);
    if (pred) {
        const uint32_t pos = base + (uint32_t)__popcll(m & lanemask_lt());
        if (pos < cap) list[pos] = item;
        else atomicOr(overflow, 1ull);
    }
}
// Block-wide append: one global atomic per block and call instead of one per
// wave (per-wave atomics on one counter serialise across the chip). Every
// thread of a kBlock-thread block must call it; returns the block's count.
struct BlockAppend {
    uint32_t wsum[kWavesPerBlock];
    uint32_t base, total;
};
__device__ __forceinline__ uint32_t block_append(bool pred, uint32_t item, uint32_t *list, uint32_t *cnt, uint32_t cap,
                                                 unsigned long long *overflow, BlockAppend &sh) {
    const uint64_t m = __ballot(pred);
    const uint32_t w = threadIdx.x / kWave;
    if (lane_id() == 0) sh.wsum[w] = (uint32_t)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int i = 0; i < kWavesPerBlock; ++i) {
            const uint32_t c = sh.wsum[i];
            sh.wsum[i] = t;  // exclusive offset of each wave
            t += c;
        }
        sh.total = t;
        sh.base = t ? atomicAdd(cnt, t) : 0u;
    }
    __syncthreads();
    if (pred) {
        const uint32_t pos = sh.base + sh.wsum[w] + (uint32_t)__popcll(m & lanemask_lt());
        if (pos < cap) list[pos] = item;
        else atomicOr(overflow, 1ull);
    }
    const uint32_t total = sh.total;
    __syncthreads();  // the LDS words are reused by the next call
    return total;
}

__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long x) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) x += __shfl_xor(x, d, kWave);
    return x;
}

// 64-bit minimum on integers (the generic min template goes through double).
__host__ __device__ __forceinline__ unsigned long long min_u64(unsigned long long a, unsigned long long b) {
    return a < b ? a : b;
}

// Coarse filter over a vertex bitmap: one bit per 2^shift vertices with
// shift = max(6, ceil(log2 nv) - 16), so the filter has at most 65536 bits
// (kFilterWords words) and a block can keep a copy in LDS.
constexpr uint32_t kFilterWords = 2048;
__host__ __device__ inline uint32_t coarse_shift_for(uint32_t nv) {
    uint32_t s = 6;
    while ((((uint64_t)nv + (1ull << s) - 1) >> s) > 32ull * kFilterWords) ++s;
    return s;
}
__host__ __device__ inline uint32_t coarse_words(uint32_t nv, uint32_t shift) {
    return (uint32_t)(((((uint64_t)nv + (1ull << shift) - 1) >> shift) + 31) / 32);
}
__device__ __forceinline__ void coarse_mark(uint32_t *coarse, uint32_t shift, uint32_t v) {
    atomicOr(&coarse[v >> (shift + 5)], 1u << ((v >> shift) & 31));
}
__device__ __forceinline__ bool coarse_test(const uint32_t *coarse, uint32_t shift, uint32_t v) {
    return (coarse[v >> (shift + 5)] >> ((v >> shift) & 31)) & 1u;
}

template <class T> __device__ __forceinline__ uint32_t to_bits(T x);
template <> __device__ __forceinline__ uint32_t to_bits<uint32_t>(uint32_t x) { return x; }
template <> __device__ __forceinline__ uint32_t to_bits<float>(float x) { return __float_as_uint(x); }
template <class T> __device__ __forceinline__ T from_bits(uint32_t x);
template <> __device__ __forceinline__ uint32_t from_bits<uint32_t>(uint32_t x) { return x; }
template <> __device__ __forceinline__ float from_bits<float>(uint32_t x) { return __uint_as_float(x); }

__device__ __forceinline__ uint64_t ld_relaxed(const unsigned long long *p) {
    return __hip_atomic_load(const_cast<unsigned long long *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Plain (cacheable) load for pre-tests of values that only decrease during a
// phase: a stale copy is never below the current value, so a pre-test that
// passes on the current value also passes on the copy.
__device__ __forceinline__ uint64_t ld_peek(const unsigned long long *p) { return *p; }

// ---- per-wave output staging -------------------------------------------------
// Activated vertices are collected in a per-wave LDS buffer and appended to
// the global frontier kOutStage at a time: one atomicAdd per flush instead of
// one per wave-iteration, and coalesced stores.
constexpr uint32_t kOutStage = 512;
constexpr uint32_t kWaveBudget = 1024;  // default light-tier edges per 64-item batch of a wave
constexpr int kIlp = 8;                 // edges per lane per iteration

struct OutStage {
    uint32_t *buf;              // this wave's LDS slice [cap]
    uint32_t n;                 // wave-uniform fill
    uint32_t cap = kOutStage;   // slice size (>= kWave)
    unsigned long long fedges = 0;  // per lane: out-degrees of the items it appended (io.fdeg)
};

__device__ __forceinline__ void stage_flush(OutStage &st, const PassIO &io) {
    if (st.n == 0) return;
    uint32_t base = 0;
    if (lane_id() == 0) base = atomicAdd(io.out_cnt, st.n);
    base = __shfl(base, 0, kWave);
    for (uint32_t i = lane_id(); i < st.n; i += kWave) {
        const uint32_t pos = base + i;
        if (pos < io.out_cap) io.out_list[pos] = st.buf[i];
        else atomicOr(io.stats + 3, 1ull);
    }
    wave_lds_sync();  // read by every lane before the slice fills again
    st.n = 0;
}

__device__ __forceinline__ void stage_push(bool pred, uint32_t item, OutStage &st, const PassIO &io) {
    const uint64_t m = __ballot(pred);
    if (m == 0) return;
    if (io.fdeg && pred) st.fedges += io.fdeg[item];
    const uint32_t c = (uint32_t)__popcll(m);
    if (st.n + c > st.cap) stage_flush(st, io);
    if (pred) st.buf[st.n + (uint32_t)__popcll(m & lanemask_lt())] = item;
    st.n += c;
}

// item[j] of the lanes with pred[j], N per lane.
template <int N>
__device__ __forceinline__ void stage_push_n(const bool (&pred)[N], const uint32_t (&item)[N], OutStage &st,
                                             const PassIO &io) {
    uint32_t c = 0;
#pragma unroll
    for (int j = 0; j < N; ++j) c += pred[j] ? 1u : 0u;
    if (__ballot(c != 0) == 0) return;
    if (io.fdeg) {
#pragma unroll
        for (int j = 0; j < N; ++j)
            if (pred[j]) st.fedges += io.fdeg[item[j]];
    }
    const uint32_t incl = wave_incl_scan(c);
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
    if (st.n + total > st.cap) stage_flush(st, io);
    if (total > st.cap) {  // more than a slice at once: straight to the list
        uint32_t pos = 0;
        if (lane_id() == 0) pos = atomicAdd(io.out_cnt, total);
        pos = (uint32_t)__builtin_amdgcn_readfirstlane((int)pos) + incl - c;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            if (!pred[j]) continue;
            if (pos < io.out_cap) io.out_list[pos] = item[j];
            else atomicOr(io.stats + 3, 1ull);
            ++pos;
        }
        return;
    }
    uint32_t at = st.n + incl - c;
#pragma unroll
    for (int j = 0; j < N; ++j)
        if (pred[j]) st.buf[at++] = item[j];
    st.n += total;
}

// The waves of a block append what they still hold with one atomic (every
// thread of a block of kWaves waves; s_n: kWaves + 1 words).
template <int kWaves>
__device__ __forceinline__ void block_flush(OutStage &st, const PassIO &io, uint32_t *s_n) {
    const uint32_t w = threadIdx.x / kWave;
    if (lane_id() == 0) s_n[w] = st.n;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int i = 0; i < kWaves; ++i) {
            const uint32_t c = s_n[i];
            s_n[i] = t;
            t += c;
        }
        s_n[kWaves] = t ? atomicAdd(io.out_cnt, t) : 0u;
    }
    __syncthreads();
    const uint32_t base = s_n[kWaves] + s_n[w];
    for (uint32_t i = lane_id(); i < st.n; i += kWave) {
        if (base + i < io.out_cap) io.out_list[base + i] = st.buf[i];
        else atomicOr(io.stats + 3, 1ull);
    }
    st.n = 0;
}

// One atomic per wave: the out-edges of what the wave appended (io.ecnt_out).
__device__ __forceinline__ void stage_count_flush(OutStage &st, const PassIO &io) {
    if (!io.ecnt_out) return;
    const unsigned long long t = wave_sum_u64(st.fedges);
    if (lane_id() == 0 && t) atomicAdd(io.ecnt_out, t);
    st.fedges = 0;
}

// Per-wave counters, reduced per block at the end of a kernel.
struct WaveStats {
    unsigned long long edges = 0, verts = 0, hedges = 0, cedges = 0;
};

// LDS of the light tier (per wave). own: list of each of the kIlp * 64 edges
// of a step.
struct StagedList {
    uint64_t base;  // slot of edge k of the staged union: base + k
    uint32_t src, push;
};
struct alignas(16) LightWave {
    StagedList list[kWave];
    uint8_t own[kIlp * kWave];
    uint32_t out[kOutStage];
};
// LDS accesses of another width than the array's
typedef uint32_t lds_u32x2 __attribute__((ext_vector_type(2), may_alias));

// One step of edges: their updates, EFn::kUpdates of a lane at a time, then what
// they activate. The loads of a step are in flight together, and so are the
// destination updates and the stamp exchanges of a group.
template <class EFn>
__device__ __forceinline__ void apply_edges(const PassIO &io, const EFn &efn, const uint32_t (&src)[kIlp],
                                            const uint32_t (&v)[kIlp], const uint32_t (&push)[kIlp], OutStage &st) {
    constexpr int kN = EFn::kUpdates;
    uint64_t peek[kIlp];
#pragma unroll
    for (int j = 0; j < kIlp; ++j) peek[j] = efn.load(v[j] != kGap ? v[j] : 0u);
    bool enq[kIlp];
#pragma unroll
    for (int h = 0; h < kIlp; h += kN) {
        uint32_t s[kN], x[kN], p[kN];
        uint64_t b[kN];
        bool q[kN];
#pragma unroll
        for (int j = 0; j < kN; ++j) {
            s[j] = src[h + j];
            x[j] = v[h + j];
            p[j] = push[h + j];
            b[j] = peek[h + j];
        }
        efn.template apply_n<kN>(s, x, p, b, q);
#pragma unroll
        for (int j = 0; j < kN; ++j) enq[h + j] = q[j];
    }
    if constexpr (EFn::kAppendSource) stage_push_n<kIlp>(enq, src, st, io);
    else stage_push_n<kIlp>(enq, v, st, io);
}

// Edge loop of one wave over the union of its lanes' lists: lane i's list has
// d edges from slot start, the union's edges [excl, excl + d); total edges.
// kIlp edges per lane per step. The list of each edge of a step comes from
// marks at the list starts, filled forward by a maximum scan (a binary search
// per edge is six dependent LDS reads, and was half of a step).
template <class EFn>
__device__ __forceinline__ void walk_staged(const GraphView &g, const PassIO &io, const EFn &efn, uint32_t total,
                                            uint32_t excl, uint32_t d, uint64_t start, uint32_t src_l, uint32_t push_l,
                                            LightWave &sh, OutStage &st) {
    if (total == 0) return;
    const uint32_t lane = lane_id();
    sh.list[lane] = StagedList{start - excl, src_l, push_l};
    lds_u32x2 *const own8 = reinterpret_cast<lds_u32x2 *>(sh.own) + lane;
    for (uint32_t k0 = 0; k0 < total; k0 += kIlp * kWave) {
        *own8 = lds_u32x2{0u, 0u};
        wave_lds_sync();
        if (d && excl > k0 && excl - k0 < kIlp * kWave) sh.own[excl - k0] = (uint8_t)lane;
        // the list open at k0: the last non-empty one that starts at or before it
        const uint32_t open = 63u - (uint32_t)__builtin_clzll(__ballot(d != 0 && excl <= k0) | 1ull);
        wave_lds_sync();
        lds_u32x2 o = *own8;
        uint32_t m = 0;
        uint32_t b[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            m = max(m, (o[j / 4] >> (8 * (j & 3))) & 0xFFu);
            b[j] = m;
        }
        const uint32_t before = max(wave_shr1(wave_max_scan(m)), open);
        o = lds_u32x2{0u, 0u};
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j / 4] |= max(b[j], before) << (8 * (j & 3));
        *own8 = o;
        wave_lds_sync();
        uint32_t v[kIlp], src[kIlp], push[kIlp];
        uint64_t slot[kIlp];
#pragma unroll
        for (int j = 0; j < kIlp; ++j) {
            const uint32_t k = min(k0 + j * kWave + lane, total - 1);
            const StagedList l = sh.list[sh.own[min(j * kWave + lane, total - 1 - k0)]];
            src[j] = l.src;
            push[j] = l.push;
            slot[j] = l.base + k;
        }
#pragma unroll
        for (int j = 0; j < kIlp; ++j) v[j] = edge_at(g, slot[j]);
#pragma unroll
        for (int j = 0; j < kIlp; ++j)
            if (k0 + j * kWave + lane >= total) v[j] = kGap;
        wave_lds_sync();
        apply_edges(io, efn, src, v, push, st);
    }
}

// Power of two in [1, kWave] at least ceil(n / nwaves).
__device__ __forceinline__ uint32_t light_width(uint32_t n, uint64_t nwaves) {
    const uint64_t q = (n + nwaves - 1) / nwaves;
    uint32_t per = 1;
    while (per < (uint32_t)kWave && per < q) per <<= 1;
    return per;
}

// Light tier body: waves [gwave, +nwaves) take up to 64 work items at a time
// (light_width), run the vertex functor, and walk the scheduled lists that
// fit the wave budget; longer lists, and lists past the budget, are cut into
// kChunk-edge descriptors for the heavy tier, so no wave carries more than
// budget + heavy_deg edges per batch.
template <class VFn, class EFn>
__device__ __forceinline__ void light_body(const GraphView &g, const PassIO &io, const VFn &vfn, const EFn &efn,
                                           uint32_t n, uint64_t gwave, uint64_t nwaves, LightWave &sh, OutStage &st,
                                           WaveStats &ws) {
    const uint32_t lane = lane_id();
    // frontier vertices per wave batch: 64 when the frontier fills every wave,
    // fewer (a power of two, down to 1) when it is small, so that its lists
    // spread over all waves instead of a few waves walking 64 lists each
    const uint32_t per = light_width(n, nwaves);
    // dense round: the functor records each frontier vertex's push for the
    // pull pass and no list is walked here
    bool dense = false;
    if constexpr (VFn::kDense) dense = io.dense_thr && io.ecnt_in && *io.ecnt_in > io.dense_thr;
    for (uint64_t base = gwave * per; base < n; base += nwaves * per) {
        const uint64_t idx = base + lane;
        uint32_t u = 0, d = 0, push = 0;
        uint64_t start = 0;
        bool self = false, sched = false;
        if constexpr (VFn::kItems) {  // the functor names the vertex of item idx and its push
            if (lane < per && idx < n) sched = vfn.item((uint32_t)idx, u, push);
            if (__ballot(sched) == 0) continue;
            if (sched) {
                d = g.deg[u];
                start = list_start(g, u);
            }
        } else if (lane < per && idx < n) {
            u = io.in_list ? io.in_list[idx] : io.range_lo + (uint32_t)idx;
            const uint32_t du = g.deg[u];
            sched = vfn(u, du, push, self);
            if constexpr (VFn::kDense) {
                if (dense) {
                    if (sched && du) {
                        vfn.take(u, push);
                        count_hot(g, u);  // a pusher: its list is hot for the HBM edge cache
                    }
                    sched = false;
                }
            }
            if (sched && du) {
                d = du;
                start = list_start(g, u);
                count_hot(g, u);
            }
        }
        stage_push(self, u, st, io);
        ws.verts += sched ? 1 : 0;
        const uint32_t incl0 = wave_incl_scan(d);
        const bool heavy = d > io.heavy_deg || (d > 0 && incl0 > io.budget);
        const uint32_t nch = heavy ? (d + kChunk - 1) / kChunk : 0;
        const uint32_t nch_incl = wave_incl_scan(nch);
        const uint32_t nch_tot = __shfl(nch_incl, kWave - 1, kWave);
        if (nch_tot) {
            uint32_t hb = 0;
            if (lane == 0) hb = atomicAdd(io.heavy_cnt, nch_tot);
            hb = __shfl(hb, 0, kWave) + nch_incl - nch;
            if (heavy) {
                if (hb + nch <= io.heavy_cap) {
                    for (uint32_t c = 0; c < nch; ++c) {
                        const uint64_t len = (c + 1 < nch) ? kChunk : d - c * kChunk;
                        HeavyDesc hd;
                        hd.start_len = ((start + (uint64_t)c * kChunk) << kLenBits) | (len - 1);
                        hd.u = u;
                        hd.push = push;
                        io.heavy[hb + c] = hd;
                    }
                } else {
                    atomicOr(io.stats + 3, 2ull);
                }
            }
        }
        if (heavy) d = 0;
        const uint32_t incl = wave_incl_scan(d);
        const uint32_t total = __shfl(incl, kWave - 1, kWave);
        wave_lds_sync();
        walk_staged(g, io, efn, total, incl - d, d, start, u, push, sh, st);
        ws.edges += total;
        if (g.coff) ws.cedges += wave_sum_u64(start >= g.cap ? d : 0u);
        __builtin_amdgcn_wave_barrier();
    }
}

// Heavy tier body: one wave per kChunk-edge descriptor.
template <class EFn>
__device__ __forceinline__ void heavy_body(const GraphView &g, const PassIO &io, const EFn &efn, uint32_t nh,
                                           uint64_t gwave, uint64_t nwaves, OutStage &st, WaveStats &ws) {
    const uint32_t lane = lane_id();
    for (uint64_t i = gwave; i < nh; i += nwaves) {
        const HeavyDesc hd = io.hin[i];
        const uint64_t hstart = hd.start_len >> kLenBits;
        const uint32_t hlen = (uint32_t)(hd.start_len & ((1u << kLenBits) - 1)) + 1;
        for (uint32_t k0 = 0; k0 < hlen; k0 += kIlp * kWave) {
            uint32_t v[kIlp], src[kIlp], push[kIlp];
#pragma unroll
            for (int j = 0; j < kIlp; ++j) {
                src[j] = hd.u;
                push[j] = hd.push;
                v[j] = edge_at(g, hstart + min(k0 + j * kWave + lane, hlen - 1));
            }
#pragma unroll
            for (int j = 0; j < kIlp; ++j)
                if (k0 + j * kWave + lane >= hlen) v[j] = kGap;
            apply_edges(io, efn, src, v, push, st);
        }
        ws.hedges += hlen;
        if (hstart >= g.cap) ws.cedges += hlen;
    }
}

// One atomic per block for the pass counters.
template <int kWaves>
__device__ __forceinline__ void block_stats(const WaveStats &ws, unsigned long long (*red)[4], unsigned long long *stats) {
    const uint32_t w = threadIdx.x / kWave;
    const unsigned long long v = wave_sum_u64(ws.verts);
    if (lane_id() == 0) {
        red[w][0] = ws.edges;
        red[w][1] = v;
        red[w][2] = ws.hedges;
        red[w][3] = ws.cedges;  // lane 0 holds the wave's cached-edge total
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        unsigned long long t = 0;
        for (int i = 0; i < kWaves; ++i) t += red[i][threadIdx.x];
        // [0] edges, [1] vertices, [2] spilled-chunk edges, [5] edges read from the cache
        const int slot = threadIdx.x == 3 ? 5 : (int)threadIdx.x;
        if (t) atomicAdd(stats + slot, t);
    }
}

// ---- one pass ---------------------------------------------------------------------
// Light items of this pass, then the descriptors the previous pass spilled;
// the edge updates of every operator are order-insensitive (min-relaxations,
// residual pushes), so the spilled lists of round R-1 are walked in round R
// and whatever they activate joins round R+1.
// A round waits for memory 70 % of its waves' time (SSSP, 65 M edges), so waves
// in flight count: with all eight updates of a lane in flight SSSP and BFS took
// 210 registers (2 waves per SIMD) and CC 148 (3). Five or six waves spill and
// are slower again.
constexpr int kRoundWaves = 4;  // per SIMD
template <class VFn, class EFn>
__global__ void __launch_bounds__(kBlock, kRoundWaves) k_round(GraphView g, PassIO io, VFn vfn, EFn efn) {
    __shared__ LightWave s_wave[kWavesPerBlock];
    __shared__ unsigned long long s_red[kWavesPerBlock][4];
    __shared__ uint32_t s_n[kWavesPerBlock + 1];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (io.zero_cnt) *io.zero_cnt = 0;
        if (io.heavy_zero) *io.heavy_zero = 0;
        if (io.ecnt_zero) *io.ecnt_zero = 0;
        if (io.log) {  // the inputs of round R are what round R - 1 produced
            const uint32_t i = 2 * ((io.round + kRoundLog - 1) % kRoundLog);
            io.log[i] = *io.in_cnt;
            io.log[i + 1] = io.hin_cnt ? *io.hin_cnt : 0u;
        }
    }
    // a list never holds more than its capacity (appends past it are dropped and flagged)
    const uint32_t n = io.in_list ? min(*io.in_cnt, io.in_cap) : io.range_n;
    const uint32_t nh = io.hin ? min(*io.hin_cnt, io.heavy_cap) : 0;
    const uint32_t w = threadIdx.x / kWave;
    const uint64_t gwave = (uint64_t)blockIdx.x * kWavesPerBlock + w, nwaves = (uint64_t)gridDim.x * kWavesPerBlock;
    OutStage st{s_wave[w].out, 0};
    WaveStats ws;
    light_body(g, io, vfn, efn, n, gwave, nwaves, s_wave[w], st, ws);
    heavy_body(g, io, efn, nh, gwave, nwaves, st, ws);
    block_flush<kWavesPerBlock>(st, io, s_n);
    stage_count_flush(st, io);
    block_stats<kWavesPerBlock>(ws, s_red, io.stats);
}

// ---- vertex functors ---------------------------------------------------------
// Signature: bool (uint32_t u, uint32_t deg, uint32_t &push_bits, bool &enqueue_self)
// returns whether u's out-edges are expanded with push_bits.

// Data-driven relax round: commit the buffer, push (RelaxCTADB, sync_push_dd.cuh:196-230).
template <class Op>
struct VCombine {
    static constexpr bool kDense = false;
    static constexpr bool kItems = false;
    Op op;
    typename Op::value_t *value;
    typename Op::buffer_t *buffer;
    __device__ bool operator()(uint32_t u, uint32_t deg, uint32_t &push, bool &self) const {
        self = false;
        auto p = op.CombineValueBuffer(u, &value[u], &buffer[u], deg);
        push = to_bits<typename Op::push_t>(p.value);
        return p.scheduled;
    }
};

// Re-push of committed values scaled by type: PR cancel (-1) / compensate (+1)
// (RelaxCTADBAmend, sync_push_dd.cuh:375-470).
template <class Op>
struct VAmend {
    static constexpr bool kDense = false;
    static constexpr bool kItems = false;
    Op op;
    int type;
    typename Op::value_t *value;
    typename Op::buffer_t *buffer;
    __device__ bool operator()(uint32_t u, uint32_t deg, uint32_t &push, bool &self) const {
        self = false;
        auto p = op.CombineValueBufferAmend(u, type, &value[u], &buffer[u], deg);
        push = to_bits<typename Op::push_t>(p.value);
        return p.scheduled;
    }
};

// Traversal boundary sweep after invalidation: every vertex with a finite best
// value pushes it, edges only act on invalidated targets; invalidated vertices
// that are active on their own (CC: own label) join the frontier
// (the reference pushes to every target: RelaxCTADB_all_vertices,
// sync_push_dd.cuh:1470-1557).
template <class Op>
struct VSweep {
    static constexpr bool kDense = false;
    static constexpr bool kItems = false;
    Op op;
    typename Op::value_t *value;
    typename Op::buffer_t *buffer;
    const uint32_t *inval;   // bitmap
    uint32_t *stamp;
    uint32_t stamp_val;
    __device__ bool operator()(uint32_t u, uint32_t, uint32_t &push, bool &self) const {
        const uint64_t b = ld_relaxed(&buffer[u]);
        self = false;
        if ((inval[u >> 5] >> (u & 31)) & 1u) {
            if (op.IsActiveNode(u, b, value[u])) self = atomicExch(&stamp[u], stamp_val) != stamp_val;
        }
        push = op.PushValue(b);
        return push != api::kInf;
    }
};

// Invalidation propagation: expand every invalidated vertex.
struct VAll {
    static constexpr bool kDense = false;
    static constexpr bool kItems = false;
    __device__ bool operator()(uint32_t u, uint32_t, uint32_t &push, bool &self) const {
        self = false;
        push = u;
        return true;
    }
};

// ---- edge functors -------------------------------------------------------------
// load(v) peeks the destination state; apply_n(src, v, push, peek, enq) updates
// N destinations of the lane (v[j] = kGap: none) and says which join the output
// (src[j], the walked list's owner, when kAppendSource: a pull over in-lists).

// How the built-in programs fold the offer of an edge, a word pack(key, src),
// into the destination's: kFoldMin takes the smaller word, kFoldKey a smaller
// key only. Any other operator (also one derived from these) is called through
// its own AccumulateBuffer.
enum : int { kFoldNone = 0, kFoldMin = 1, kFoldKey = 2 };
template <class Op>
struct EdgeFold {
    static constexpr int kKind = kFoldNone;
    __device__ static uint32_t key(uint32_t, uint32_t) { return 0; }
};
template <>
struct EdgeFold<api::SSSP> {
    static constexpr int kKind = kFoldMin;
    __device__ static uint32_t key(uint32_t weight, uint32_t pushed) { return pushed + weight; }
};
template <>
struct EdgeFold<api::BFS> {
    static constexpr int kKind = kFoldMin;
    __device__ static uint32_t key(uint32_t, uint32_t pushed) { return pushed; }
};
template <>
struct EdgeFold<api::CC> {
    static constexpr int kKind = kFoldKey;
    __device__ static uint32_t key(uint32_t, uint32_t pushed) { return pushed; }
};

template <class Op>
struct ERelax {
    static constexpr bool kAppendSource = false;
    // Groups of 2, 4 and 8 updates at 4 waves per SIMD (8: spilling, so 2 waves
    // for SSSP and BFS, 3 for CC), static solves in us: SSSP on 65 M edges 1817,
    // 1848, 2002; BFS on 65 M 1189, 1232, 1446, on 12 M 388, 407, 486, on 1 M
    // 155, 168, 188; CC on 65 M 3360, 3333, 3557, on 4 M 653, 590, 589, on 1 M
    // 373, 340, 360. One at a time: 4 to 20 % more than 2.
    static constexpr int kUpdates = !Op::kTraversal ? kIlp : EdgeFold<Op>::kKind == kFoldMin ? 2 : 4;
    Op op;
    typename Op::buffer_t *buffer;
    uint32_t *stamp;
    uint32_t stamp_val;
    uint32_t wmode;
    uint64_t wseed;
    __device__ ERelax with_round(uint32_t stamp_next) const {
        ERelax e = *this;
        e.stamp_val = stamp_next;
        return e;
    }
    __device__ uint64_t load(uint32_t v) const {
        if constexpr (Op::kTraversal) return ld_peek(&buffer[v]);
        else return 0;
    }
    __device__ bool apply(uint32_t u, uint32_t v, uint32_t push, uint64_t peek) const {
        const uint32_t w = Op::kWeighted ? sg_weight(wmode, wseed, u, v) : 0u;
        const auto p = from_bits<typename Op::push_t>(push);
        if constexpr (Op::kTraversal) {
            if (!op.MayImprove(u, w, p, peek)) return false;
        }
        if (!op.AccumulateBuffer(u, v, w, &buffer[v], p)) return false;
        return atomicExch(&stamp[v], stamp_val) != stamp_val;
    }
    template <int N>
    __device__ __forceinline__ void apply_n(const uint32_t (&u)[N], const uint32_t (&v)[N], const uint32_t (&push)[N],
                                            const uint64_t (&peek)[N], bool (&enq)[N]) const {
        if constexpr (!Op::kTraversal) {  // PageRank: the crossing rule of AccumulateBuffer
            float old[N];
#pragma unroll
            for (int j = 0; j < N; ++j) {
                old[j] = 0.0f;
                if (v[j] != kGap) old[j] = unsafeAtomicAdd(&buffer[v[j]], from_bits<float>(push[j]));
            }
#pragma unroll
            for (int j = 0; j < N; ++j) enq[j] = v[j] != kGap && op.Crosses(old[j], from_bits<float>(push[j]));
        } else {
            uint32_t w[N];
#pragma unroll
            for (int j = 0; j < N; ++j) {
                w[j] = Op::kWeighted ? sg_weight(wmode, wseed, u[j], v[j]) : 0u;
                enq[j] = v[j] != kGap && op.MayImprove(u[j], w[j], from_bits<typename Op::push_t>(push[j]), peek[j]);
            }
            if constexpr (EdgeFold<Op>::kKind == kFoldMin) {
                unsigned long long old[N];
#pragma unroll
                for (int j = 0; j < N; ++j) {
                    old[j] = 0;
                    if (enq[j]) old[j] = atomicMin(&buffer[v[j]], api::pack(EdgeFold<Op>::key(w[j], push[j]), u[j]));
                }
#pragma unroll
                for (int j = 0; j < N; ++j) enq[j] = enq[j] && EdgeFold<Op>::key(w[j], push[j]) < api::hi32(old[j]);
            } else if constexpr (EdgeFold<Op>::kKind == kFoldKey) {
                unsigned long long old[N];
#pragma unroll
                for (int j = 0; j < N; ++j) {
                    old[j] = 0;
                    if (enq[j]) old[j] = atomicCAS(&buffer[v[j]], peek[j], api::pack(EdgeFold<Op>::key(w[j], push[j]), u[j]));
                }
#pragma unroll
                for (int j = 0; j < N; ++j)  // another offer came between: fold as usual
                    if (enq[j] && old[j] != peek[j])
                        enq[j] = op.AccumulateBuffer(u[j], v[j], w[j], &buffer[v[j]], from_bits<typename Op::push_t>(push[j]));
            } else {
#pragma unroll
                for (int j = 0; j < N; ++j)
                    if (enq[j])
                        enq[j] = op.AccumulateBuffer(u[j], v[j], w[j], &buffer[v[j]], from_bits<typename Op::push_t>(push[j]));
            }
        }
        claim<N>(v, enq);
    }
    // of the vertices to append, those not yet on the next frontier
    template <int N>
    __device__ __forceinline__ void claim(const uint32_t (&v)[N], bool (&enq)[N]) const {
        uint32_t was[N];
#pragma unroll
        for (int j = 0; j < N; ++j) {
            was[j] = stamp_val;
            if (enq[j]) was[j] = atomicExch(&stamp[v[j]], stamp_val);
        }
#pragma unroll
        for (int j = 0; j < N; ++j) enq[j] = was[j] != stamp_val;
    }
};

// Relax restricted to invalidated targets (boundary sweep). The probe reads a
// coarse bitmap (one bit per 64 vertices, small enough to stay in the vector
// L1) before the fine one, so most edges never touch L2 for the test.
template <class Op>
struct ERelaxInval {
    static constexpr bool kAppendSource = false;
    ERelax<Op> r;
    const uint32_t *inval;
    const uint32_t *coarse;  // coarse filter of inval (the sweep tests it first, in LDS)
    uint32_t cshift;
    __device__ ERelaxInval with_round(uint32_t stamp_next) const {
        ERelaxInval e = *this;
        e.r.stamp_val = stamp_next;
        return e;
    }
    __device__ uint32_t load(uint32_t v) const { return inval[v >> 5]; }
    __device__ bool test(uint32_t v, uint32_t word) const { return (word >> (v & 31)) & 1u; }
    // v is invalidated: relax it from u
    __device__ bool apply(uint32_t u, uint32_t v, uint32_t push) const { return r.apply(u, v, push, r.load(v)); }
};

// Reset tree children of u (AccumulateBuffer_del via PushFunctorDB_Del,
// push_functor.h:960-1034), claiming each child once through the bitmap.
template <class Op>
struct EInvalidate {
    static constexpr bool kAppendSource = false;
    static constexpr int kUpdates = kIlp;
    Op op;
    typename Op::value_t *value;
    typename Op::buffer_t *buffer;
    uint32_t *inval;
    uint32_t *coarse;
    uint32_t cshift;
    __device__ EInvalidate with_round(uint32_t) const { return *this; }
    __device__ uint64_t load(uint32_t v) const { return ld_relaxed(&buffer[v]); }
    template <int N>
    __device__ __forceinline__ void apply_n(const uint32_t (&u)[N], const uint32_t (&v)[N], const uint32_t (&)[N],
                                            const uint64_t (&b)[N], bool (&enq)[N]) const {
        uint32_t was[N];
#pragma unroll
        for (int j = 0; j < N; ++j) {
            was[j] = ~0u;
            if (v[j] != kGap && Op::Parent(b[j]) == u[j]) was[j] = atomicOr(&inval[v[j] >> 5], 1u << (v[j] & 31));
        }
#pragma unroll
        for (int j = 0; j < N; ++j) {
            enq[j] = !((was[j] >> (v[j] & 31)) & 1u);  // each child once; counted by the frontier it joins
            if (!enq[j]) continue;
            coarse_mark(coarse, cshift, v[j]);
            typename Op::buffer_t bb = b[j];
            op.AccumulateBuffer_del(u[j], v[j], &bb, &value[v[j]]);
            buffer[v[j]] = bb;
        }
    }
};


}  // namespace sg

#endif
