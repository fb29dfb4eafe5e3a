// Sort of an update batch by source, in at most three kernels.
//
//   inserts  keys (u << 32 | position in the batch): sources ascending, file
//            order within a source; out: sources and targets
//   deletes  keys (u << 32 | v); out: the keys
//
// A sample sort: every block sorts the same small sample of its side in LDS
// and takes splitters from it; the keys are counted per bucket
// (k_sort_count), moved to their buckets (k_sort_move) and the buckets sorted
// in LDS, one block each (k_sort_buckets). A batch of at most kSortOne pairs a
// side is one bucket, read straight from the pairs: one kernel.
// Keys equal to a splitter get a bucket of their own that needs no sort, so
// many copies of one delete fill no other bucket.
//
// Both sides go through the same launches. The library's sorts take a launch
// per merge step (two sorts of 100,000: 30 launches, 120 us and the gaps
// between them); batches past kSortMost still go there.
#ifndef SG_SORT_H
#define SG_SORT_H

#include "sg_kernels.h"

namespace sg {

constexpr uint32_t kSortOne = 2048;            // pairs of a side sorted as one bucket
constexpr uint32_t kSortMost = 1u << 20;       // pairs of a side sorted here
constexpr uint32_t kSortBucket = 768;          // aimed-at keys per bucket
constexpr uint32_t kSortMaxSplit = 512;        // splitters at most (buckets: 2 * splitters + 1)
constexpr uint32_t kSortOver = 8;              // sample keys per splitter
constexpr uint32_t kSortRows = 128;            // counting blocks of a side at most
constexpr int kSortBlock = 512;
constexpr uint32_t kSortLds = 8192;            // keys a block sorts in LDS

struct SortSide {
    const uint32_t *pairs;     // [2 * n]
    uint32_t n;
    uint32_t nsplit;           // splitters (0: one bucket)
    uint32_t rows, tile;       // counting blocks, pairs per block
    unsigned long long *split; // [nsplit]
    uint32_t *start;           // [nbuckets + 1]
    uint32_t *hist;            // [rows][nbuckets]
    unsigned long long *tmp;   // [n] keys by bucket
    uint32_t *out_key, *out_val;      // inserts
    unsigned long long *out_del;      // deletes
    __host__ __device__ uint32_t nbuckets() const { return 2 * nsplit + 1; }
};
struct SortBatch {
    SortSide side[2];  // inserts, deletes
    uint32_t nv;
    int a, b;                   // column of the source and of the target
    const uint32_t *relabel;    // id that the targets are recorded by (null: as given)
    unsigned long long *dropped;  // pairs with an id >= nv, counted once
};

// Key of pair i: dropped pairs (an id >= nv) sort past every other.
__device__ __forceinline__ unsigned long long sort_key(const SortBatch &sb, int s, uint32_t i) {
    const SortSide &x = sb.side[s];
    const uint32_t u = x.pairs[2ull * i + sb.a], v = x.pairs[2ull * i + sb.b];
    const bool ok = u < sb.nv && v < sb.nv;
    if (s == 0) return ((unsigned long long)(ok ? u : kGap) << 32) | i;
    return ok ? ((unsigned long long)u << 32) | (sb.relabel ? sb.relabel[v] : v) : ~0ull;
}
// Target of insert i as the store records it.
__device__ __forceinline__ uint32_t sort_target(const SortBatch &sb, uint32_t i) {
    const uint32_t v = sb.side[0].pairs[2ull * i + sb.b];
    return sb.relabel && v < sb.nv ? sb.relabel[v] : v;
}
__device__ __forceinline__ bool sort_dropped(int s, unsigned long long key) {
    return s == 0 ? (uint32_t)(key >> 32) == kGap : key == ~0ull;
}

// n keys of s (LDS, room for T * E; T threads) in ascending order: each thread
// sorts E in registers, then runs are merged pairwise along merge paths.
template <int T, int E>
__device__ __forceinline__ void lds_sort(unsigned long long *s, uint32_t n) {
    const uint32_t t = threadIdx.x;
    unsigned long long k[E];
#pragma unroll
    for (int j = 0; j < E; ++j) k[j] = t * E + j < n ? s[t * E + j] : ~0ull;
#pragma unroll
    for (int r = 0; r < E; ++r) {  // odd-even transposition
#pragma unroll
        for (int j = r & 1; j + 1 < E; j += 2) {
            const unsigned long long a = min_u64(k[j], k[j + 1]), b = k[j] ^ k[j + 1] ^ a;
            k[j] = a;
            k[j + 1] = b;
        }
    }
    for (uint32_t w = E; w < n; w *= 2) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < E; ++j) s[t * E + j] = k[j];
        __syncthreads();
        // the thread's outputs [d, d + E) of its pair of runs A = s[g, g + w), B = s[g + w, g + 2w)
        const uint32_t g = t * E / (2 * w) * (2 * w), d = t * E - g;
        const unsigned long long *const A = s + g, *const B = s + g + w;
        const uint32_t room = (uint32_t)(T * E) - g;  // keys from g on (B may be short at the end)
        const uint32_t na = min(w, room), nb = room > w ? min(w, room - w) : 0u;
        uint32_t lo = d > nb ? d - nb : 0u, hi = min(d, na);
        while (lo < hi) {
            const uint32_t m = (lo + hi) / 2;
            if (A[m] <= B[d - 1 - m]) lo = m + 1; else hi = m;
        }
        uint32_t ia = lo, ib = d - lo;
        unsigned long long x = ia < na ? A[ia] : ~0ull, y = ib < nb ? B[ib] : ~0ull;
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const bool first = ib >= nb || (ia < na && x <= y);
            k[j] = first ? x : y;
            if (first) {
                ++ia;
                x = ia < na ? A[ia] : ~0ull;
            } else {
                ++ib;
                y = ib < nb ? B[ib] : ~0ull;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < E; ++j) s[t * E + j] = k[j];
    __syncthreads();
}
template <int T>
__device__ __forceinline__ void lds_sort_any(unsigned long long *s, uint32_t n) {
    if (n <= T * 2) lds_sort<T, 2>(s, n);
    else if (n <= T * 4) lds_sort<T, 4>(s, n);
    else if (n <= T * 8) lds_sort<T, 8>(s, n);
    else lds_sort<T, 16>(s, n);
}

// Bucket of a key among sorted splitters: 2 i + 1 when it equals splitter i
// (the first such), else 2 i with i the splitters below it.
__device__ __forceinline__ uint32_t sort_bucket(const unsigned long long *split, uint32_t nsplit, unsigned long long key) {
    uint32_t lo = 0, hi = nsplit;
    while (lo < hi) {
        const uint32_t m = (lo + hi) / 2;
        if (split[m] < key) lo = m + 1; else hi = m;
    }
    return 2 * lo + (lo < nsplit && split[lo] == key ? 1u : 0u);
}

__global__ void __launch_bounds__(kSortBlock) k_sort_count(SortBatch sb) {
    __shared__ unsigned long long s_samp[kSortMaxSplit * kSortOver];
    __shared__ uint32_t s_hist[2 * kSortMaxSplit + 1];
    __shared__ unsigned long long s_split[kSortMaxSplit];
    static_assert(kSortMaxSplit * kSortOver <= kSortBlock * 16, "the sample fits one block's sort");
    const int s = blockIdx.x < sb.side[0].rows ? 0 : 1;
    const SortSide &x = sb.side[s];
    const uint32_t row = blockIdx.x - (s ? sb.side[0].rows : 0u), nb = x.nbuckets();
    const uint32_t ns = x.nsplit * kSortOver;  // <= n
    for (uint32_t i = threadIdx.x; i < ns; i += kSortBlock) {  // one pair of each n / ns of the batch
        const uint32_t a = (uint32_t)((unsigned long long)i * x.n / ns), e = (uint32_t)((unsigned long long)(i + 1) * x.n / ns);
        s_samp[i] = sort_key(sb, s, a + (i * 2654435761u >> 8) % (e - a));
    }
    __syncthreads();
    lds_sort_any<kSortBlock>(s_samp, ns);
    for (uint32_t i = threadIdx.x; i < x.nsplit; i += kSortBlock) {
        s_split[i] = s_samp[i * kSortOver + kSortOver / 2];
        if (row == 0) x.split[i] = s_split[i];
    }
    for (uint32_t i = threadIdx.x; i < nb; i += kSortBlock) s_hist[i] = 0;
    __syncthreads();
    const uint32_t e = min(x.n, (row + 1) * x.tile);
    uint32_t drop = 0;
    for (uint32_t i = row * x.tile + threadIdx.x; i < e; i += kSortBlock) {
        const unsigned long long k = sort_key(sb, s, i);
        drop += sort_dropped(s, k);
        atomicAdd(&s_hist[sort_bucket(s_split, x.nsplit, k)], 1u);
    }
    if (drop) atomicAdd(sb.dropped, (unsigned long long)drop);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < nb; i += kSortBlock) x.hist[(uint64_t)row * nb + i] = s_hist[i];
}

// Start of the row's part of every bucket in s_off (block-wide); row 0's are
// the starts of the buckets.
__device__ __forceinline__ void sort_offsets(const SortSide &x, uint32_t row, uint32_t *s_off, uint32_t *s_w) {
    const uint32_t nb = x.nbuckets();
    uint32_t carry = 0;
    for (uint32_t b0 = 0; b0 < nb; b0 += kSortBlock) {
        const uint32_t b = b0 + threadIdx.x;
        uint32_t total = 0, before = 0;
        if (b < nb) {
#pragma unroll 4
            for (uint32_t r = 0; r < x.rows; ++r) {
                const uint32_t c = x.hist[(uint64_t)r * nb + b];
                total += c;
                before += r < row ? c : 0u;
            }
        }
        const uint32_t inc = wave_incl_scan(total), w = threadIdx.x / kWave;
        if (lane_id() == kWave - 1) s_w[w] = inc;
        __syncthreads();
        uint32_t off = carry;
        for (uint32_t i = 0; i < (uint32_t)(kSortBlock / kWave); ++i) {
            if (i < w) off += s_w[i];
            carry += s_w[i];
        }
        if (b < nb) s_off[b] = off + inc - total + before;
        __syncthreads();
    }
}

__global__ void __launch_bounds__(kSortBlock) k_sort_move(SortBatch sb) {
    __shared__ uint32_t s_off[2 * kSortMaxSplit + 1];
    __shared__ uint32_t s_w[kSortBlock / kWave];
    __shared__ unsigned long long s_split[kSortMaxSplit];
    const int s = blockIdx.x < sb.side[0].rows ? 0 : 1;
    const SortSide &x = sb.side[s];
    const uint32_t row = blockIdx.x - (s ? sb.side[0].rows : 0u);
    for (uint32_t i = threadIdx.x; i < x.nsplit; i += kSortBlock) s_split[i] = x.split[i];
    sort_offsets(x, row, s_off, s_w);
    if (row == 0) {
        for (uint32_t i = threadIdx.x; i < x.nbuckets(); i += kSortBlock) x.start[i] = s_off[i];
        if (threadIdx.x == 0) x.start[x.nbuckets()] = x.n;
        __syncthreads();
    }
    const uint32_t e = min(x.n, (row + 1) * x.tile);
    for (uint32_t i = row * x.tile + threadIdx.x; i < e; i += kSortBlock) {
        const unsigned long long k = sort_key(sb, s, i);
        x.tmp[atomicAdd(&s_off[sort_bucket(s_split, x.nsplit, k)], 1u)] = k;
    }
}

// One block per bucket of keys that equal no splitter; those that do are
// copied by the block of the bucket before them.
__global__ void __launch_bounds__(kSortBlock) k_sort_buckets(SortBatch sb) {
    __shared__ unsigned long long s_key[kSortLds];
    const uint32_t n0 = sb.side[0].n ? sb.side[0].nsplit + 1 : 0u;
    const int s = blockIdx.x < n0 ? 0 : 1;
    const SortSide &x = sb.side[s];
    const uint32_t q = blockIdx.x - (s ? n0 : 0u);
    uint32_t lo = 0, hi = x.n, end = x.n;  // the bucket, and its run of equal keys [hi, end)
    if (x.nsplit) {
        lo = x.start[2 * q];
        hi = x.start[2 * q + 1];
        end = q < x.nsplit ? x.start[2 * q + 2] : hi;
    }
    auto put = [&](uint32_t i, unsigned long long k) {
        if (s) {
            x.out_del[i] = k;
        } else {
            x.out_key[i] = (uint32_t)(k >> 32);
            x.out_val[i] = sort_target(sb, (uint32_t)k);
        }
    };
    for (uint32_t i = hi + threadIdx.x; i < end; i += kSortBlock) put(i, x.tmp[i]);
    const uint32_t n = hi - lo;
    if (n <= kSortLds) {
        uint32_t drop = 0;
        for (uint32_t i = threadIdx.x; i < n; i += kSortBlock) {
            const unsigned long long k = x.nsplit ? x.tmp[lo + i] : sort_key(sb, s, i);
            if (x.nsplit == 0) drop += sort_dropped(s, k);  // counted by k_sort_count otherwise
            s_key[i] = k;
        }
        if (drop) atomicAdd(sb.dropped, (unsigned long long)drop);
        __syncthreads();
        lds_sort_any<kSortBlock>(s_key, n);
        for (uint32_t i = threadIdx.x; i < n; i += kSortBlock) put(lo + i, s_key[i]);
        return;
    }
    // a bucket past LDS (ten times the aimed-at size: the sample missed): sorted
    // where it lies, a bitonic network padded with keys past every other
    unsigned long long *const k = x.tmp + lo;
    for (uint64_t size = 2; size < 2ull * n; size *= 2) {
        for (uint64_t stride = size / 2; stride > 0; stride /= 2) {
            __syncthreads();
            for (uint64_t i = threadIdx.x; i < n; i += kSortBlock) {
                // first step of a size compares mirrored positions, so that all runs ascend
                const uint64_t j = stride == size / 2 ? i ^ (size - 1) : i ^ stride;
                if (j > i && j < n && k[j] < k[i]) {
                    const unsigned long long y = k[i];
                    k[i] = k[j];
                    k[j] = y;
                }
            }
            __threadfence_block();
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n; i += kSortBlock) put(lo + i, k[i]);
}

}  // namespace sg

#endif
