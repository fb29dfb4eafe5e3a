// A pull plan of given lists at any id width, built and pulled by the engine's
// kernels on emulated memory (the width the engine picks follows from the
// number of vertices, so wide ones would need large graphs).
#include "sg_engine.hip"

using namespace sg;

namespace {
template <class T>
T *array(size_t n, const T *from = nullptr) {
    T *p = nullptr;
    if (hipMalloc(&p, n * sizeof(T))) abort();
    if (from) memcpy(p, from, n * sizeof(T));
    else memset(p, 0, n * sizeof(T));
    return p;
}
}  // namespace

// Lists deg[0 .. nv) of ids (list after list). words: the packed tiles.
// sums (or null; then ids may be any of `bits` bits): per list, the sum of
// push[id] over its ids. Returns the device's error.
extern "C" int emulation_pull_plan(uint32_t bits, uint32_t nv, const uint32_t *deg, const uint32_t *ids, uint64_t ne,
                                   const float *push, uint32_t *words, float *sums) {
    const uint64_t nt = (ne + kPullTile - 1) / kPullTile, tile = pull_tile_words(bits);
    const uint32_t nb = (nv + kScanSpan - 1) / kScanSpan;
    uint64_t *const off = array<uint64_t>((size_t)nv + 1);
    for (uint32_t v = 0; v < nv; ++v) off[v + 1] = off[v] + deg[v] + v % 3;  // with gaps
    uint32_t *const col = array<uint32_t>(off[nv] + 1);
    memset(col, 0xFF, (off[nv] + 1) * 4);
    for (uint32_t v = 0, k = 0; v < nv; ++v)
        for (uint32_t i = 0; i < deg[v]; ++i) col[off[v] + i] = ids[k++];
    GraphView g{};
    g.nv = nv;
    g.off = off;
    g.deg = array<uint32_t>(nv, deg);
    g.col = col;
    g.cap = off[nv];
    unsigned long long *const bsum = array<unsigned long long>(nb + 1), *const bcnt = array<unsigned long long>(nb + 1);
    unsigned long long *const start = array<unsigned long long>((size_t)nv + 1);
    uint32_t *const heads = array<uint32_t>(nt * (kPullTile / 32)), *const dst = array<uint32_t>((size_t)nv + kWave);
    uint32_t *const n = array<uint32_t>(1), *const packed = array<uint32_t>(nt * tile);
    PullTileMeta *const meta = array<PullTileMeta>(nt);
    const PullPlan plan{packed, nullptr, heads, dst, meta, nt, nt, ne, bits};
    hipLaunchKernelGGL(k_plan_sums, dim3(nb), dim3(kScanBlock), 0, 0, nv, g.deg, bsum, bcnt, heads, nt * (kPullTile / 32));
    hipLaunchKernelGGL(k_plan_lists, dim3(nb), dim3(kScanBlock), 0, 0, nv, g.deg, (const unsigned long long *)bsum,
                       (const unsigned long long *)bcnt, start, dst, heads, n);
    hipLaunchKernelGGL(k_plan_meta, dim3(1), dim3(256), 0, 0, nt, ne, (const unsigned long long *)start, (const uint32_t *)n,
                       (const uint32_t *)heads, meta);
    hipLaunchKernelGGL(k_plan_ids, dim3(2), dim3(kBlock), 0, 0, g, plan, (const unsigned long long *)start, (uint64_t)0, nt, packed);
    if (sums && !emulation::status()) {
        PrState p{};
        p.op.m_error = 1.0;
        p.value = array<float>(nv);
        p.res = array<float>(nv);
        p.pv_in = array<float>((size_t)nv + 4);
        memcpy((float *)p.pv_in, push, nv * sizeof(float));
        p.accg = array<float>(nv);
        p.relabel = p.unlabel = p.deg = g.deg;
        p.hot = 8;
        p.host_waves64 = 8;
        PassIO io{};
        io.stats = array<unsigned long long>(16);
        hipLaunchKernelGGL(k_pr_step<true>, dim3(8), dim3(kPrBlock), 0, 0, g, plan, PullSlots{}, p, io, (int)kPrAccum);
        hipLaunchKernelGGL(k_pr_tail<true>, dim3(8), dim3(kPrBlock), 0, 0, g, plan, (const unsigned long long *)nullptr,
                           SweepTiles{}, p, io, (int)kPrAccum);
        if (!emulation::status()) memcpy(sums, p.res, nv * sizeof(float));
    }
    if (!emulation::status()) memcpy(words, packed, nt * tile * 4);
    return emulation::status();
}
