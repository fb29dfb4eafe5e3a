// The part of HIP that the engine uses, for a CPU build of its kernels.
//
// A launch runs its blocks one after the other, the lanes of a block as fibers:
// a wave operation (ballot, shuffle, DPP move, wave barrier) completes when
// every live lane of the wave has come to the same one, __syncthreads when
// every live thread of the block has. Each allocation ends at a page that
// cannot be touched, and stays so as a whole once it is freed, so an access out
// of bounds or after a free fails the launch as it would on the device
// (hipErrorIllegalAddress from then on). Plain C++ is what is checked:
// the device's memory order, its atomics and its timing are not modelled.
#ifndef EMULATION_HIP_RUNTIME_H
#define EMULATION_HIP_RUNTIME_H

#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <cmath>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <utility>

#define __global__
#define __device__
#define __host__
#define __shared__ static  // one block at a time
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(n) __attribute__((aligned(n)))
#define HIP_SYMBOL(x) x

struct dim3 {
    uint32_t x, y, z;
    dim3(uint32_t a = 1, uint32_t b = 1, uint32_t c = 1) : x(a), y(b), z(c) {}
};
extern dim3 blockIdx, blockDim, gridDim;

namespace emulation {
extern std::recursive_mutex mu;  // one launch or copy at a time
struct Lane {
    uint32_t tid;
};
extern Lane *cur;
// Wait for the wave; what its lanes brought is in snap(), the live ones in the result.
uint64_t wave_sync(uint64_t word, int line);
const uint64_t *snap();
void block_sync(int line);
[[noreturn]] void lane_error(const char *what, int line);
void run(const void *kernel, dim3 grid, dim3 block, void (*fn)(void *), void *arg);
int status();
void *alloc(size_t bytes);
void release(void *p);

template <class... P, class... A>
void launch(void (*kernel)(P...), dim3 grid, dim3 block, A &&...args) {
    struct Call {
        void (*kernel)(P...);
        std::tuple<std::decay_t<P>...> args;
    } call{kernel, std::tuple<std::decay_t<P>...>(std::forward<A>(args)...)};
    run((const void *)kernel, grid, block, [](void *p) {
        Call *const c = static_cast<Call *>(p);
        std::apply(c->kernel, c->args);  // by value: each lane its own
    }, &call);
}
template <class T>
uint64_t bits(T x) {
    uint64_t b = 0;
    memcpy(&b, &x, sizeof x);
    return b;
}
template <class T>
T from(uint64_t b) {
    T x;
    memcpy(&x, &b, sizeof x);
    return x;
}
}  // namespace emulation

#define hipLaunchKernelGGL(kernel, grid, block, lds, stream, ...) \
    emulation::launch(kernel, grid, block, ##__VA_ARGS__)
#define threadIdx (dim3(emulation::cur->tid))

// ---- wave and block operations ----------------------------------------------------
static inline uint32_t __lane_id() { return emulation::cur->tid & 63u; }
static inline void __syncthreads(int line = __builtin_LINE()) { emulation::block_sync(line); }
static inline uint64_t __ballot(bool p, int line = __builtin_LINE()) {
    const uint64_t live = emulation::wave_sync(p, line);
    uint64_t m = 0;
    for (int i = 0; i < 64; ++i)
        if ((live >> i) & 1) m |= (emulation::snap()[i] & 1) << i;
    return m;
}
template <class T>
T __shfl(T x, int lane, int = 64, int line = __builtin_LINE()) {
    emulation::wave_sync(emulation::bits(x), line);
    return emulation::from<T>(emulation::snap()[lane & 63]);
}
template <class T>
T __shfl_xor(T x, int d, int = 64, int line = __builtin_LINE()) {
    return __shfl(x, (int)__lane_id() ^ d, 64, line);
}
static inline int emulated_readlane(int x, int lane, int line) {
    const uint64_t live = emulation::wave_sync(emulation::bits(x), line);
    if (lane < 0) lane = __builtin_ctzll(live);  // the first live lane
    if (lane > 63) emulation::lane_error("a lane past the wave is read", line);
    return emulation::from<int>(emulation::snap()[lane]);
}
static inline int emulated_dpp(int old, int x, int ctrl, int rows, int line) {
    if (~emulation::wave_sync(emulation::bits(x), line)) emulation::lane_error("a lane move needs every lane", line);
    const int lane = (int)__lane_id(), row = lane / 16;
    int src = -1;
    if (ctrl > 0x110 && ctrl < 0x120) src = lane % 16 >= ctrl - 0x110 ? lane - (ctrl - 0x110) : -1;  // row_shr
    else if (ctrl == 0x138) src = lane - 1;                                                          // wave_shr
    else if (ctrl == 0x142) src = row * 16 - 1;                                                      // row_bcast15
    else if (ctrl == 0x143) src = row >= 2 ? 31 : -1;                                                // row_bcast31
    else emulation::lane_error("unknown lane move", line);
    return src < 0 || !((rows >> row) & 1) ? old : emulation::from<int>(emulation::snap()[src]);
}
#define __builtin_amdgcn_readlane(x, lane) emulated_readlane(x, lane, __LINE__)
#define __builtin_amdgcn_readfirstlane(x) emulated_readlane(x, -1, __LINE__)
#define __builtin_amdgcn_update_dpp(old, x, ctrl, rows, banks, bound) emulated_dpp(old, x, ctrl, rows, __LINE__)
#define __builtin_amdgcn_wave_barrier() ((void)emulation::wave_sync(0, __LINE__))
#define __builtin_amdgcn_fence(...) ((void)0)
#define __builtin_amdgcn_alignbit(hi, lo, s) ((uint32_t)((((uint64_t)(hi) << 32) | (uint32_t)(lo)) >> ((s) & 31)))
static inline void __threadfence_system() {}
static inline void __threadfence_block() {}

// ---- arithmetic ---------------------------------------------------------------------
static inline int __popc(uint32_t x) { return __builtin_popcount(x); }
static inline int __popcll(unsigned long long x) { return __builtin_popcountll(x); }
static inline int __ffsll(unsigned long long x) { return __builtin_ffsll((long long)x); }
static inline int __clzll(long long x) { return x ? __builtin_clzll((unsigned long long)x) : 64; }
static inline uint32_t __float_as_uint(float x) { return emulation::from<uint32_t>(emulation::bits(x)); }
static inline float __uint_as_float(uint32_t x) { return emulation::from<float>(x); }
static inline long long __double_as_longlong(double x) { return emulation::from<long long>(emulation::bits(x)); }
static inline double __longlong_as_double(long long x) { return emulation::from<double>((uint64_t)x); }
template <class A, class B>
std::common_type_t<A, B> min(A a, B b) {
    using C = std::common_type_t<A, B>;
    return (C)a < (C)b ? (C)a : (C)b;
}
template <class A, class B>
std::common_type_t<A, B> max(A a, B b) {
    using C = std::common_type_t<A, B>;
    return (C)a < (C)b ? (C)b : (C)a;
}
struct uint4 {
    uint32_t x, y, z, w;
};
struct float4 {
    float x, y, z, w;
};

// ---- atomics: one lane runs at a time -------------------------------------------------
#define EMULATED_ATOMIC(name, value)      \
    template <class T, class U>           \
    T name(T *p, U v) {                   \
        const T old = *p;                 \
        *p = (T)(value);                  \
        return old;                       \
    }
EMULATED_ATOMIC(atomicAdd, old + (T)v)
EMULATED_ATOMIC(unsafeAtomicAdd, old + (T)v)
EMULATED_ATOMIC(atomicOr, old | (T)v)
EMULATED_ATOMIC(atomicExch, v)
EMULATED_ATOMIC(atomicMin, (T)v < old ? (T)v : old)
EMULATED_ATOMIC(atomicMax, old < (T)v ? (T)v : old)
template <class T, class U, class V>
T atomicCAS(T *p, U expected, V v) {
    const T old = *p;
    if (old == (T)expected) *p = (T)v;
    return old;
}
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __HIP_MEMORY_SCOPE_SYSTEM 0
#define __hip_atomic_load(p, order, scope) (*(p))
#define __hip_atomic_store(p, v, order, scope) __atomic_store_n(p, v, __ATOMIC_RELEASE)

// ---- runtime: every call completes before it returns ----------------------------------
typedef int hipError_t;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorNotReady = 600, hipErrorIllegalAddress = 700, hipErrorNotSupported = 801 };
typedef void *hipStream_t, *hipEvent_t, *hipGraph_t, *hipGraphExec_t, *hipGraphNode_t;
enum { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice, hipMemcpyDefault };
enum { hipHostMallocDefault = 0, hipHostMallocMapped = 2, hipHostMallocCoherent = 4 };
enum { hipStreamNonBlocking = 1, hipEventDisableTiming = 2 };
struct hipDeviceProp_t {
    int multiProcessorCount, warpSize;
    char gcnArchName[64];
};
struct hipKernelNodeParams {
    void *func;
    dim3 gridDim, blockDim;
    unsigned sharedMemBytes;
    void **kernelParams, **extra;
};
static inline const char *hipGetErrorString(hipError_t e) {
    return e == hipErrorIllegalAddress ? "an illegal memory access was encountered" : "not emulated";
}
template <class T>
hipError_t hipMalloc(T **p, size_t n) {
    *p = (T *)emulation::alloc(n);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
template <class T>
hipError_t hipHostMalloc(T **p, size_t n, unsigned = 0) { return hipMalloc(p, n); }
static inline hipError_t hipFree(void *p) { return emulation::release(p), hipSuccess; }
static inline hipError_t hipHostFree(void *p) { return hipFree(p); }
static inline hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) { return *d = h, hipSuccess; }
static inline hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, int, hipStream_t = nullptr) {
    std::lock_guard<std::recursive_mutex> lock(emulation::mu);
    if (emulation::status()) return emulation::status();
    memmove(to, from, n);
    return hipSuccess;
}
static inline hipError_t hipMemcpy(void *to, const void *from, size_t n, int kind) { return hipMemcpyAsync(to, from, n, kind); }
static inline hipError_t hipGetLastError() { return hipSuccess; }  // a failed kernel shows at a wait, a copy or a query
static inline hipError_t hipSetDevice(int) { return hipSuccess; }
static inline hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
static inline hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
static inline hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {
    return *p = hipDeviceProp_t{8, 64, "gfx950"}, hipSuccess;
}
static inline hipError_t hipMemGetInfo(size_t *free, size_t *total) { return *free = *total = 64ull << 30, hipSuccess; }
template <class T>
hipError_t hipGetSymbolAddress(void **p, T &x) { return *p = (void *)&x, hipSuccess; }
template <class K>
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, K, int, size_t) { return *n = 1, hipSuccess; }
static inline hipError_t hipStreamCreate(hipStream_t *s) { return *s = s, hipSuccess; }
static inline hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = s, hipSuccess; }
static inline hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
static inline hipError_t hipStreamSynchronize(hipStream_t) { return emulation::status(); }
static inline hipError_t hipStreamQuery(hipStream_t) { return emulation::status(); }
static inline hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
static inline hipError_t hipEventCreate(hipEvent_t *e) { return *e = e, hipSuccess; }
static inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = e, hipSuccess; }
static inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
static inline hipError_t hipEventRecord(hipEvent_t, hipStream_t = nullptr) { return hipSuccess; }
static inline hipError_t hipEventQuery(hipEvent_t) { return emulation::status(); }
static inline hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 0.0f, hipSuccess; }
// (graphs are not emulated)
static inline hipError_t hipGraphCreate(hipGraph_t *, unsigned) { return hipErrorNotSupported; }
static inline hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
static inline hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, void *, void *, size_t) { return hipErrorNotSupported; }
static inline hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
static inline hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
static inline hipError_t hipGraphAddKernelNode(hipGraphNode_t *, hipGraph_t, const hipGraphNode_t *, size_t,
                                               const hipKernelNodeParams *) { return hipErrorNotSupported; }
static inline hipError_t hipGraphExecKernelNodeSetParams(hipGraphExec_t, hipGraphNode_t, const hipKernelNodeParams *) {
    return hipErrorNotSupported;
}

#endif
