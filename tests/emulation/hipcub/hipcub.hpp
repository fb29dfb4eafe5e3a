// The device-wide sorts, scans and selections that the engine calls, on the CPU.
#ifndef EMULATION_HIPCUB_H
#define EMULATION_HIPCUB_H

#include <algorithm>
#include <numeric>
#include <vector>

#include <hip/hip_runtime.h>

namespace hipcub {

template <class T>
struct CountingInputIterator {
    T first;
    explicit CountingInputIterator(T x) : first(x) {}
    T operator[](size_t i) const { return (T)(first + i); }
};
template <class V, class F, class I>
struct TransformInputIterator {
    I it;
    F f;
    TransformInputIterator(I i, F g) : it(i), f(g) {}
    V operator[](size_t i) const { return f(it[i]); }
};

struct DeviceRadixSort {
    // bits [b0, b1) of a key in its order
    template <class K>
    static uint64_t key(K k, int b0, int b1) {
        uint64_t b = emulation::bits(k);
        if (std::is_floating_point<K>::value) b = b >> 31 ? (uint32_t)~b : b | 0x80000000u;
        return b1 - b0 < 64 ? (b >> b0) & ((1ull << (b1 - b0)) - 1) : b;
    }
    template <class K, class V, class N>
    static hipError_t sort(void *tmp, size_t &bytes, const K *kin, K *kout, const V *vin, V *vout, N n, int b0, int b1, bool down) {
        if (!tmp) return bytes = 64, hipSuccess;
        std::vector<size_t> at((size_t)n);
        std::iota(at.begin(), at.end(), 0);
        std::stable_sort(at.begin(), at.end(), [&](size_t x, size_t y) {
            const uint64_t a = key(kin[x], b0, b1), b = key(kin[y], b0, b1);
            return down ? a > b : a < b;
        });
        const std::vector<K> k(kin, kin + n);
        const std::vector<V> v(vin, vin + (vout ? (size_t)n : 0));
        for (size_t i = 0; i < (size_t)n; ++i) {
            kout[i] = k[at[i]];
            if (vout) vout[i] = v[at[i]];
        }
        return hipSuccess;
    }
    template <class K, class V, class N>
    static hipError_t SortPairs(void *tmp, size_t &bytes, const K *kin, K *kout, const V *vin, V *vout, N n, int b0 = 0,
                                int b1 = sizeof(K) * 8, hipStream_t = nullptr) {
        return sort(tmp, bytes, kin, kout, vin, vout, n, b0, b1, false);
    }
    template <class K, class V, class N>
    static hipError_t SortPairsDescending(void *tmp, size_t &bytes, const K *kin, K *kout, const V *vin, V *vout, N n,
                                          int b0 = 0, int b1 = sizeof(K) * 8, hipStream_t = nullptr) {
        return sort(tmp, bytes, kin, kout, vin, vout, n, b0, b1, true);
    }
    template <class K, class N>
    static hipError_t SortKeys(void *tmp, size_t &bytes, const K *kin, K *kout, N n, int b0 = 0, int b1 = sizeof(K) * 8,
                               hipStream_t = nullptr) {
        return sort(tmp, bytes, kin, kout, kin, (K *)nullptr, n, b0, b1, false);
    }
};
struct DeviceScan {
    template <class I, class O, class N>
    static hipError_t ExclusiveSum(void *tmp, size_t &bytes, I in, O out, N n, hipStream_t = nullptr) {
        if (!tmp) return bytes = 64, hipSuccess;
        unsigned long long sum = 0;
        for (size_t i = 0; i < (size_t)n; ++i) {
            const unsigned long long x = in[i];
            out[i] = sum;
            sum += x;
        }
        return hipSuccess;
    }
};
struct DeviceSelect {
    template <class I, class F, class O, class C, class N>
    static hipError_t Flagged(void *tmp, size_t &bytes, I in, F keep, O out, C count, N n, hipStream_t = nullptr) {
        if (!tmp) return bytes = 64, hipSuccess;
        size_t k = 0;
        for (size_t i = 0; i < (size_t)n; ++i)
            if (keep[i]) out[k++] = in[i];
        *count = k;
        return hipSuccess;
    }
};

}  // namespace hipcub

#endif
