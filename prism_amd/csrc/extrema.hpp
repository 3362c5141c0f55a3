// extrema.hpp -- device pieces of the exact min / max (StatBuffer::findMinMax,
// compressor.cu:228-302) shared by the extrema kernels and the launch that
// runs the extrema beside the auto-tuner.
#pragma once
#include <rocprim/warp/warp_reduce.hpp>

#include "common.hpp"

namespace pa {

// order-preserving integer image of a double (and back): min / max become
// unsigned integer atomics
__device__ inline unsigned long long order_key(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}
__device__ inline double key_value(unsigned long long k) {
    const unsigned long long b = (k >> 63) ? (k & 0x7FFFFFFFFFFFFFFFull) : ~k;
    return __longlong_as_double((long long)b);
}

constexpr int64_t kExtBatch = 8 * 256;  // vectors per load batch (8 per lane in flight)

struct FMin {
    __device__ double operator()(double a, double b) const { return fmin(a, b); }
};
struct FMax {
    __device__ double operator()(double a, double b) const { return fmax(a, b); }
};

// min / max over the 64 lanes of a wave with DPP row shifts (exact: the
// order of the comparisons does not matter); valid in every lane
__device__ inline void wave_minmax(double& mn, double& mx) {
    using Reduce = rocprim::warp_reduce<double, 64>;
    typename Reduce::storage_type storage;
    double a, b;
    Reduce().reduce(mn, a, storage, FMin());
    Reduce().reduce(mx, b, storage, FMax());
    mn = a;
    mx = b;
}

// Running minimum and maximum of 16-byte vectors, in T (exact, as in double).
template <typename T>
struct MinMax {
    static constexpr int V = 16 / sizeof(T);
    using Vec = typename std::conditional<sizeof(T) == 4, float4, double2>::type;
    T mn = (T)__builtin_inf(), mx = -(T)__builtin_inf();
    __device__ __forceinline__ void take(T v) {
        mn = sizeof(T) == 4 ? (T)fminf((float)mn, (float)v) : (T)fmin((double)mn, (double)v);
        mx = sizeof(T) == 4 ? (T)fmaxf((float)mx, (float)v) : (T)fmax((double)mx, (double)v);
    }
    __device__ __forceinline__ void take(const Vec& v) {
        const T* e = reinterpret_cast<const T*>(&v);
#pragma unroll
        for (int j = 0; j < V; ++j) take(e[j]);
    }
};

// Min and max of a workgroup of WAVES waves; valid in thread 0.
template <int WAVES>
__device__ inline void group_minmax(double& mn, double& mx) {
    __shared__ double s_min[WAVES], s_max[WAVES];
    wave_minmax(mn, mx);
    if ((threadIdx.x & 63) == 0) {
        s_min[threadIdx.x >> 6] = mn;
        s_max[threadIdx.x >> 6] = mx;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < WAVES; ++w) {
            mn = fmin(mn, s_min[w]);
            mx = fmax(mx, s_max[w]);
        }
    }
}

// Workgroup `wg` of a field streams `span` 16-byte vectors of it in batches
// of 8 loads per lane (the tail elements go to the last one).  Its result is
// valid in thread 0.
template <typename T>
__device__ inline void extrema_span(const T* in, int64_t n, int64_t wg, int64_t span, double& mn, double& mx) {
    MinMax<T> m;
    using Vec = typename MinMax<T>::Vec;
    const int64_t nv = n / MinMax<T>::V;
    const Vec* vin = reinterpret_cast<const Vec*>(in);
    const int64_t v0 = wg * span;
    const int64_t v1 = v0 + span < nv ? v0 + span : nv;
    for (int64_t b = v0; b < v1; b += kExtBatch) {
        Vec v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int64_t i = b + threadIdx.x + k * 256;
            if (i < v1) v[k] = vin[i];
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int64_t i = b + threadIdx.x + k * 256;
            if (i < v1) m.take(v[k]);
        }
    }
    if (v0 + span >= nv) {  // last workgroup of the field: scalar tail
        for (int64_t i = nv * MinMax<T>::V + threadIdx.x; i < n; i += 256) m.take(in[i]);
    }
    mn = (double)m.mn;
    mx = (double)m.mx;
    group_minmax<4>(mn, mx);
}

// A workgroup's result joins the field's running keys.  Atomics on one address
// from every workgroup serialise (about 12 ns each on MI355X); one that cannot
// improve the running value skips its atomic.
__device__ inline void join_keys(double mn, double mx, unsigned long long* keys) {
    const unsigned long long kmn = order_key(mn), kmx = order_key(mx);
    if (kmn < __hip_atomic_load(keys, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(keys, kmn);
    if (kmx > __hip_atomic_load(keys + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(keys + 1, kmx);
}

}  // namespace pa
