// extrema.hip -- exact min / max of a field (StatBuffer::findMinMax,
// compressor.cu:228-302) on gfx950.
//
// One streaming pass with 16-byte loads; wave64 (DPP) then workgroup reduction,
// folded into two 64-bit words with atomicMin / atomicMax on an
// order-preserving integer image of the double value.  Min and max are
// exact, so the result does not depend on the reduction order.
#include "batch.hpp"
#include "common.hpp"
#include "extrema.hpp"

namespace pa {
namespace {

__global__ void extrema_init_kernel(unsigned long long* keys) {
    keys[0] = ~0ull;  // running min
    keys[1] = 0ull;   // running max
}

// One workgroup of 16 waves per CU: as many loads in flight as four of 4
// waves, and a quarter of the atomics on the keys, which all workgroups of a
// field below about 50 MB reach at the same time (24 MB: 35 us with 1024
// workgroups of 4 waves, most of it in up to 2048 atomics of 12 ns).
constexpr int kExtThreads = 1024;
template <typename T>
__global__ __launch_bounds__(kExtThreads) void extrema_kernel(const T* __restrict__ in, int64_t n,
                                                              unsigned long long* __restrict__ keys) {
    MinMax<T> m;
    using Vec = typename MinMax<T>::Vec;
    constexpr int V = MinMax<T>::V;
    const int64_t nv = n / V;
    const Vec* vin = reinterpret_cast<const Vec*>(in);
    const int64_t stride = (int64_t)gridDim.x * kExtThreads;
    // Each workgroup streams one contiguous chunk of whole 64 KiB batches; a
    // batch puts kBatch independent 16-byte loads per lane in flight before
    // any is reduced.
    constexpr int kBatch = 4;
    constexpr int64_t kSpan = (int64_t)kBatch * kExtThreads;  // vectors per batch
    const int64_t batches = nv / kSpan;
    const int64_t per = (batches + gridDim.x - 1) / gridDim.x;
    const int64_t b0 = blockIdx.x * per, b1 = b0 + per < batches ? b0 + per : batches;
    for (int64_t bt = b0; bt < b1; ++bt) {
        const Vec* p = vin + bt * kSpan + threadIdx.x;
        Vec v[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; ++k) v[k] = p[k * kExtThreads];
#pragma unroll
        for (int k = 0; k < kBatch; ++k) m.take(v[k]);
    }
    const int64_t at = blockIdx.x * (int64_t)kExtThreads + threadIdx.x;
    for (int64_t i = batches * kSpan + at; i < nv; i += stride) m.take(vin[i]);
    for (int64_t i = nv * V + at; i < n; i += stride) m.take(in[i]);
    double mn = (double)m.mn, mx = (double)m.mx;
    group_minmax<kExtThreads / 64>(mn, mx);
    if (threadIdx.x == 0) join_keys(mn, mx, keys);
}

__global__ void extrema_finish_kernel(const unsigned long long* keys, double* out) {
    out[0] = key_value(keys[0]);
    out[1] = key_value(keys[1]);
}

}  // namespace
}  // namespace pa

using namespace pa;

extern "C" int pa_extrema(const void* d_data, int dtype, int64_t n, double* d_minmax, void* stream) {
    if (!d_data || !d_minmax || n <= 0 || (dtype != PA_F32 && dtype != PA_F64)) return PA_ERR_ARG;
    if (((uintptr_t)d_data & 15) != 0) return PA_ERR_ARG;
    hipStream_t st = as_stream(stream);
    // two 64-bit keys kept right after the two doubles of the result
    unsigned long long* keys = reinterpret_cast<unsigned long long*>(d_minmax + 2);
    hipLaunchKernelGGL(extrema_init_kernel, dim3(1), dim3(1), 0, st, keys);
    PA_LAUNCH_CHECK();
    const int64_t work = (n + kExtThreads - 1) / kExtThreads;
    const int blocks = (int)(work < device_cus() ? work : device_cus());
    if (dtype == PA_F32)
        hipLaunchKernelGGL(extrema_kernel<float>, dim3(blocks), dim3(kExtThreads), 0, st, (const float*)d_data, n, keys);
    else
        hipLaunchKernelGGL(extrema_kernel<double>, dim3(blocks), dim3(kExtThreads), 0, st, (const double*)d_data, n,
                           keys);
    PA_LAUNCH_CHECK();
    hipLaunchKernelGGL(extrema_finish_kernel, dim3(1), dim3(1), 0, st, keys, d_minmax);
    PA_LAUNCH_CHECK();
    return PA_OK;
}

extern "C" int pa_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

int64_t pa::batch_ext_blocks(const pa_layout* L, int dtype, int ext_batches) {
    const int64_t nv = L->n / (16 / dtype);      // 16-byte vectors of the field
    return nv / (ext_batches * kExtBatch) + 1;  // the last workgroup also takes the scalar tail
}

