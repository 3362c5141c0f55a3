// spline_rules.hpp -- the predictor's formulas and its quantiser, and the
// small device helpers that its kernels share.  Arithmetic is in T (FP64 for
// double fields), evaluated in the reference's order with no FMA contraction,
// so the compressor and the decompressor reproduce identical values.
#pragma once

#include <rocprim/warp/warp_reduce.hpp>

#include "common.hpp"

namespace pa {
namespace {

constexpr int kThreads = 256;

enum Mode { COMPRESS, DECOMPRESS };

template <typename T>
__device__ __forceinline__ T cubic(T a, T b, T c, T d, bool natural = false) {
    if (natural) return ((((T)-3 * a + (T)23 * b) + (T)23 * c) - (T)3 * d) / (T)40;
    return (((-a + (T)9 * b) + (T)9 * c) - d) / (T)16;
}
template <typename T>
__device__ __forceinline__ T quad_l(T t0, T t1, T t2) {
    return ((-t0 + (T)6 * t1) + (T)3 * t2) / (T)8;
}
template <typename T>
__device__ __forceinline__ T quad_r(T t1, T t2, T t3) {
    return (((T)3 * t1 + (T)6 * t2) - t3) / (T)8;
}
template <typename T>
__device__ __forceinline__ T lin(T t1, T t2) {
    return (t1 + t2) / (T)2;
}

// s / 3, correctly rounded: a rounded product by 1 / 3, its exact remainder
// (fma) and one corrected step (Markstein's division by a constant).  s / 3 is
// never within 1 / 6 ulp of a rounding boundary, subnormal results included, and
// the step's error is below 2^-20 ulp, so the result is that of the division;
// infinities and NaN pass through.  4 instructions instead of 10 (float32).
__host__ __device__ __forceinline__ float third_of(float s) {
    const float c = 1.0f / 3.0f, q = s * c;
    const float d = __builtin_fmaf(__builtin_fmaf(-3.0f, q, s), c, q);
    return __builtin_fabsf(s) < __builtin_inff() ? d : q;
}
__host__ __device__ __forceinline__ double third_of(double s) {
    const double c = 1.0 / 3.0, q = s * c;
    const double d = __builtin_fma(__builtin_fma(-3.0, q, s), c, q);
    return __builtin_fabs(s) < __builtin_inf() ? d : q;
}

// The thread id through an opaque move: index arithmetic derived from it in
// one phase of the kernel is not merged with that of another phase and kept
// live in registers between them.
__device__ __forceinline__ int thread_id() {
    int v;
    asm volatile("v_mov_b32 %0, %1" : "=v"(v) : "v"((int)threadIdx.x));
    return v;
}
// lane of a unit's 256 lanes (a workgroup holds one or two units); lanes
// 0..63 are those of the unit's wave `first`
__device__ __forceinline__ int lane_id(int first = 0) { return (thread_id() - 64 * first) & (kThreads - 1); }

// A uniform read, through the scalar cache, of memory that nothing in the
// launch writes.
template <typename V>
__device__ __forceinline__ V scalar_load(const V* p) {
    return *(const __attribute__((address_space(4))) V*)(uintptr_t)p;
}

// Barrier for LDS producer/consumer hand-off between stages: waits for this
// wave's LDS operations only, so outstanding global loads (prefetched codes)
// and stores (emitted codes) stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Quantise v against pred, write the reconstruction back and return the
// code (InterpolationPredictor.cu:1327-1341).
template <typename T>
__device__ __forceinline__ int32_t quantize_val(T& v, T pred, T eb_r, T ebx2) {
    const T err = v - pred;
    // |err| eb_r + 1 with err's sign (that of a zero does not matter: +-1 / 2
    // truncates to 0)
    T code = copysign(fabs(err) * eb_r + (T)1, err);
    const int qv = (int)(code / (T)2);
    code = (T)qv;
    v = pred + code * ebx2;
    return qv;
}

// Range of the codes that a lane stores, 0 included: a code passes through and
// is counted (two instructions for two codes: the compiler joins the
// comparisons of a pair; an OR of the magnitudes took three a code, 8 % of the
// tile kernels' instructions).
struct CodeRange {
    int32_t lo = 0, hi = 0;
    __device__ __forceinline__ int32_t operator()(int32_t c) {
        lo = min(lo, c);
        hi = max(hi, c);
        return c;
    }
    // the bits of the largest magnitudes c ^ (c >> 31)
    __device__ __forceinline__ uint32_t mags() const { return (uint32_t)hi | (uint32_t)(lo ^ (lo >> 31)); }
};
struct Mags {
    CodeRange fine, coarse;  // level 0's, the other levels'
};

// A wave's part in live_words: its XCD's word as it was when the wave began
// (read with the wave's first loads), and its own magnitudes joined at the end.
// The bits settle after a few workgroups, so nearly every wave finds them
// there and ends without another access; the others read the word again
// before they pay for an atomic.
struct OrU32 {
    __device__ uint32_t operator()(uint32_t a, uint32_t b) const { return a | b; }
};
__device__ __forceinline__ unsigned long long* live_word(uint64_t* live) {
    return reinterpret_cast<unsigned long long*>(live) + (blockIdx.x % kLiveLines) * kLiveStep;
}
__device__ __forceinline__ uint64_t live_seen(uint64_t* live) {
    return live ? __hip_atomic_load(live_word(live), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) : ~0ull;
}
__device__ __forceinline__ uint32_t wave_or(uint32_t v) {
    using Reduce = rocprim::warp_reduce<uint32_t, 64>;  // (DPP: no LDS)
    typename Reduce::storage_type storage;
    uint32_t out;
    Reduce().reduce(v, out, storage, OrU32());
    return __builtin_amdgcn_readfirstlane(out);
}
__device__ __forceinline__ void live_join(const Mags& g, uint64_t seen, uint64_t* live) {
    if (!live) return;
    const uint32_t fine = g.fine.mags(), coarse = g.coarse.mags();
    if (__ballot(((fine & ~(uint32_t)seen) | (coarse & ~(uint32_t)(seen >> 32))) != 0) == 0) return;
    const uint64_t all = ((uint64_t)wave_or(coarse) << 32) | wave_or(fine);
    if ((threadIdx.x & 63) != 0) return;
    unsigned long long* w = live_word(live);
    if (all & ~__hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicOr(w, (unsigned long long)all);
}

// In a decompressing tile a point's slot holds the bit pattern of its code
// until the point is reconstructed.
__device__ __forceinline__ float code_slot(int32_t q, float) { return __int_as_float(q); }
__device__ __forceinline__ double code_slot(int32_t q, double) {
    return __longlong_as_double((long long)(uint32_t)q);
}
__device__ __forceinline__ int32_t slot_code(float v) { return __float_as_int(v); }
__device__ __forceinline__ int32_t slot_code(double v) { return (int32_t)(uint32_t)__double_as_longlong(v); }

template <typename T>
struct LevelEb {
    T eb_r[4], ebx2[4];
};

}  // namespace
}  // namespace pa
