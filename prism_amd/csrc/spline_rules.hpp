// spline_rules.hpp -- the predictor's formulas and its quantiser, and the
// small device helpers that its kernels share.  Arithmetic is in T (FP64 for
// double fields), evaluated in the reference's order with no FMA contraction,
// so the compressor and the decompressor reproduce identical values.
#pragma once

#include "common.hpp"

namespace pa {
namespace {

constexpr int kThreads = 256;

enum Mode { COMPRESS, DECOMPRESS, TUNE };

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

// The lane id through an opaque move: index arithmetic derived from it in
// one phase of the kernel is not merged with that of another phase and kept
// live in registers between them.
__device__ __forceinline__ int lane_id() {
    int v;
    asm volatile("v_mov_b32 %0, %1" : "=v"(v) : "v"((int)threadIdx.x));
    __builtin_assume(v >= 0 && v < kThreads);
    return v;
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
    T code = (err < (T)0 ? -err : err) * eb_r + (T)1;
    code = copysign(code, err);  // (a negative zero's sign: +-1 / 2 truncates to 0 all the same)
    const int qv = (int)(code / (T)2);
    code = (T)qv;
    v = pred + code * ebx2;
    return qv;
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
