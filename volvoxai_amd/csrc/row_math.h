// The element rules of the row operations in front of a decoder's linears, shared by the row kernels
// (row_prepare.hip) and by the streaming linear when it carries such an operation in its own
// prologue (gemv_stream.hip), so that both give the same bits.
#ifndef VXHIP_ROW_MATH_H
#define VXHIP_ROW_MATH_H

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "wave_ops.h"

namespace vxhip {

// RMSNorm in double, rounded to f32 once per element: y = f32(x * (1 / sqrt(mean(x^2) + eps)) * gain).
//
// The row's sum of squares has one order for every kernel that forms it.  The row is cut into blocks of
// kNormBlock elements; pair p of a block is its elements 2p and 2p + 1; a pair's squares are added, then
// the pairs of the same p over the blocks in ascending order, then the kNormBlock / 2 of these sums as the
// full binary tree over p (neighbours first).  A thread of a 256-thread workgroup holds the pairs 2t and
// 2t + 1 of every block (one 16-byte load), a thread of a 512-thread workgroup the pair t: both trees are
// the same one.
constexpr uint32_t kNormBlock = 1024;

// The pair sums of the workgroup's threads (two of a 256-thread workgroup, one of a 512-thread one) to
// the row's total, in every thread.  `slots`: LDS for THREADS / 64 doubles.  Holds one barrier.
template <int THREADS>
__device__ __forceinline__ double norm_total(const double (&pair)[512 / THREADS], double* slots) {
    static_assert(THREADS == 256 || THREADS == 512, "one or two pairs a thread");
    double v = pair[0];
    if constexpr (THREADS == 256) v += pair[1];
    // (the mirrored exchanges meet lanes that all hold the same partial sum by then: lane ^ 4, lane ^ 8)
    v += lane_exchange<kDppXor1>(v);
    v += lane_exchange<kDppXor2>(v);
    v += lane_exchange<kDppHalfMirror>(v);
    v += lane_exchange<kDppMirror>(v);
    v += lane_down16(v);
    v += lane_down32(v);
    if ((threadIdx.x & 63u) == 0u) slots[threadIdx.x >> 6] = v;
    __syncthreads();
    if constexpr (THREADS == 256) return (slots[0] + slots[1]) + (slots[2] + slots[3]);
    else return ((slots[0] + slots[1]) + (slots[2] + slots[3])) + ((slots[4] + slots[5]) + (slots[6] + slots[7]));
}
__device__ __forceinline__ double square(float v) { return (double)v * (double)v; }
__device__ __forceinline__ double rms_inverse(double total, uint32_t d, double eps) {
    const double var = total / (double)d;
    return 1.0 / sqrt(var + eps);
}
__device__ __forceinline__ float rms_scaled(float v, double inv_std, float gain) {
    return (float)((double)v * inv_std * (double)gain);
}

// SwiGLU: silu(gate) * up with silu(g) = g / (1 + exp(-g)), every step rounded to f32.
__device__ __forceinline__ float swiglu_value(float gate, float up) {
    const float s = __fdiv_rn(gate, __fadd_rn(1.0f, expf(-gate)));
    return __fmul_rn(s, up);
}

}  // namespace vxhip
#endif
