// Kernels on either side of the linear: activation staging and the
// QuantizeLinear / DequantizeLinear boundaries.  All HBM-bound elementwise or
// per-row work.
#include "common.h"
#include "device_math.h"
#include "wave_ops.h"

namespace vxhip {

// ---- activation staging -----------------------------------------------------
// Copies raw I8/U8 rows into a 16-byte aligned, zero padded signed buffer and
// writes each row's sum of signed bytes (the operand-sum term of the
// zero-point fold, cf. native/src/kernels/qlinear_vnni_kernel.inc:113-116).
// One wavefront per row.
__global__ __launch_bounds__(256) void stage_activations_kernel(
        const uint8_t* __restrict__ x, uint32_t rows, uint32_t k, uint32_t flip,
        int8_t* __restrict__ staged, uint32_t ld, int32_t* __restrict__ rowsum) {
    const uint32_t row = blockIdx.x * 4u + (threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    if (row >= rows) return;
    const uint8_t* src = x + (size_t)row * k;
    int32_t sum = 0;
    for (uint32_t kk = lane; kk < ld; kk += 64u) {
        int8_t v = 0;
        if (kk < k) v = (int8_t)(src[kk] ^ (flip ? 0x80u : 0u));
        sum += v;
        if (staged) staged[(size_t)row * ld + kk] = v;
    }
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_down(sum, off, 64);
    if (lane == 0 && rowsum) rowsum[row] = sum;
}

VxHipStatus launch_stage_activations(hipStream_t s, const void* x, uint32_t rows, uint32_t k,
                                     bool flip, int8_t* staged, uint32_t ld, int32_t* rowsum) {
    hipLaunchKernelGGL(stage_activations_kernel, dim3((rows + 3u) / 4u), dim3(256), 0, s,
                       (const uint8_t*)x, rows, k, flip ? 1u : 0u, staged, ld, rowsum);
    VXHIP_TRY(hipGetLastError());
    return VXHIP_OK;
}

// one thread per 16-byte chunk of a row
__global__ __launch_bounds__(256) void unblock_activations_kernel(const int8_t* __restrict__ blocked,
                                                                  uint32_t rows, uint32_t chunks,
                                                                  int8_t* __restrict__ row_major, uint32_t ld) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= rows * chunks) return;
    const uint32_t row = i / chunks, chunk = i % chunks;
    *reinterpret_cast<uint4*>(row_major + (size_t)row * ld + chunk * 16u) =
        *reinterpret_cast<const uint4*>(blocked + ((size_t)chunk * kOperandOrderRows + row) * 16u);
}

VxHipStatus launch_unblock_activations(hipStream_t s, const int8_t* blocked, uint32_t rows, uint32_t k,
                                       int8_t* row_major, uint32_t ld) {
    const uint32_t chunks = (k + 15u) / 16u;
    if (rows > kOperandOrderRows || ld < chunks * 16u || (ld % 16u) != 0u || ((uintptr_t)blocked % 16u) != 0u ||
        ((uintptr_t)row_major % 16u) != 0u)
        return VXHIP_INVALID_ARGUMENT;
    if (!rows) return VXHIP_OK;
    hipLaunchKernelGGL(unblock_activations_kernel, dim3((rows * chunks + 255u) / 256u), dim3(256), 0, s, blocked,
                       rows, chunks, row_major, ld);
    VXHIP_TRY(hipGetLastError());
    return VXHIP_OK;
}

__global__ __launch_bounds__(256) void fill_u32_kernel(uint32_t* p, uint32_t count, uint32_t value) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) p[i] = value;
}

VxHipStatus launch_fill_u32(hipStream_t s, uint32_t* p, uint32_t count, uint32_t value) {
    if (!count) return VXHIP_OK;
    hipLaunchKernelGGL(fill_u32_kernel, dim3((count + 255u) / 256u), dim3(256), 0, s, p, count, value);
    VXHIP_TRY(hipGetLastError());
    return VXHIP_OK;
}

// ---- exactness proof of the short division ------------------------------------
// Division by a fixed divisor scales exactly with the dividend's exponent (as long as nothing
// leaves the normal range), so trying all 2^23 mantissas at one exponent decides it for every
// dividend.  Thread t checks mantissas 4t .. 4t+3.
__global__ __launch_bounds__(256) void division_proof_kernel(float s, float r, uint32_t* counters) {
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;
    uint32_t bad1 = 0, bad2 = 0;
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) {
        const float p = __uint_as_float(0x3f800000u | (t * 4u + i));
        const float want = __fdiv_rn(p, s);
        bad1 += div_by_uniform_once(p, s, r) != want;
        bad2 += div_by_uniform(p, s, r) != want;
    }
    if (bad1) atomicAdd(counters, bad1);
    if (bad2) atomicAdd(counters + 1, bad2);
}

VxHipStatus launch_division_proof(hipStream_t s, float divisor, float recip, uint32_t* counters) {
    VxHipStatus st = launch_fill_u32(s, counters, 2, 0);
    if (st != VXHIP_OK) return st;
    hipLaunchKernelGGL(division_proof_kernel, dim3((1u << 23) / 4u / 256u), dim3(256), 0, s, divisor, recip,
                       counters);
    VXHIP_TRY(hipGetLastError());
    return VXHIP_OK;
}

// ---- QuantizeLinear / DequantizeLinear --------------------------------------
// q = saturate(ties-to-even(f32(x / s) + f32(zp))); NaN -> zp; +-Inf saturate
// (native/src/kernels/quantize_linear_ops.inc:156-169).
__global__ __launch_bounds__(256) void quantize_kernel(const float* __restrict__ x, uint32_t n,
                                                       uint8_t* __restrict__ y, float scale,
                                                       int32_t zp, int32_t lo, int32_t hi) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float v = x[i];
    int32_t q;
    if (v != v) {
        q = zp;
    } else {
        const float t = __fadd_rn(__fdiv_rn(v, scale), (float)zp);
        if (t <= (float)lo) q = lo;
        else if (t >= (float)hi) q = hi;
        else q = (int32_t)__builtin_rintf(t);
    }
    y[i] = (uint8_t)q;
}

// y = f32((double)(q - zp) * (double)s)   (quantize_linear_ops.inc:9-16)
__global__ __launch_bounds__(256) void dequantize_kernel(const uint8_t* __restrict__ x, uint32_t n,
                                                         float scale, int32_t zp, uint32_t is_i8,
                                                         float* __restrict__ y) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int32_t q = is_i8 ? (int32_t)(int8_t)x[i] : (int32_t)x[i];
    y[i] = (float)((double)(q - zp) * (double)scale);
}

// RequantizeLinear: q' = saturate(ties-to-even(f32(f32(f32(q - zp_in) * m) + f32(zp_out)))), m = f32(s_in / s_out)
// formed by the host (native/src/kernels/portable_inference_kernels.inc:2437-2463); 16 bytes per thread
// where the tensors allow it.
__device__ __forceinline__ uint32_t requantize_byte(uint32_t byte, uint32_t in_i8, int32_t zp_in, float m, float zp_out_f,
                                                    float lo_f, float hi_f) {
    const int32_t q = in_i8 ? (int32_t)(int8_t)byte : (int32_t)byte;
    const float t = __fadd_rn(__fmul_rn((float)(q - zp_in), m), zp_out_f);
    // (t is finite: a byte difference times a finite multiplier plus a byte)
    return (uint32_t)(int32_t)__builtin_rintf(fminf(fmaxf(t, lo_f), hi_f)) & 255u;
}
__global__ __launch_bounds__(256) void requantize_kernel(const uint8_t* __restrict__ x, uint32_t n, uint8_t* __restrict__ y,
                                                         float m, int32_t zp_in, int32_t zp_out, uint32_t in_i8,
                                                         uint32_t out_i8, uint32_t vectors) {
    const float zp_out_f = (float)zp_out, lo_f = out_i8 ? -128.0f : 0.0f, hi_f = out_i8 ? 127.0f : 255.0f;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < vectors) {
        const uint4 v = reinterpret_cast<const uint4*>(x)[i];
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        uint32_t o[4];
#pragma unroll
        for (int d = 0; d < 4; d++) {
            o[d] = 0u;
#pragma unroll
            for (int b = 0; b < 4; b++)
                o[d] |= requantize_byte((w[d] >> (8 * b)) & 255u, in_i8, zp_in, m, zp_out_f, lo_f, hi_f) << (8 * b);
        }
        reinterpret_cast<uint4*>(y)[i] = make_uint4(o[0], o[1], o[2], o[3]);
    } else {
        const uint32_t e = vectors * 16u + (i - vectors);  // the tail (or everything, for unaligned tensors) byte by byte
        if (e < n) y[e] = (uint8_t)requantize_byte(x[e], in_i8, zp_in, m, zp_out_f, lo_f, hi_f);
    }
}

VxHipStatus launch_requantize(hipStream_t s, const void* x, uint32_t n, void* y, float multiplier, int32_t zp_in,
                              int32_t zp_out, bool in_i8, bool out_i8) {
    if (!n) return VXHIP_OK;
    const bool aligned = ((uintptr_t)x % 16u) == 0u && ((uintptr_t)y % 16u) == 0u;
    const uint32_t vectors = aligned ? n / 16u : 0u;
    const uint32_t threads = vectors + (n - vectors * 16u);
    hipLaunchKernelGGL(requantize_kernel, dim3((threads + 255u) / 256u), dim3(256), 0, s, (const uint8_t*)x, n,
                       (uint8_t*)y, multiplier, zp_in, zp_out, in_i8 ? 1u : 0u, out_i8 ? 1u : 0u, vectors);
    VXHIP_TRY(hipGetLastError());
    return VXHIP_OK;
}

VxHipStatus launch_quantize(hipStream_t s, const float* x, uint32_t n, void* y, float scale,
                            int32_t zp, bool is_i8) {
    if (!n) return VXHIP_OK;
    hipLaunchKernelGGL(quantize_kernel, dim3((n + 255u) / 256u), dim3(256), 0, s, x, n,
                       (uint8_t*)y, scale, zp, is_i8 ? -128 : 0, is_i8 ? 127 : 255);
    VXHIP_TRY(hipGetLastError());
    return VXHIP_OK;
}

VxHipStatus launch_dequantize(hipStream_t s, const void* x, uint32_t n, float scale, int32_t zp,
                              bool is_i8, float* y) {
    if (!n) return VXHIP_OK;
    hipLaunchKernelGGL(dequantize_kernel, dim3((n + 255u) / 256u), dim3(256), 0, s,
                       (const uint8_t*)x, n, scale, zp, is_i8 ? 1u : 0u, y);
    VXHIP_TRY(hipGetLastError());
    return VXHIP_OK;
}

}  // namespace vxhip
