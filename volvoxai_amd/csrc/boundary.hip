// Kernels on either side of the linear: activation staging and the
// QuantizeLinear / DequantizeLinear boundaries.  All HBM-bound elementwise or
// per-row work.
#include "common.h"
#include "device_math.h"
#include "wave_ops.h"

namespace vxhip {

// ---- activation staging -----------------------------------------------------
// What a QLinear's kernels read in place of its rows: signed codes in 16-byte aligned, zero padded rows, and each
// row's sum of them where weights have zero points (the operand-sum term of the zero-point fold, cf.
// native/src/kernels/qlinear_vnni_kernel.inc:113-116).  Bytes are copied (top bits flipped where they are
// unsigned); the f32 rows of a QuantizeLinear in front are quantized on the way, so that the two are one launch.
//
// Bound by the latency of a launch and of its loads until there are tens of megabytes, so a row's pieces are all
// requested before the first is used: a wavefront a row and 16 bytes a lane (bytes), or T threads a row and four
// elements a thread (f32).  A byte a lane and pass, behind a quantization launch of its own, took 6.5 + 2.3 us of the
// 15.3 us of 77 f32 rows of 1001 -> 1531 with row sums; that call is 10.3 now.  Whole calls of up to 32 rows, drawn
// lengths of 256 to 4096: f32 rows to unsigned codes 10.6 -> 6.0 us, bytes with row sums 7.9 -> 5.9, bytes of odd
// lengths 8.4 -> 6.5.
typedef uint32_t dword_any __attribute__((aligned(1)));
typedef float v4f_any __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ int32_t wave_sum_i32(int32_t v) {
    v += lane_exchange<kDppXor1>(v);
    v += lane_exchange<kDppXor2>(v);
    v += lane_exchange<kDppHalfMirror>(v);
    v += lane_exchange<kDppMirror>(v);
    return __builtin_amdgcn_readlane(v, 0) + __builtin_amdgcn_readlane(v, 16) + __builtin_amdgcn_readlane(v, 32) +
           __builtin_amdgcn_readlane(v, 48);
}

__global__ __launch_bounds__(256) void stage_activations_kernel(
        const uint8_t* __restrict__ x, uint32_t rows, uint32_t k, uint32_t flip_mask,
        int8_t* __restrict__ staged, uint32_t ld, int32_t* __restrict__ rowsum) {
    const uint32_t row = blockIdx.x * 4u + (threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    if (row >= rows) return;
    const uint8_t* src = x + (size_t)row * k;
    const uint32_t chunks = (k + 15u) / 16u;
    int32_t sum = 0;
    for (uint32_t c0 = lane; c0 - lane < chunks; c0 += 256u) {
        v4i v[4];
#pragma unroll
        for (uint32_t i = 0; i < 4u; i++) {
            const uint32_t at = (c0 + i * 64u) * 16u;
            v[i] = v4i{0, 0, 0, 0};
            if (at + 16u <= k) {
#pragma unroll
                for (uint32_t d = 0; d < 4u; d++)
                    v[i][d] = (int)(*reinterpret_cast<const dword_any*>(src + at + d * 4u) ^ flip_mask);
            } else if (at < k && k >= 4u) {
                // the row's last chunk by dwords, the last of them moved to where the row ends
#pragma unroll
                for (uint32_t d = 0; d < 4u; d++) {
                    const uint32_t want = at + d * 4u, from = min(want, k - 4u), past = (want - from) * 8u;
                    const uint32_t bytes = *reinterpret_cast<const dword_any*>(src + from) ^ flip_mask;
                    v[i][d] = past < 32u ? (int)(bytes >> past) : 0;
                }
            } else if (at < k) {
                for (uint32_t e = 0; e < k; e++) v[i][0] |= (int)((src[e] ^ (flip_mask & 0xffu)) << (8u * e));
            }
        }
#pragma unroll
        for (uint32_t i = 0; i < 4u; i++) {
            const uint32_t c = c0 + i * 64u;
#pragma unroll
            for (uint32_t d = 0; d < 4u; d++) sum = __builtin_amdgcn_sdot4(v[i][d], 0x01010101, sum, false);
            if (staged && c < chunks) *reinterpret_cast<v4i*>(staged + (size_t)row * ld + c * 16u) = v[i];
        }
    }
    if (rowsum) {
        sum = wave_sum_i32(sum);
        if (lane == 0u) rowsum[row] = sum;
    }
}

VxHipStatus launch_stage_activations(hipStream_t s, const void* x, uint32_t rows, uint32_t k,
                                     bool flip, int8_t* staged, uint32_t ld, int32_t* rowsum) {
    // (whole 16-byte chunks are written)
    if (staged && (ld != (k + 15u) / 16u * 16u || ((uintptr_t)staged % 16u) != 0u)) return VXHIP_INVALID_ARGUMENT;
    hipLaunchKernelGGL(stage_activations_kernel, dim3((rows + 3u) / 4u), dim3(256), 0, s,
                       (const uint8_t*)x, rows, k, flip ? 0x80808080u : 0u, staged, ld, rowsum);
    VXHIP_TRY(hipGetLastError());
    return VXHIP_OK;
}

// What a QuantizeLinear's kernels are told.  recip: the scale's reciprocal, correctly rounded, or zero where the scale is so
// small or large that every element takes a division of its own.
struct QuantizeRule {
    float scale, recip;
    int32_t zp, lo, hi;
    uint32_t flip;
    __device__ __forceinline__ uint32_t code(float v) const {
        const int32_t q = recip != 0.0f ? quantize_code<true>(v, scale, recip, zp, lo, hi)
                                        : quantize_code<false>(v, scale, recip, zp, lo, hi);
        return ((uint32_t)q ^ flip) & 0xffu;
    }
};
QuantizeRule quantize_rule(float scale, int32_t zp, bool is_i8, uint32_t flip) {
    // (1 / s in double is within 2^-53 of the true quotient, which no f32 rounding boundary is that close to)
    const bool near = scale >= 0x1p-60f && scale <= 0x1p60f;  // fast_div_in_range
    return QuantizeRule{scale, near ? (float)(1.0 / (double)scale) : 0.0f, zp, is_i8 ? -128 : 0, is_i8 ? 127 : 255, flip};
}

__device__ __forceinline__ uint32_t quantized4(const float (&v)[4], const QuantizeRule& rule) {
    uint32_t codes = 0u;
#pragma unroll
    for (uint32_t e = 0; e < 4u; e++) codes |= rule.code(v[e]) << (8u * e);
    return codes;
}
// elements j .. j + 3 of a row of k (zeros past its end)
__device__ __forceinline__ void take4(const float* src, uint32_t j, uint32_t k, float (&v)[4]) {
    if (j + 4u <= k) {
        const v4f_any q = *reinterpret_cast<const v4f_any*>(src + j);
#pragma unroll
        for (uint32_t e = 0; e < 4u; e++) v[e] = q[e];
    } else {
#pragma unroll
        for (uint32_t e = 0; e < 4u; e++) v[e] = j + e < k ? src[j + e] : 0.0f;
    }
}
// the codes of elements past the row's end are zero, not the zero point's
__device__ __forceinline__ uint32_t codes_inside(uint32_t codes, uint32_t j, uint32_t k) {
    return j + 4u <= k ? codes : j >= k ? 0u : codes & ((1u << (8u * (k - j))) - 1u);
}

// Rows that are whole chunks and no sums: the elements in one run, four a thread where there are many.  (Up to a few
// hundred thousand every one has a thread of its own: four quotients in a thread are 0.1 to 0.4 us longer than one.)
__global__ __launch_bounds__(256) void quantize_run_kernel(const float* __restrict__ x, uint32_t quads, QuantizeRule rule,
                                                           uint32_t* __restrict__ codes) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= quads) return;
    const v4f_any q = reinterpret_cast<const v4f_any*>(x)[i];
    const float v[4] = {q[0], q[1], q[2], q[3]};
    codes[i] = quantized4(v, rule);
}
__global__ __launch_bounds__(256) void quantize_kernel(const float* __restrict__ x, uint32_t n,
                                                       uint8_t* __restrict__ y, QuantizeRule rule) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = (uint8_t)rule.code(x[i]);
}

// T threads a row (64 or 256), 256 / T rows a workgroup; PASSES pieces of four elements a thread are requested
// together.  Without sums a workgroup takes the pieces of one pass, blockIdx.y.
template <int T, uint32_t PASSES, bool SUMS>
__global__ __launch_bounds__(256) void quantize_rows_kernel(const float* __restrict__ x, uint32_t rows, uint32_t k,
                                                            QuantizeRule rule, int8_t* __restrict__ staged, uint32_t ld,
                                                            int32_t* __restrict__ rowsum) {
    static_assert(SUMS || PASSES == 1u, "a pass a workgroup");
    const uint32_t row = blockIdx.x * (256u / T) + threadIdx.x / T, t = threadIdx.x % T;
    if (row >= rows) return;  // (T = 256: never)
    const float* src = x + (size_t)row * k;
    int8_t* dst = staged + (size_t)row * ld;
    if constexpr (!SUMS) {
        const uint32_t j = (blockIdx.y * T + t) * 4u;
        if (j >= ld) return;
        float v[4];
        take4(src, j, k, v);
        *reinterpret_cast<uint32_t*>(dst + j) = codes_inside(quantized4(v, rule), j, k);
    } else {
        int32_t sum = 0;
        for (uint32_t first = 0; first < ld; first += PASSES * 4u * T) {
            float v[PASSES][4];
#pragma unroll
            for (uint32_t i = 0; i < PASSES; i++) take4(src, first + (i * T + t) * 4u, k, v[i]);
#pragma unroll
            for (uint32_t i = 0; i < PASSES; i++) {
                const uint32_t j = first + (i * T + t) * 4u;
                const uint32_t codes = codes_inside(quantized4(v[i], rule), j, k);
                sum = __builtin_amdgcn_sdot4((int)codes, 0x01010101, sum, false);
                if (j < ld) *reinterpret_cast<uint32_t*>(dst + j) = codes;
            }
        }
        sum = wave_sum_i32(sum);
        if constexpr (T == 64) {
            if (t == 0u) rowsum[row] = sum;
        } else {
            __shared__ int32_t sums[4];
            if ((t & 63u) == 0u) sums[t >> 6] = sum;
            __syncthreads();
            if (t == 0u) rowsum[row] = (sums[0] + sums[1]) + (sums[2] + sums[3]);
        }
    }
}

// Where the line lies, us of a call with its linear of 1024 channels, an element a thread | four: 3 x 1024 4.6 | 5.0,
// 8 x 4096 6.7 | 7.0, 32 x 4096 8.8 | 9.0, 512 x 256 6.5 | 6.7, 128 x 2048 9.94 | 10.03, 64 x 4096 13.66 | 13.73; past it four
// are up to 6 % faster (2323 x 768 9.9 | 9.4).
constexpr uint32_t kRunOfElements = 1u << 18;

VxHipStatus launch_quantize_rows(hipStream_t s, const float* x, uint32_t rows, uint32_t k, float scale, int32_t zp,
                                 bool is_i8, int8_t* staged, uint32_t ld, int32_t* rowsum) {
    if (ld != (k + 15u) / 16u * 16u || ((uintptr_t)staged % 16u) != 0u || (uint64_t)rows * k > UINT32_MAX)
        return VXHIP_INVALID_ARGUMENT;
    const QuantizeRule rule = quantize_rule(scale, zp, is_i8, is_i8 ? 0u : 0x80u);
#define VXHIP_QUANTIZE_ROWS(T, PASSES, SUMS)                                                                              \
    hipLaunchKernelGGL((quantize_rows_kernel<T, PASSES, SUMS>),                                                           \
                       dim3((rows + 256u / T - 1u) / (256u / T), SUMS ? 1u : (ld + 4u * T - 1u) / (4u * T)), dim3(256), 0, \
                       s, x, rows, k, rule, staged, ld, rowsum)
    if (!rowsum && ld == k && rows * k <= kRunOfElements) {
        hipLaunchKernelGGL(quantize_kernel, dim3((rows * k + 255u) / 256u), dim3(256), 0, s, x, rows * k, (uint8_t*)staged,
                           rule);
    } else if (!rowsum && ld == k) {
        const uint32_t quads = rows * (k / 4u);
        hipLaunchKernelGGL(quantize_run_kernel, dim3((quads + 255u) / 256u), dim3(256), 0, s, x, quads, rule,
                           (uint32_t*)staged);
    } else if (!rowsum) {
        if (ld <= 512u) VXHIP_QUANTIZE_ROWS(64, 1u, false);
        else VXHIP_QUANTIZE_ROWS(256, 1u, false);
    } else {
        // (a pass past the row's end divides zeros: as many as the row has, up to four)
        if (ld <= 256u) VXHIP_QUANTIZE_ROWS(64, 1u, true);
        else if (ld <= 1024u) VXHIP_QUANTIZE_ROWS(256, 1u, true);
        else if (ld <= 2048u) VXHIP_QUANTIZE_ROWS(256, 2u, true);
        else VXHIP_QUANTIZE_ROWS(256, 4u, true);
    }
#undef VXHIP_QUANTIZE_ROWS
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

__global__ void publish_u32_kernel(const uint32_t* p, uint32_t* host) {
    __hip_atomic_store(host, *p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

VxHipStatus launch_publish_u32(hipStream_t s, const uint32_t* p, uint32_t* host) {
    hipLaunchKernelGGL(publish_u32_kernel, dim3(1), dim3(1), 0, s, p, host);
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
                       (uint8_t*)y, quantize_rule(scale, zp, is_i8, 0u));
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
