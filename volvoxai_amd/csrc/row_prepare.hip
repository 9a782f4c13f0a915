// The activation preparation of PackedLinear rows (native/src/kernels/packed_linear_ops.inc:97-217,
// 1574-1597), alone or behind a decoder's row operation, one workgroup per row:
//
//   plain    the f32 row itself
//   norm     RMSNorm (native/src/kernels/softmax_rmsnorm.inc:3-17: double accumulation, x * inv_std * gain
//            in double, one rounding to f32), the row first updated in place by a residual add if asked
//   swiglu   silu(gate) * up of a row [gate | up]
//
// then scale = max|v| / 127 (1 for a zero row, floored at 2^-126) and code = ties-to-even(v / scale) clamped to
// +-127, with the quotients of true f32 divisions (CodeDivisor; a plain product with a reciprocal moves half-way values,
// ibid. :34-36).  A
// row holding NaN or Inf gets zero codes and a NaN scale, which makes every output of that row NaN
// downstream as the reference requires (:1495).
//
// Few rows are bound by latency: a launch, the row's first touch, a reduction or two.  So a thread holds its
// elements in registers from the load to the codes (16-byte loads, all requested before the first is used; four
// codes per store), a reduction costs one barrier, nothing but its slots is in LDS, and a workgroup has four
// wavefronts or, of more, no more than the row has 64 16-byte pieces.  In a recorded decode step of 32 rows, cost per launch against
// kernels that walked LDS copies of the row an element at a time with 1024 threads: RMSNorm of 1024 elements
// 4.65 -> 3.0 us, SwiGLU of 3072 4.5 -> 3.3, plain 2048 3.8 -> 2.9 (a launch that reads one row of its
// predecessor and writes it back costs 2.2-2.9).  Many rows are bound by the rows' bytes
// beside some ten instructions an element: 2048 x 14336 24.9 us, 5.9 TB/s (27.0 with a division instruction sequence an
// element).
#include "common.h"
#include "device_math.h"
#include "row_math.h"
#include "wave_ops.h"

namespace vxhip {
namespace {

// four f32 at an address of any f32 alignment
typedef float v4f_any __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32_any __attribute__((aligned(1)));

struct RowArgs {
    float* x;             // the rows; updated in place where delta is given
    const float* delta;   // norm: residual add in front (may be null)
    const float* gain;    // norm
    double eps;           // norm
    uint32_t d;           // elements of a prepared row (swiglu: the row holds 2 * d)
    int8_t* codes;
    ActivationLayout layout;
    float* scales;
    float* values;        // optional: the f32 rows the codes are made of
};

// elements j .. j + 3 of a row of d (zeros past its end); WHOLE: d is a multiple of four
template <bool WHOLE, bool STREAM = false>
__device__ __forceinline__ v4f row_load(const float* src, uint32_t j, uint32_t d) {
    v4f v = {0.f, 0.f, 0.f, 0.f};
    if (WHOLE ? j < d : j + 4u <= d) {
        if constexpr (STREAM) v = __builtin_nontemporal_load(reinterpret_cast<const v4f_any*>(src + j));
        else v = *reinterpret_cast<const v4f_any*>(src + j);
    } else if constexpr (!WHOLE) {
#pragma unroll
        for (uint32_t e = 0; e < 4u; e++)
            if (j + e < d) v[e] = src[j + e];
    }
    return v;
}
template <bool WHOLE>
__device__ __forceinline__ void row_store(float* dst, uint32_t j, uint32_t d, const v4f& v) {
    if (WHOLE ? j < d : j + 4u <= d) {
        *reinterpret_cast<v4f_any*>(dst + j) = v;
    } else if constexpr (!WHOLE) {
#pragma unroll
        for (uint32_t e = 0; e < 4u; e++)
            if (j + e < d) dst[j + e] = v[e];
    }
}

// T threads, NB passes of 4 * T elements held in registers; WHOLE: rows and their codes are whole groups of four.
// Plain rows may be longer than that: the rest is read again for its codes.
template <RowOp OP, int T, int NB, bool WHOLE>
__global__ __launch_bounds__(T) void row_prepare_kernel(const RowArgs a) {
    static_assert(OP != RowOp::Norm || T == 256, "the sum of squares is ordered for 16 bytes a thread of 256");
    constexpr int WAVES = T / 64;
    constexpr bool STREAM = OP == RowOp::Plain && T == 256;  // (many rows, read once)
    __shared__ uint32_t slots[WAVES];
    const uint32_t row = blockIdx.x, d = a.d;
    float* src = a.x + (size_t)row * (OP == RowOp::Swiglu ? 2u * (size_t)d : d);
    auto at = [&](int i) { return (uint32_t)i * (4u * T) + threadIdx.x * 4u; };
    v4f v[NB];
#pragma unroll
    for (int i = 0; i < NB; i++) v[i] = row_load<WHOLE, STREAM>(src, at(i), d);
    if constexpr (OP == RowOp::Swiglu) {
        v4f up[NB];
#pragma unroll
        for (int i = 0; i < NB; i++) up[i] = row_load<WHOLE>(src + d, at(i), d);
#pragma unroll
        for (int i = 0; i < NB; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) v[i][e] = swiglu_value(v[i][e], up[i][e]);
    }
    if constexpr (OP == RowOp::Norm) {
        __shared__ double norm_slots[4];
        v4f gain[NB];
        if (a.delta) {
            const float* delta = a.delta + (size_t)row * d;
            v4f add[NB];
#pragma unroll
            for (int i = 0; i < NB; i++) add[i] = row_load<WHOLE>(delta, at(i), d);
#pragma unroll
            for (int i = 0; i < NB; i++) gain[i] = row_load<WHOLE>(a.gain, at(i), d);
#pragma unroll
            for (int i = 0; i < NB; i++) {
#pragma unroll
                for (int e = 0; e < 4; e++) v[i][e] = __fadd_rn(v[i][e], add[i][e]);
                row_store<WHOLE>(src, at(i), d, v[i]);
            }
        } else {
#pragma unroll
            for (int i = 0; i < NB; i++) gain[i] = row_load<WHOLE>(a.gain, at(i), d);
        }
        double pair[2] = {0.0, 0.0};
#pragma unroll
        for (int i = 0; i < NB; i++) {
            pair[0] += square(v[i][0]) + square(v[i][1]);
            pair[1] += square(v[i][2]) + square(v[i][3]);
        }
        const double inv_std = rms_inverse(norm_total<256>(pair, norm_slots), d, a.eps);
#pragma unroll
        for (int i = 0; i < NB; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) v[i][e] = rms_scaled(v[i][e], inv_std, gain[i][e]);
    }
    if constexpr (OP != RowOp::Plain) {
        if (a.values) {
#pragma unroll
            for (int i = 0; i < NB; i++) row_store<WHOLE>(a.values + (size_t)row * d, at(i), d, v[i]);
        }
    }

    // one reduction for both questions: what is not finite is above every finite magnitude
    uint32_t maximum = 0u;
    auto offer = [&](const v4f& t) {
#pragma unroll
        for (int e = 0; e < 4; e++) maximum = max(maximum, magnitude_bits(t[e]));
    };
#pragma unroll
    for (int i = 0; i < NB; i++) offer(v[i]);
    if constexpr (OP == RowOp::Plain)
        for (uint32_t j = at(NB); j < d; j += 4u * T) offer(row_load<WHOLE>(src, j, d));
    maximum = wave_max(maximum);
    if ((threadIdx.x & 63u) == 0u) slots[threadIdx.x >> 6] = maximum;
    __syncthreads();
    maximum = slots[0];
#pragma unroll
    for (int w = 1; w < WAVES; w++) maximum = max(maximum, slots[w]);
    const bool bad = maximum >= kNotFinite;
    const float scale = row_code_scale(maximum);
    const CodeDivisor divisor(scale);
    // (elements past d are zeros: the padding of the row's last 16-byte chunk, where the layout has one)
    // (a thread's codes of neighbouring passes are as far apart in either layout, whatever the row)
    int8_t* const first = a.codes + activation_offset(a.layout, row, threadIdx.x * 4u);
    const uint32_t step = 4u * T * (a.layout.operand_order ? kOperandOrderRows : 1u);
    auto put = [&](uint32_t i, const v4f& t) {
        const uint32_t j = at((int)i);
        if (j >= a.layout.ld) return;
        const uint32_t q = bad ? 0u : divisor.codes4(t[0], t[1], t[2], t[3]);
        int8_t* dst = first + i * (size_t)step;
        if (WHOLE || j + 4u <= a.layout.ld) {
            *reinterpret_cast<u32_any*>(dst) = q;
        } else {
            for (uint32_t e = 0; j + e < a.layout.ld; e++) dst[e] = (int8_t)(q >> (8u * e));
        }
    };
#pragma unroll
    for (int i = 0; i < NB; i++) put((uint32_t)i, v[i]);
    if constexpr (OP == RowOp::Plain)
        for (uint32_t i = NB; at((int)i) < a.layout.ld; i++) put(i, row_load<WHOLE>(src, at((int)i), d));
    if (threadIdx.x == 0) a.scales[row] = bad ? __builtin_nanf("") : scale;
}

template <RowOp OP, int T, int NB>
void launch(hipStream_t s, uint32_t rows, const RowArgs& a) {
    // (Rows of 6145 to 10240 elements: LDS that nobody uses, so that six workgroups share a compute unit and not eight.
    // With all rows of a launch resident every one of them loads first and computes then; 2048 x 8192 15.7 against 16.7 us.)
    const size_t lds = OP == RowOp::Plain && T == 256 && (NB == 8 || NB == 10) ? 26u * 1024u : 0u;
    // (a row's codes end where the row does or at the end of a 16-byte chunk)
    if (a.d % 4u == 0u && a.layout.ld % 4u == 0u)
        hipLaunchKernelGGL((row_prepare_kernel<OP, T, NB, true>), dim3(rows), dim3(T), lds, s, a);
    else
        hipLaunchKernelGGL((row_prepare_kernel<OP, T, NB, false>), dim3(rows), dim3(T), lds, s, a);
}

// Many rows: 256 threads, as many passes as the row has (or one more: an idle pass costs 2-4 %, 1246 x 9216 in fourteen
// passes 12.3 us, in ten 11.6).  Few rows (no more than compute units) leave a
// workgroup alone on its compute unit and latency bound: then as many threads as the row has 16-byte
// pieces, up to 1024.
template <RowOp OP>
void launch_op(hipStream_t s, uint32_t rows, const RowArgs& a) {
    const uint32_t d = a.layout.ld > a.d ? a.layout.ld : a.d;
    if constexpr (OP != RowOp::Norm) {
        if (rows <= 256u && d > 1024u) {
            if (d <= 2048u) launch<OP, 512, 1>(s, rows, a);
            else if (d <= 4096u) launch<OP, 1024, 1>(s, rows, a);
            else if (d <= 8192u) launch<OP, 1024, 2>(s, rows, a);
            else launch<OP, 1024, 4>(s, rows, a);
            return;
        }
    }
    if (d <= 1024u) launch<OP, 256, 1>(s, rows, a);
    else if (d <= 2048u) launch<OP, 256, 2>(s, rows, a);
    else if (d <= 3072u) launch<OP, 256, 3>(s, rows, a);
    else if (d <= 4096u) launch<OP, 256, 4>(s, rows, a);
    else if (d <= 6144u) launch<OP, 256, 6>(s, rows, a);
    else if (d <= 8192u) launch<OP, 256, 8>(s, rows, a);
    else if (d <= 10240u) launch<OP, 256, 10>(s, rows, a);
    else if (d <= 12288u) launch<OP, 256, 12>(s, rows, a);
    else if (d <= 14336u) launch<OP, 256, 14>(s, rows, a);
    else launch<OP, 256, 15>(s, rows, a);
}

}  // namespace

VxHipStatus launch_row_prepare(hipStream_t s, RowOp op, float* x, const float* delta, const float* gain, double eps,
                               uint32_t rows, uint32_t d, int8_t* codes, ActivationLayout layout, float* scales,
                               float* values) {
    // (the rows of operand order are whole 16-byte chunks)
    if (layout.operand_order && layout.ld != (d + 15u) / 16u * 16u) return VXHIP_INVALID_ARGUMENT;
    if (op != RowOp::Plain && d > kMaxRowOpLength) return VXHIP_INVALID_ARGUMENT;
    const RowArgs a{x, delta, gain, eps, d, codes, layout, scales, values};
    switch (op) {
        case RowOp::Plain: launch_op<RowOp::Plain>(s, rows, a); break;
        case RowOp::Norm: launch_op<RowOp::Norm>(s, rows, a); break;
        case RowOp::Swiglu: launch_op<RowOp::Swiglu>(s, rows, a); break;
    }
    VXHIP_TRY(hipGetLastError());
    return VXHIP_OK;
}

}  // namespace vxhip
