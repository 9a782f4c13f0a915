// Device-side scalar rules of the W8A8 contract.  Every f32 operation that the
// reference rounds separately is written with an explicit round-to-nearest
// intrinsic, so the compiler can neither contract a multiply-add into an FMA
// nor reassociate: a fused value can cross a ties-to-even boundary and change
// the output byte (reference: native/src/kernels/w8a8_affine.h:133-144).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace vxhip {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));

// A store of output that nothing in the launch reads again, for launches whose whole output would
// otherwise sit dirty in the L2s until the kernel ends and leave in one burst behind the last wave
// (`streamed`, uniform over the launch): it then goes out while the kernel still runs.  Measured on the
// 256 x 256 requantizing tile at K=N=4096: 3072 / 4096 / 6144 / 8192 rows 0.5-1.3 us faster, 16384 rows the
// same, 2048 rows and fewer 0.4 us slower (their stores cover half lines, which the L2 otherwise merges).
// (STREAMED is a compile-time tag: under a run-time condition the compiler folds the two stores into a plain one)
template <bool STREAMED, class T>
__device__ __forceinline__ void store_stream(T* p, const T& v) {
    if constexpr (STREAMED) __builtin_nontemporal_store(v, p);
    else *p = v;
}

__device__ __forceinline__ bool scale_valid(float v) {
    // finite and strictly positive (w8a8_affine.h:63-65)
    return v > 0.0f && v < __builtin_inff();
}

// multiplier = f32(f32(s_in * s_w) / s_out)   (w8a8_affine.h:155-181)
__device__ __forceinline__ float requant_multiplier(float s_in, float s_w, float s_out) {
    return __fdiv_rn(__fmul_rn(s_in, s_w), s_out);
}

// p / s for a divisor that is the same for the whole launch, given r = RN(1/s)
// from the host.  Two Newton corrections with exact FMA residuals: after the
// first the quotient is faithful, and Markstein's theorem then makes the second
// the correctly rounded quotient, i.e. the same bits as an IEEE division -- as
// long as nothing under- or overflows, which fast_div_in_range() guarantees.
// Five full-rate operations instead of the ~11 of the generic divide sequence.
__device__ __forceinline__ float div_by_uniform(float p, float s, float r) {
    float q = __fmul_rn(p, r);
    float e = __fmaf_rn(-q, s, p);
    q = __fmaf_rn(e, r, q);
    e = __fmaf_rn(-q, s, p);
    return __fmaf_rn(e, r, q);
}

// The same with one correction.  Markstein's theorem makes it exact whenever the first product
// is already faithful; callers use it only for divisors where launch_division_proof counted no
// mismatch over all dividend mantissas.
__device__ __forceinline__ float div_by_uniform_once(float p, float s, float r) {
    const float q = __fmul_rn(p, r);
    const float e = __fmaf_rn(-q, s, p);
    return __fmaf_rn(e, r, q);
}

// Operands between 2^-60 and 2^60 keep every intermediate of div_by_uniform a
// normal number (quotient within 2^+-120, residuals 2^-24 below the operands).
__device__ __forceinline__ bool fast_div_in_range(float v) {
    return v >= 0x1p-60f && v <= 0x1p60f;
}

// t = f32(f32(acc) * mult) + f32(zp)          (w8a8_affine.h:139-144)
__device__ __forceinline__ float transform_accumulator(int32_t acc, float mult, float zp_f) {
    return __fadd_rn(__fmul_rn((float)acc, mult), zp_f);
}

// Saturating ties-to-even round into [lo, hi]; NaN maps to the zero point
// (w8a8_affine.h:114-131).  v_rndne_f32 is ties-to-even and equals the
// reference's floor-based rule for every value strictly inside the range.
__device__ __forceinline__ int32_t requantize(float t, float lo_f, float hi_f, int32_t zp) {
    if (t != t) return zp;
    float c = fminf(fmaxf(t, lo_f), hi_f);
    return (int32_t)__builtin_rintf(c);
}

// The largest magnitude of a row is kept as the bits of an f32 without its sign: their integer order is the order of
// the magnitudes, with infinities and then NaN above every finite value.
__device__ __forceinline__ uint32_t magnitude_bits(float v) { return __float_as_uint(v) & 0x7fffffffu; }
constexpr uint32_t kNotFinite = 0x7f800000u;  // and everything above

// scale = max|v| / 127 (1 for a zero row and for one that is not finite, floored at 2^-126): the quotient of a true
// division for every finite maximum (every mantissa compared, in the middle, at the floor and at the largest exponent)
__device__ __forceinline__ float row_code_scale(uint32_t maximum) {
    const float scale = maximum == 0u || maximum >= kNotFinite ? 1.0f : div_by_uniform(__uint_as_float(maximum), 127.0f, 0x1.020408p-7f);
    return scale < 0x1p-126f ? 0x1p-126f : scale;
}

// The codes of one row: ties-to-even(v / scale) clamped to +-127, with the bits of a true f32 division by the row's
// scale but without its cost.  An exact division is some twenty instructions, some of them at a quarter of
// the rate; the reciprocal of a divisor that all elements share leaves five (div_by_uniform).  What makes those exact
// here: the first product is at most 1.5 units in the last place off, the first correction leaves a faithful quotient
// (its residual is exact, or off by 2^-24 of itself, which the result cannot show), and the correction of a
// faithful quotient by an exact residual with a correctly rounded reciprocal is the correctly rounded quotient (Markstein, IBM
// J. Res. Dev. 34, 1990).  A residual is exact while it is no denormal, so small scales (which are at least
// 2^-126) and their elements are scaled up first, exactly; a quotient below 1/4, where this may fail, is code 0
// either way.  (Scales are at most 2^121: their reciprocals are normal.)  Row preparation of 24 x 14336 4.3 -> 3.3 us, of
// 2048 x 8192 15.6 -> 14.0.
struct CodeDivisor {
    float lift, scale, recip;
    __device__ __forceinline__ explicit CodeDivisor(float row_scale) {
        lift = row_scale < 0x1p-60f ? 0x1p64f : 1.0f;
        scale = __fmul_rn(row_scale, lift);
        // the correctly rounded reciprocal of every mantissa but one from any start within two units in the last place
        // (followed over all of them); of the largest mantissa it may be one unit low, and then some of its codes are others
        recip = __builtin_amdgcn_rcpf(scale);
#pragma unroll
        for (int i = 0; i < 2; i++) recip = __fmaf_rn(__fmaf_rn(-scale, recip, 1.0f), recip, recip);
        const uint32_t bits = __float_as_uint(scale);
        if ((bits & 0x7fffffu) == 0x7fffffu) recip = __uint_as_float((253u - (bits >> 23)) << 23 | 1u);
    }
    // the divisor of another lane's row, uniform over the wavefront
    __device__ __forceinline__ CodeDivisor(const CodeDivisor& d, int lane) {
        auto of = [&](float v) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane)); };
        lift = of(d.lift), scale = of(d.scale), recip = of(d.recip);
    }
    // the code in the lowest byte; the others are not zero
    __device__ __forceinline__ uint32_t code_bits(float v) const {
        const float q = div_by_uniform(__fmul_rn(v, lift), scale, recip);
        // (adding 1.5 * 2^23 rounds to an integer, ties to even, and leaves it in the sum's lowest bits)
        return __float_as_uint(__fadd_rn(fminf(fmaxf(q, -127.0f), 127.0f), 12582912.0f));
    }
    __device__ __forceinline__ uint32_t code(float v) const { return code_bits(v) & 0xffu; }
    __device__ __forceinline__ uint32_t codes4(float a, float b, float c, float d) const {
        const uint32_t lo = __builtin_amdgcn_perm(code_bits(b), code_bits(a), 0x0c0c0400u);
        const uint32_t hi = __builtin_amdgcn_perm(code_bits(d), code_bits(c), 0x0c0c0400u);
        return lo | (hi << 16);
    }
};

// q = saturate(ties-to-even(f32(x / s) + f32(zp))); NaN -> zp; +-Inf saturate
// (native/src/kernels/quantize_linear_ops.inc:156-169).  NEAR: the scale is such that fast_div_in_range: the division by way
// of its reciprocal, as above; elements past any code are brought nearer first, where the corrections would overflow.
template <bool NEAR>
__device__ __forceinline__ int32_t quantize_code(float v, float scale, float recip, int32_t zp, int32_t lo, int32_t hi) {
    if (v != v) return zp;
    float q;
    if constexpr (NEAR) q = div_by_uniform(fminf(fmaxf(v, -1024.0f * scale), 1024.0f * scale), scale, recip);
    else q = __fdiv_rn(v, scale);
    const float t = __fadd_rn(q, (float)zp);
    return t <= (float)lo ? lo : t >= (float)hi ? hi : (int32_t)__builtin_rintf(t);
}

__device__ __forceinline__ uint32_t pack4_bytes(int32_t a, int32_t b, int32_t c, int32_t d) {
    return (uint32_t)(a & 255) | ((uint32_t)(b & 255) << 8) | ((uint32_t)(c & 255) << 16) |
           ((uint32_t)(d & 255) << 24);
}

}  // namespace vxhip
