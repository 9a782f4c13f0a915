// PackedLinear of three to eight f32 rows in one launch: the rows' preparation (the rules of row_prepare.hip,
// native/src/kernels/packed_linear_ops.inc:97-217) inside the linear (ibid. :1471-1535), as gemv_row.hip has it for one and
// two.
//
// Split as there: a workgroup of 512 threads owns CH (16, 32 or 64) output channels over all of K, asks for the
// rows and then for its weights, and prepares the rows while those are under way.  The dots are matrix
// instructions, since every weight is used by all rows: a wavefront's 16 bytes a lane are sixteen channels of two
// adjacent 1 KiB blocks (common.h), the A operand of v_mfma_i32_16x16x64_i8 as they come, and the codes lie in LDS with the
// rows' 16-byte chunks side by side, so that a B operand is one conflict-free read.  A scale group's dots leave
// the accumulators as products f32(dot) * (s_a * s_w) and one thread per output adds them in ascending group order, the
// sum the reference forms (packed_linear_ops.inc:1498-1504), bit for bit.
//
// Bound by latency, and by the preparation that every workgroup repeats: of 16384 elements a thread takes 32, 1.5 us
// beside a launch of its own that costs 2.4.
#include "common.h"
#include "device_math.h"
#include "row_math.h"
#include "wave_ops.h"

#include <stdio.h>
#include <string.h>

namespace vxhip {
namespace {

extern __shared__ __attribute__((aligned(16))) char few_lds[];

constexpr int kThreads = 512, kWaves = kThreads / 64;

typedef float v2f_any __attribute__((ext_vector_type(2), aligned(4)));

// K up to NB * 1024, up to RT rows.
template <int GK, bool W4, int CH, int NB, int RT>
__global__ __launch_bounds__(kThreads) void gemv_few_kernel(const LinearArgs a) {
    constexpr int KPAD = NB * 1024, NH = CH / 16;      // halves of a panel
    constexpr int SLAB = W4 ? 128 : 64;                // columns of a pair of blocks
    constexpr int STEPS = SLAB / 32;                   // k-steps of a slab
    constexpr int SPU = GK > STEPS ? GK / STEPS : 1;   // slabs of a unit: whole scale groups
    constexpr int NSUB = GK < STEPS ? STEPS / GK : 1;  // scale groups of a slab
    constexpr int UNITS = KPAD / (SLAB * SPU), NU = (UNITS + kWaves - 1) / kWaves, NL = NU * SPU;
    // slabs of a wavefront that are requested before the rows are looked at
    constexpr int AHEAD = NL * NH <= (NH == 4 ? 16 : 8) ? NL : NH == 4 ? 4 : 8 / NH;
    constexpr int GROUPS = KPAD / (32 * GK), NS = (GROUPS * CH + kThreads - 1) / kThreads;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    constexpr int PARTS = CH < 32 ? 32 / CH : 1, PANELS = CH < 32 ? 1 : CH / 32;  // workgroups per panel, or panels per workgroup
    const uint32_t panel = blockIdx.x / PARTS * PANELS, sub = blockIdx.x % PARTS, ch0 = panel * 32u + sub * CH;
    const uint32_t c = lane & 15, chunk = lane >> 4;  // operand: channel (row) c, 16 bytes `chunk` of 64
    const uint32_t k = a.k, rows = a.rows;

    // the rows (elements past k: zeros; rows past the last: the last): a thread holds the pair 2t of every 1024 elements
    float x[RT][NB][2];
#pragma unroll
    for (int r = 0; r < RT; r++) {
        const float* src = a.x_f32 + (size_t)min((uint32_t)r, rows - 1u) * a.ldx;
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const uint32_t j = (uint32_t)b * 1024u + threadIdx.x * 2u, at = min(j, k - 2u);
            const v2f_any p = *reinterpret_cast<const v2f_any*>(src + at);
            x[r][b][0] = j < k ? (j == at ? p.x : p.y) : 0.0f;
            x[r][b][1] = j + 1u < k ? p.y : 0.0f;
        }
    }
    // (loads return in the order of their issue: the rows have to be asked for before the rest)
    __builtin_amdgcn_sched_barrier(0);
    float sreg[NS];  // the workgroup's group scales, [group][channel]
#pragma unroll
    for (int i = 0; i < NS; i++) {
        const uint32_t e = threadIdx.x + i * kThreads;
        sreg[i] = a.scales_t[(size_t)min(e / CH, a.groups - 1u) * a.n_pad + ch0 + e % CH];
    }
    const int8_t* wp = a.w + (size_t)panel * a.ksteps * 1024u + ((chunk & 1u) * 32u + sub * CH + c) * 16u;
    // slab l of the wavefront
    auto slab_of = [&](int l) { return (uint32_t)(((l / SPU) * kWaves + wave) * SPU + l % SPU); };
    v4i w[AHEAD][NH];
    auto issue = [&](int l) {
        const uint32_t block = min(slab_of(l) * 2u + (chunk >> 1), a.ksteps - 1u);
#pragma unroll
        for (int h = 0; h < NH; h++)
            w[l % AHEAD][h] = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(wp + (size_t)(h / 2 * a.ksteps + block) * 1024u + h % 2 * 256u));
    };
#pragma unroll
    for (int l = 0; l < AHEAD; l++) issue(l);
    __builtin_amdgcn_sched_barrier(0);

    // preparation: scale = max|v| / 127 (1 for a zero row, floored at 2^-126), codes = ties-to-even(v / scale)
    // clamped to +-127 (CodeDivisor); a row that is not finite gets zero codes and a NaN scale
    // [KPAD / 16][RT][16], the rows of a chunk in an order of its own: the codes of one row, written two at a time, would
    // else meet in the same banks
    int8_t* codes = reinterpret_cast<int8_t*>(few_lds);
    auto code_at = [](uint32_t at, uint32_t row) { return (at * RT + (row ^ (at % RT))) * 16u; };
    float* scales = reinterpret_cast<float*>(few_lds + RT * KPAD);         // [groups][CH]
    float* products = scales + (size_t)a.groups * CH;                      // [groups][rows][CH]
    __shared__ __attribute__((aligned(16))) uint32_t slots[RT][kWaves];
    __shared__ float row_scales[RT];
#pragma unroll
    for (int r = 0; r < RT; r++) {
        uint32_t maximum = 0u;
#pragma unroll
        for (int b = 0; b < NB; b++) maximum = max(maximum, max(magnitude_bits(x[r][b][0]), magnitude_bits(x[r][b][1])));
        maximum = wave_max(maximum);
        if (lane == 0) slots[r][wave] = maximum;
    }
    __syncthreads();
    {
        // (a lane a row: the rows' scales and reciprocals cost a wavefront two divisions and not two a row)
        const uint4* mine = reinterpret_cast<const uint4*>(slots[min((uint32_t)lane, (uint32_t)RT - 1u)]);
        const uint4 lo = mine[0], hi = mine[1];
        const uint32_t maximum = max(max(max(lo.x, lo.y), max(lo.z, lo.w)), max(max(hi.x, hi.y), max(hi.z, hi.w)));
        const bool bad = maximum >= kNotFinite;
        const float scale = row_code_scale(maximum);
        const CodeDivisor divisors(scale);
        const uint64_t bad_rows = __ballot(bad);
#pragma unroll
        for (int r = 0; r < RT; r++) {
            const CodeDivisor divisor(divisors, r);
            const bool zeros = (bad_rows >> r) & 1u;
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const uint32_t q = divisor.code(x[r][b][0]) | (divisor.code(x[r][b][1]) << 8);
                const uint32_t j = (uint32_t)b * 1024u + threadIdx.x * 2u;
                *reinterpret_cast<uint16_t*>(codes + code_at(j >> 4, r) + (j & 15u)) = (uint16_t)(zeros ? 0u : q);
            }
        }
        if (threadIdx.x < RT) row_scales[threadIdx.x] = bad ? __builtin_nanf("") : scale;
    }
#pragma unroll
    for (int i = 0; i < NS; i++) {
        const uint32_t e = threadIdx.x + i * kThreads;
        if (e < a.groups * CH) scales[e] = sreg[i];
    }
    // the tail's operand: output o = row * CH + channel
    float bias = 0.0f;
    const uint32_t on = ch0 + threadIdx.x % CH;
    bias = a.bias_f32[on];
    __syncthreads();

    const uint32_t r = min(c, (uint32_t)RT - 1u);
    const float rs = row_scales[r];
    const v4i zero = {0, 0, 0, 0};
    // the lanes of the first block of a slab, and of the second
    const int first = chunk < 2u ? -1 : 0;
#pragma unroll
    for (int u = 0; u < NU; u++) {
        v4i acc[NSUB][NH];
#pragma unroll
        for (int s = 0; s < NSUB; s++)
#pragma unroll
            for (int h = 0; h < NH; h++) acc[s][h] = zero;
#pragma unroll
        for (int i = 0; i < SPU; i++) {
            const int l = u * SPU + i;
            const uint32_t slab = min(slab_of(l), (uint32_t)(KPAD / SLAB) - 1u);
            // the 16-byte chunk of columns that the lane's weights (their low nibbles) belong to
            const uint32_t at = W4 ? (slab * 2u + (chunk >> 1)) * 4u + (chunk & 1u) : slab * 4u + chunk;
            v4i xv[W4 ? 2 : 1];
#pragma unroll
            for (int n = 0; n < (W4 ? 2 : 1); n++) xv[n] = *reinterpret_cast<const v4i*>(codes + code_at(at + 2u * n, r));
            // the part of an operand that lies in block b of the slab, where its blocks are of different groups
            auto part = [&](const v4i& v, int b) {
                v4i o;
#pragma unroll
                for (int d = 0; d < 4; d++) o[d] = v[d] & (b == 0 ? first : ~first);
                return o;
            };
#pragma unroll
            for (int h = 0; h < NH; h++) {
                const v4i raw = w[l % AHEAD][h];
                auto dot = [&](const v4i& wv, const v4i& xo, int s) {
                    acc[s][h] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wv, xo, acc[s][h], 0, 0, 0);
                };
                if constexpr (W4) {
                    v4i lo, hi;  // (each nibble at the top of its byte)
#pragma unroll
                    for (int d = 0; d < 4; d++) {
                        lo[d] = (raw[d] << 4) & (int)0xf0f0f0f0u;
                        hi[d] = raw[d] & (int)0xf0f0f0f0u;
                    }
                    if constexpr (NSUB == 4) {
                        dot(lo, part(xv[0], 0), 0), dot(hi, part(xv[1], 0), 1), dot(lo, part(xv[0], 1), 2), dot(hi, part(xv[1], 1), 3);
                    } else if constexpr (NSUB == 2) {
                        dot(lo, part(xv[0], 0), 0), dot(hi, part(xv[1], 0), 0), dot(lo, part(xv[0], 1), 1), dot(hi, part(xv[1], 1), 1);
                    } else {
                        dot(lo, xv[0], 0), dot(hi, xv[1], 0);
                    }
                } else if constexpr (NSUB == 2) {
                    dot(raw, part(xv[0], 0), 0), dot(raw, part(xv[0], 1), 1);
                } else {
                    dot(raw, xv[0], 0);
                }
            }
            if (l + AHEAD < NL) issue(l + AHEAD);
        }
#pragma unroll
        for (int s = 0; s < NSUB; s++) {
            const uint32_t group = (uint32_t)(u * kWaves + wave) * NSUB + s;
            if (group >= a.groups) continue;  // (scalar)
#pragma unroll
            for (int h = 0; h < NH; h++) {
                const v4f sw = *reinterpret_cast<const v4f*>(scales + group * CH + h * 16 + chunk * 4u);
                v4f p;
#pragma unroll
                for (int e = 0; e < 4; e++) p[e] = __fmul_rn((float)(acc[s][h][e] >> (W4 ? 4 : 0)), __fmul_rn(rs, sw[e]));
                if (c < rows) *reinterpret_cast<v4f*>(products + (group * rows + c) * CH + h * 16 + chunk * 4u) = p;
            }
        }
    }
    __syncthreads();
    if (threadIdx.x >= rows * CH) return;
    float sum = 0.0f;
    const float* p = products + threadIdx.x;
    const uint32_t pitch = rows * CH;
    uint32_t g = 0;
    for (; g + 8u <= a.groups; g += 8u) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = p[(g + i) * pitch];
#pragma unroll
        for (int i = 0; i < 8; i++) sum = __fadd_rn(sum, v[i]);
    }
    for (; g < a.groups; g++) sum = __fadd_rn(sum, p[g * pitch]);
    if (on < a.n) ((float*)a.y)[(size_t)(threadIdx.x / CH) * a.n + on] = __fadd_rn(sum, bias);
}

template <int GK, bool W4, int CH, int NB, int RT>
bool launch(hipStream_t s, const LinearArgs& a) {
    const size_t lds = (size_t)RT * NB * 1024u + (size_t)a.groups * (a.rows + 1u) * CH * 4u;
    if (lds > 150u * 1024u) return false;
    auto kern = gemv_few_kernel<GK, W4, CH, NB, RT>;
    if (lds > 48u * 1024u) {
        static std::atomic<uint64_t> configured{0};
        if (!raise_lds_limit((const void*)kern, 152 * 1024, configured)) return false;
    }
    hipLaunchKernelGGL(kern, dim3(CH < 32 ? (a.n + 31u) / 32u * (32u / CH) : (a.n + CH - 1u) / CH), dim3(kThreads), lds, s, a);
    return hipGetLastError() == hipSuccess;
}

template <int GK, bool W4, int CH>
bool launch_length(hipStream_t s, const LinearArgs& a) {
    if (a.rows <= 4u) {
        if (a.k <= 1024u) return launch<GK, W4, CH, 1, 4>(s, a);
        if (a.k <= 2048u) return launch<GK, W4, CH, 2, 4>(s, a);
        if (a.k <= 3072u) return launch<GK, W4, CH, 3, 4>(s, a);
        return launch<GK, W4, CH, 4, 4>(s, a);
    }
    if constexpr (CH <= 32) {
        if (a.k <= 1024u) return launch<GK, W4, CH, 1, 8>(s, a);
        if constexpr (CH == 16) return launch<GK, W4, CH, 2, 8>(s, a);
    }
    return false;
}

template <int GK, bool W4>
bool launch_channels(hipStream_t s, const LinearArgs& a, uint32_t ch) {
    if (ch == 16u) return launch_length<GK, W4, 16>(s, a);
    if (ch == 32u) return launch_length<GK, W4, 32>(s, a);
    if constexpr (!W4 && GK > 1) return launch_length<GK, W4, 64>(s, a);
    return false;
}

template <bool W4>
bool launch_group(hipStream_t s, const LinearArgs& a, uint32_t ch) {
    switch (a.group_size) {
        case 32: return launch_channels<1, W4>(s, a, ch);
        case 64: return launch_channels<2, W4>(s, a, ch);
        case 128: return launch_channels<4, W4>(s, a, ch);
        case 256: return launch_channels<8, W4>(s, a, ch);
        default: return false;
    }
}

}  // namespace

// Which calls, and how many channels a workgroup.  Times of a row preparation and a GEMV over those of this kernel with
// 16 | 32 channels, means over drawn lengths, widths, groups and weight widths; replayed as a graph, and in parentheses
// behind a host that launches one by one:
//   rows  K up to   N up to 4096                 8192                       14336
//   3-4   1024      1.74 | 1.71 (1.41 | 1.41)    1.35 | 1.61 (1.40 | 1.40)  1.22 | 1.44 (1.34 | 1.39)
//   3-4   2048      1.61 | 1.49 (1.41 | 1.40)    1.36 | 1.61 (1.37 | 1.41)  1.09 | 1.19 (1.09 | 1.22)
//   3-4   4096      1.45 | 1.25 (1.48 | 1.30)    1.15 | 1.37 (1.14 | 1.37)  see below
//   3-4   8192      1.17 | 1.01, 0.88 at worst   0.70 | 0.98                0.82 | 0.89
//   5-8   1024      1.38 | 1.34 (1.42 | 1.42)    1.00 | 1.27 (1.32 | 1.40)  0.86 | 1.06
//   5-8   2048      1.21 | 1.11 (1.38 | 1.31)    0.90 | 1.15, 0.95 at worst 0.83 | 0.96
//   5-8   4096      0.99 | 0.89                  0.68 | 0.92                0.64 | 0.71
//   9-16  1024      1.02 | 0.97, 0.82 at worst   0.75 | 1.03                0.63 | 0.77
// More panels than compute units, weights from memory: two launches | 32 | 64 channels  3 x 4096 -> 14336 13.6 | 13.5 | 13.0 us,
// 3 x 3072 -> 14336 11.6 | 10.5 | 10.2, 4 x 1024 -> 14336 6.9 | 5.5 | 5.3; with four bits, whose reads no longer cover the
// preparation, 4 x 4096 -> 14336 10.1 | 11.2 | 10.9.
const char* launch_gemv_few(hipStream_t s, const LinearArgs& a, int cu_count, const char* force) {
    if (a.mode != Epilogue::DequantF32 || !a.x_f32 || a.ldx < a.k || a.rows <= kMaxPrepRows || a.rows > 8u || a.k < 2u ||
        a.k > (a.rows <= 4u ? 4096u : 2048u) || (a.weight_bits != 8u && a.weight_bits != 4u) || a.row_gain || a.row_swiglu ||
        a.add_to || a.acc_out || !a.y)
        return nullptr;
    if (force && !strstr(force, "few")) return nullptr;
    if (cu_count <= 0) cu_count = 256;
    const uint32_t panels = (a.n + 31u) / 32u, cu = (uint32_t)cu_count;
    uint32_t ch = panels * 2u <= cu ? 16u : panels > cu ? 64u : 32u;
    if (!force && a.rows > 4u && panels * (a.k <= 1024u ? 1u : 2u) > cu) return nullptr;
    if (!force && a.rows <= 4u && panels > cu && a.weight_bits == 4u && a.k > 2048u) return nullptr;
    if (force && strstr(force, "few16")) ch = 16u;
    else if (force && strstr(force, "few32")) ch = 32u;
    else if (force && strstr(force, "few64")) ch = 64u;
    // (the widths that are built: the others are of rows, lengths and weights that the lines above keep from them)
    if (ch == 64u && (a.weight_bits == 4u || a.group_size == 32u || a.rows > 4u)) ch = 32u;
    if (ch == 32u && a.rows > 4u && a.k > 1024u) ch = 16u;
    if (!(a.weight_bits == 4u ? launch_group<true>(s, a, ch) : launch_group<false>(s, a, ch))) return nullptr;
    static const char* const names[2][3] = {
        {"hip.packed-linear.a8-gemv-mfma.few16", "hip.packed-linear.a8-gemv-mfma.few32", "hip.packed-linear.a8-gemv-mfma.few64"},
        {"hip.packed-linear.w4a8-gemv-mfma.few16", "hip.packed-linear.w4a8-gemv-mfma.few32", "hip.packed-linear.w4a8-gemv-mfma.few64"}};
    return names[a.weight_bits == 4u ? 1 : 0][ch == 16u ? 0 : ch == 32u ? 1 : 2];
}

}  // namespace vxhip
