// PackedLinear under DYNAMIC_I8 for few tiles of output: the dequantizing linear on prepared rows with K split over the wavefronts
// of a workgroup (native/src/kernels/packed_linear_ops.inc:1471-1535, ordered sum :1498-1504).
//
// The tiles of gemm_k64.hip walk all of K with a barrier, fragments and a fold every 128 columns; where a launch has no
// more of them than the device has compute units, that walk is its time (33 to 256 rows of 14336 -> 1024 took 30 us, 0.25 us a
// k-block).  The streaming kernels of gemv_stream.hip hold the dots of all scale groups in LDS, so 32 rows of 4096 leave a
// compute unit one workgroup and 24 of 14336 none.  Here eight wavefronts take a slab of K each, one or two scale groups,
// which they multiply on v_mfma_i32_16x16x64_i8 straight from memory; they park the products f32(dot) * (s_a * s_w), and
// behind one barrier each output's thread adds the eight or sixteen of this pass in ascending group order, the sum the
// reference forms, bit for bit.  LDS holds two passes, whatever K is.
//
// Weights are read in the order they are packed in, activations in operand order in tiles of 32 rows (ActivationLayout): 256
// bytes in a row per quarter of a load.  Row-major rows, 64 bytes a row and load, were slower everywhere (64 x 4096 -> 4096 12.1
// against 10.5 us, 128 x 14336 -> 1024 23.5 against 17.7).  The next pass's slab is requested at the top of a pass.
// What bounds it is a compute unit's path to the L2: 458 KB of 14336-long operands take it 8.5 us.  More
// bytes in flight do not help (slabs of two passes ahead, each refilled behind its MFMA: 0 to 10 % slower), nor do sixteen
// wavefronts (0.9 to 1.6 times the time), nor larger tiles, whose few passes cover no latency (32 x 4096 -> 14336
// preparation included: 64 x 32 19.2 us, 32 x 32 20.3, the streaming kernel 19.3).
#include "common.h"
#include "device_math.h"
#include "gemm_tile.h"

#include <string.h>

namespace vxhip {
namespace {

extern __shared__ __attribute__((aligned(16))) char slab_lds[];

constexpr int WAVES = 8;  // (of 128 registers: two workgroups a compute unit, more of the smaller tiles)

// Bytes of LDS: the products of one pass, or of two where that leaves room for a second workgroup (one barrier a pass, not two).
template <int GROUP, int TN, int TM>
struct SlabLds {
    static constexpr int SLOTS = WAVES * (GROUP == 32 ? 2 : 1), OUT = TN * TM * 256;
    static constexpr int BUFFERS = SLOTS * OUT * 8 <= 64 * 1024 ? 2 : 1, BYTES = SLOTS * OUT * 4 * BUFFERS;
};

// A tile of 16 * TN channels and 16 * TM rows, TN and TM of 1 and 2.
template <int GROUP, bool W4, int TN, int TM>
__global__ __launch_bounds__(WAVES * 64, 4) void linear_slab_kernel(const GemmParams p) {
    constexpr int STEPS = GROUP <= 64 ? 1 : 2;    // MFMA steps of 64 columns in a slab
    constexpr int GPS = GROUP == 32 ? 2 : 1;      // scale groups that end in a slab (GROUP == 256: in every second one)
    constexpr int HALVES = GROUP == 256 ? 2 : 1;  // slabs of a unit, which is what a wavefront takes of a pass
    constexpr int BPT = W4 ? 1 : 2;               // 1 KiB blocks of a step
    constexpr int CH = TN * 16, ROWS = TM * 16, OUT = CH * ROWS, THREADS = WAVES * 64;
    constexpr int SLOTS = SlabLds<GROUP, TN, TM>::SLOTS, BUFFERS = SlabLds<GROUP, TN, TM>::BUFFERS;  // groups of a pass
    constexpr int PARTS = 2 / TN;                 // workgroups that share a panel
    constexpr int OPT = (OUT + THREADS - 1) / THREADS;
    const LinearArgs& a = p.a;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // (consecutive workgroups are on different XCDs: the tiles of a panel follow each other on one, whose L2 then has it)
    const uint32_t within = blockIdx.x >> 3, per = p.tiles_m * PARTS, tile = within % per;
    const uint32_t panel = within / per * 8u + (blockIdx.x & 7u), ch0 = panel * 32u + tile % PARTS * CH, m0 = tile / PARTS * ROWS;
    if (ch0 >= a.n) return;

    const uint32_t slabs = a.ksteps / (uint32_t)(BPT * STEPS), units = (a.groups + GPS - 1u) / GPS;
    const uint32_t passes = (units + WAVES - 1u) / WAVES;
    const uint32_t c = lane & 15, chunk = lane >> 4, last_chunk = (a.k - 1u) / 16u;
    const int8_t* const wp = a.w + (size_t)panel * a.ksteps * 1024u + (W4 ? 0u : (chunk >> 1) * 1024u) +
                             ((chunk & 1u) * 32u + (ch0 & 16u) + c) * 16u;
    const int8_t* xp[TM];
    float rs[TM];
#pragma unroll
    for (int j = 0; j < TM; j++) {
        const uint32_t row = min(m0 + j * 16u + c, a.rows - 1u);
        xp[j] = a.x + activation_offset(ActivationLayout{a.ldx, 1u}, row, 0u);
        rs[j] = a.row_scale[row];
    }
    const float* const sp = a.scales_t + ch0 + chunk * 4u;

    // two slabs: operands by step, and the scales of the groups that end there
    v4i w[2][STEPS][TN], x[2][STEPS][TM];
    v4f sw[2][GPS][TN];
    auto slab_of = [&](uint32_t pass, uint32_t half) { return min((pass * WAVES + (uint32_t)wave) * HALVES + half, slabs - 1u); };
    auto request = [&](auto b_tag, int s, uint32_t slab) {
        constexpr int b = decltype(b_tag)::value;
        const uint32_t step = slab * STEPS + s, at = min(step * 4u + chunk, last_chunk) * (16u * kOperandOrderRows);
#pragma unroll
        for (int j = 0; j < TM; j++) x[b][s][j] = *reinterpret_cast<const v4i*>(xp[j] + at);
#pragma unroll
        for (int i = 0; i < TN; i++) w[b][s][i] = *reinterpret_cast<const v4i*>(wp + (size_t)step * (BPT * 1024u) + i * 256);
    };
    auto request_scales = [&](auto b_tag, uint32_t unit) {
        constexpr int b = decltype(b_tag)::value;
#pragma unroll
        for (int e = 0; e < GPS; e++) {
            const uint32_t g = min(unit * GPS + e, a.groups - 1u);
#pragma unroll
            for (int i = 0; i < TN; i++) sw[b][e][i] = *reinterpret_cast<const v4f*>(sp + (size_t)g * a.n_pad + i * 16);
        }
    };
    auto request_slab = [&](auto b_tag, uint32_t slab) {
        static_for<STEPS>([&](auto s) { request(b_tag, decltype(s)::value, slab); });
    };
    request_slab(IC<0>{}, slab_of(0u, 0u));
    request_scales(IC<0>{}, (uint32_t)wave);

    float sum[OPT], bias[OPT];
#pragma unroll
    for (int it = 0; it < OPT; it++) {
        const uint32_t o = threadIdx.x + it * THREADS;
        sum[it] = 0.0f;
        bias[it] = a.bias_f32[ch0 + (o / (4u * ROWS) * 4u + o % 4u) % CH];
    }
    float* const products = reinterpret_cast<float*>(slab_lds);
    const v4i zero = {0, 0, 0, 0};
    const uint32_t nib_shift = lane < 32 ? 4u : 0u;
    v4i acc[GPS][TN][TM];
    // the dots of a slab, GPS == 2: group e has the lanes of its own half of the columns, zeros in the other
    auto multiply = [&](auto b_tag, int s, bool fresh) {
        constexpr int b = decltype(b_tag)::value;
        v4i wo[TN];
#pragma unroll
        for (int i = 0; i < TN; i++) {
            wo[i] = w[b][s][i];
            if constexpr (W4) {
#pragma unroll
                for (int d = 0; d < 4; d++) wo[i][d] = (w[b][s][i][d] << nib_shift) & (int)0xf0f0f0f0u;
            }
        }
#pragma unroll
        for (int e = 0; e < GPS; e++)
#pragma unroll
            for (int j = 0; j < TM; j++) {
                v4i xo = x[b][s][j];
                if constexpr (GPS == 2) {
                    const int keep = (lane >> 5) == e ? -1 : 0;
#pragma unroll
                    for (int d = 0; d < 4; d++) xo[d] &= keep;
                }
#pragma unroll
                for (int i = 0; i < TN; i++)
                    acc[e][i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wo[i], xo, fresh ? zero : acc[e][i][j], 0, 0, 0);
            }
    };
    // products[group of the pass][channel quad][row][4]: a wavefront's 16-byte stores, and the reads behind them, meet every bank once
    auto park = [&](auto b_tag, uint32_t buffer) {
        constexpr int b = decltype(b_tag)::value;
#pragma unroll
        for (int e = 0; e < GPS; e++) {
            float* const to = products + (buffer * SLOTS + (uint32_t)wave * GPS + e) * OUT;
#pragma unroll
            for (int i = 0; i < TN; i++)
#pragma unroll
                for (int j = 0; j < TM; j++) {
                    v4f v;
#pragma unroll
                    for (int d = 0; d < 4; d++)
                        v[d] = __fmul_rn((float)(acc[e][i][j][d] >> (W4 ? 4 : 0)), __fmul_rn(rs[j], sw[b][e][i][d]));
                    *reinterpret_cast<v4f*>(to + ((i * 4u + chunk) * ROWS + j * 16u + c) * 4u) = v;
                }
        }
    };
    // (not __syncthreads: the requests in flight stay in flight)
    auto meet = [&] {
        wait_lgkm0();
        wg_barrier();
    };
    auto gather = [&](uint32_t pass, uint32_t buffer) {
        const uint32_t live = min((uint32_t)SLOTS, a.groups - pass * SLOTS);
#pragma unroll
        for (int it = 0; it < OPT; it++) {
            const uint32_t o = threadIdx.x + it * THREADS;
            if (OUT % THREADS != 0 && o >= OUT) break;
            const float* from = products + buffer * SLOTS * OUT + o;
            if (live == (uint32_t)SLOTS) {
#pragma unroll
                for (int g0 = 0; g0 < SLOTS; g0 += 8) {
                    float v[8];
#pragma unroll
                    for (int g = 0; g < 8; g++) v[g] = from[(g0 + g) * OUT];
#pragma unroll
                    for (int g = 0; g < 8; g++) sum[it] = __fadd_rn(sum[it], v[g]);
                }
            } else {
                for (uint32_t g = 0; g < live; g++) sum[it] = __fadd_rn(sum[it], from[g * OUT]);
            }
        }
    };
    auto pass_of = [&](auto b_tag, uint32_t pass) {
        constexpr int b = decltype(b_tag)::value;
        const uint32_t unit = pass * WAVES + (uint32_t)wave, buffer = BUFFERS == 2 ? pass & 1u : 0u;
        if constexpr (HALVES == 1) {
            request_slab(IC<b ^ 1>{}, slab_of(pass + 1u, 0u));
            request_scales(IC<b ^ 1>{}, unit + WAVES);
            if (unit < units) {
                static_for<STEPS>([&](auto s_tag) { multiply(b_tag, decltype(s_tag)::value, decltype(s_tag)::value == 0); });
                park(b_tag, buffer);
            }
        } else {
            request_slab(IC<1>{}, slab_of(pass, 1u));
            request_scales(IC<b ^ 1>{}, unit + WAVES);
            if (unit < units) static_for<STEPS>([&](auto s_tag) { multiply(IC<0>{}, decltype(s_tag)::value, decltype(s_tag)::value == 0); });
            request_slab(IC<0>{}, slab_of(pass + 1u, 0u));
            if (unit < units) {
                if (unit * 2u + 1u < slabs) static_for<STEPS>([&](auto s_tag) { multiply(IC<1>{}, decltype(s_tag)::value, false); });
                park(b_tag, buffer);
            }
        }
        meet();
        gather(pass, buffer);
        if constexpr (BUFFERS == 1) meet();
    };
    for (uint32_t pass = 0; pass < passes; pass += 2u) {
        pass_of(IC<0>{}, pass);
        if (pass + 1u < passes) pass_of(IC<1>{}, pass + 1u);
    }
#pragma unroll
    for (int it = 0; it < OPT; it++) {
        const uint32_t o = threadIdx.x + it * THREADS;
        if (OUT % THREADS != 0 && o >= OUT) break;
        const uint32_t m = m0 + o / 4u % ROWS, n = ch0 + o / (4u * ROWS) * 4u + o % 4u;
        if (m < a.rows && n < a.n) ((float*)a.y)[(size_t)m * a.n + n] = __fadd_rn(sum[it], bias[it]);
    }
}

template <int GROUP, bool W4, int TN, int TM>
bool launch(hipStream_t s, const LinearArgs& a) {
    constexpr int LDS = SlabLds<GROUP, TN, TM>::BYTES;
    static std::atomic<uint64_t> configured{0};
    auto kern = linear_slab_kernel<GROUP, W4, TN, TM>;
    if (!raise_lds_limit((const void*)kern, LDS, configured)) return false;
    GemmParams p;
    p.a = a;
    p.tiles_n = (a.n + 31u) / 32u;
    p.tiles_m = (a.rows + TM * 16u - 1u) / (TM * 16u);
    hipLaunchKernelGGL(kern, dim3((p.tiles_n + 7u) / 8u * 8u * p.tiles_m * (2u / TN)), dim3(WAVES * 64), LDS, s, p);
    return hipGetLastError() == hipSuccess;
}
template <bool W4, int TN, int TM>
bool launch_group(hipStream_t s, const LinearArgs& a) {
    switch (a.group_size) {
        case 32: return launch<32, W4, TN, TM>(s, a);
        case 64: return launch<64, W4, TN, TM>(s, a);
        case 128: return launch<128, W4, TN, TM>(s, a);
        case 256: return launch<256, W4, TN, TM>(s, a);
        default: return false;
    }
}
template <int TN, int TM>
bool launch_bits(hipStream_t s, const LinearArgs& a) {
    return a.weight_bits == 4u ? launch_group<true, TN, TM>(s, a) : launch_group<false, TN, TM>(s, a);
}

}  // namespace

// Which calls (f32 rows, so that the preparation can write operand order), and which tile.  A tile's time is about constant
// while there are no more of them than compute units and grows by 0.6 of that for each further one a compute unit gets; a 16x32
// tile (channels x rows) costs 1.38 of a 16x16 one and a 32x32 tile 1.95 (groups of 32, whose products are four times as
// many: 1.25 and 2.2, which the rule never takes: by name only).  us, preparation included, with the kernels that took the call before | 16x16 | 16x32 | 32x32:
//   8 bits, groups of 128    32 x 2048 -> 1024   6.3 |  5.5 |  6.0 |  6.9    32 x 4096 -> 4096    9.4 |  9.4 |  8.7 | 10.2
//                            64 x 3000 -> 1531  10.6 |  8.2 |  7.6 |  8.8    64 x 4096 -> 4096   12.3 | 12.8 | 11.3 | 10.5
//                            32 x 14336 -> 4096 35.4 | 25.5 | 22.6 | 26.4    64 x 14336 -> 4096  32.2 | 37.7 | 31.4 | 27.0
//                            64 x 14336 -> 1024 30.1 | 13.1 | 15.9 | 20.9    200 x 14336 -> 1024 32.5 | 29.0 | 24.7 | 23.6
//   4 bits, groups of 32     32 x 14336 -> 4096 55.9 | 27.4 | 27.1 | 44.4    64 x 2500 -> 1500   13.2 |  8.6 |  8.9 | 12.3
//   4 bits, groups of 128    16 x 2000 -> 8000   8.1 |  7.2 |  8.3 |  8.3    32 x 4096 -> 14336  21.3 | 21.6 | 19.5 | 17.1
// Past a cost of 2 the tiles of gemm_k64.hip and the streaming kernel's straight-line instances up to K = 4096 are as fast or faster
// (128 x 4096 -> 4096 13.9 | 19.8 | 16.9 | 14.4, 32 x 4096 -> 14336 19.4 | 25.5 | 22.8 | 19.7); the general streaming kernel, the straight-line
// one in groups of 32 and 64 and the longer ones are slower up to 2.7 (16 x 4096 -> 14336 in groups of 64 28.9 | 20.2 | 21.0 | 18.8, 16 x 8192 ->
// 14336 36.3 | 32.8 | 34.2 | 30.0).  Groups of 256 have the cheapest fold there (150 x 2500 -> 1500 9.1 | 11.7 | 10.2 | 9.2, 239 x 2304 -> 736, a cost
// of 1.74, 8.4 | - | 9.6), short rows the fewest k-blocks (207 x 1440 -> 1056 7.5 us, 32x32 9.3; 118 x 1536 -> 1280, 1.59, 7.3 | - | 7.7).
// What stands behind a call is asked of its launcher (streaming_kernel).  Up to eight rows a straight-line instance that has them
// in LDS keeps its calls (6 x 3000 -> 1531 6.2 | 6.5, 4 x 8192 -> 14336 25.6 | 28.9); one that reads them from memory does not (8 x 4096 ->
// 14336 in groups of 64 23.6 | 18.6; 8 x 14336 -> 8192 36.5 | 26.7, with four bits 44.6 | 21.3).  With more rows whole panels up to K = 4096 stay
// (16 x 4096 -> 8192 10.5 | 13.1, 16 x 2048 -> 14336 in groups of 64 12.0 | 13.6); past it none do, and where the instance's LDS does not
// suffice there was no streaming kernel either (16 x 14336 -> 8192 41.1 | 30.2 | 31.3 | 26.6, 24 x 8192 -> 8192 25.6 | 25.3 | 21.8 | 18.5).
// The general kernel keeps weights of more than 26 MB once a compute unit gets a second tile (10 x 6000 -> 8192 14.7 | 17.5, 8 x 10000 ->
// 5055 17.4 | 19.0, in groups of 256 8 x 3500 -> 8192 10.7 | 11.6, 20 x 4384 -> 6433 12.6 | - | 16.2; before that 8 x 13000 -> 4096 19.6 | 17.2; fewer
// bytes, in groups of 64 6 x 3000 -> 1531, whose last group is half a group, 9.2 | 7.3, 8 x 2500 -> 8192 9.7 | 8.5, of four bits 8 x 6000 ->
// 8192 12.4 | 11.9), where each of its workgroups has a compute unit or its products leave room for a second one (10 x 2784 -> 13830
// 13.7 | 16.1, in groups of 256 8 x 4115 -> 10232 15.3 | 16.5; not 13 x 10240 -> 8704 32.7 | 30.1, in groups of 64 9 x 6176 -> 8376 26.9 | 21.6).
// 150 drawn calls, most of 3 to 32 rows of long K: all take 0.84 of the time they took before these kernels (geometric mean), the worst 1.03.
constexpr uint64_t kStreamedWeights = 26000000u;
SlabTile pick_slab_tile(const LinearArgs& a, int cu_count, const char* force) {
    if (a.weight_bits != 8u && a.weight_bits != 4u) return SlabTile::None;
    if (force) {
        return strstr(force, "slab16x16")   ? SlabTile::T16x16
               : strstr(force, "slab16x32") ? SlabTile::T16x32
               : strstr(force, "slab32x32") ? SlabTile::T32x32
                                            : SlabTile::None;
    }
    const bool four = a.weight_bits == 4u;
    if (a.rows <= kMaxPrepRows || a.rows > 256u) return SlabTile::None;
    const uint32_t panels = (a.n + 31u) / 32u, cu = cu_count > 0 ? (uint32_t)cu_count : 256u, columns = a.ksteps * (four ? 64u : 32u);
    if (a.k < (a.rows <= 4u ? 4097u : a.rows <= 8u ? 2049u : 1280u)) return SlabTile::None;
    const auto cost = [&](uint32_t tile_n, uint32_t tile_m, float one) {
        const float per = (float)((uint64_t)((a.n + tile_n - 1u) / tile_n) * ((a.rows + tile_m - 1u) / tile_m)) / (float)cu;
        return one * (per > 1.0f ? 1.0f + 0.6f * (per - 1.0f) : 1.0f);
    };
    const bool fine = a.group_size == 32u;
    const float c0 = cost(16u, 16u, 1.0f), c1 = cost(16u, 32u, fine ? 1.25f : 1.38f), c2 = cost(32u, 32u, fine ? 2.2f : 1.95f);
    const float least = c0 <= c1 && c0 <= c2 ? c0 : c1 <= c2 ? c1 : c2;
    const SlabTile cheapest = least == c0 ? SlabTile::T16x16 : least == c1 ? SlabTile::T16x32 : SlabTile::T32x32;
    // (nothing below declines these, and asking takes the host a tenth of a microsecond)
    if (a.rows > 8u && a.rows <= 32u && a.k >= 2048u && panels * 2u <= cu && least <= 1.6f) return cheapest;
    const Streams behind = a.rows <= 32u ? streaming_kernel(a, cu_count) : Streams::None;
    if (a.rows <= 8u && behind == Streams::RowsInLds) return SlabTile::None;
    if (behind == Streams::General && panels * 2u > cu && (panels <= cu || a.groups * (a.rows + 1u) * 128u <= 80u * 1024u) &&
        (uint64_t)a.n * a.k * a.weight_bits > kStreamedWeights * 8u)
        return SlabTile::None;
    const bool fits = a.rows > 8u && (behind == Streams::RowsInMemory || behind == Streams::RowsInLds) && columns <= 4096u;
    if (fits && a.k < 2048u) return SlabTile::None;
    // (whole panels: the products of all groups leave a compute unit room for two workgroups, or are at least few)
    if (fits && panels * 4u >= cu * 3u && (a.group_size >= 128u || a.groups * a.rows * 128u <= 80u * 1024u)) return SlabTile::None;
    const bool slow_stream = a.rows <= 8u ? behind == Streams::RowsInMemory : a.rows <= 32u && !(fits && a.group_size >= 128u);
    const float line = slow_stream                          ? 2.7f
                       : a.rows > 32u && a.k < 2048u        ? 1.5f
                       : a.group_size == 256u && a.k < 4096u ? 1.6f
                                                            : 2.0f;
    return least > line ? SlabTile::None : cheapest;
}

// a.x: operand order in tiles of 32 rows, ldx = the columns rounded up to 16.
const char* launch_linear_slabs(hipStream_t s, const LinearArgs& a, SlabTile tile) {
    if (a.mode != Epilogue::DequantF32 || !a.x || !a.x_operand_order || !a.y || !a.rows || a.acc_out || a.add_to || a.x_flip_mask ||
        a.ldx != (a.k + 15u) / 16u * 16u || (uintptr_t)a.x % 16u)
        return nullptr;
    bool ok = false;
    switch (tile) {
        case SlabTile::T16x16: ok = launch_bits<1, 1>(s, a); break;
        case SlabTile::T16x32: ok = launch_bits<1, 2>(s, a); break;
        case SlabTile::T32x32: ok = launch_bits<2, 2>(s, a); break;
        case SlabTile::None: break;
    }
    if (!ok) return nullptr;
    static const char* const names[2][3] = {
        {"hip.packed-linear.a8-mfma.slab16x16", "hip.packed-linear.a8-mfma.slab16x32", "hip.packed-linear.a8-mfma.slab32x32"},
        {"hip.packed-linear.w4a8-mfma.slab16x16", "hip.packed-linear.w4a8-mfma.slab16x32", "hip.packed-linear.w4a8-mfma.slab32x32"}};
    return names[a.weight_bits == 4u ? 1 : 0][(int)tile - 1];
}

}  // namespace vxhip
