// QLinear of few tiles of output: K split over the wavefronts of a workgroup (native/src/kernels/portable_inference_kernels.inc:1006-1028;
// the reference's large-row route is native/src/kernels/packed_quant_gemm.c:2411-2600).
//
// A tile of gemm_mfma.hip walks all of K, 0.22 us every 128 columns, which is its launch's time where the device has a compute unit for
// every tile: 33 to 1024 rows of 4096 -> 512 all took 10 us.  Here four wavefronts divide the k-blocks of a 32 x 32 tile between them, each with
// two LDS stages of its own and no barrier until their sums meet; integer sums have no order, so the bytes are the same.  64 KiB of LDS
// let two workgroups share a compute unit.  Bound by the loads' latency and, at two tiles a compute unit, by its path to
// the L2 (512 KB of operands in 6 us).  Eight wavefronts a tile gain nothing (33 x 4096 -> 512 5.4 us both) and leave no room for a second
// tile; larger tiles, of four wavefronts a group that share their stages behind barriers, are slower in every launch of few tiles
// (64 x 4096 -> 4096: 64 x 64 11.6 us, 64 x 32 9.1, 32 x 32 7.0).
#include "common.h"
#include "device_math.h"
#include "epilogue.h"
#include "gemm_tile.h"

#include <string.h>

namespace vxhip {
namespace {

extern __shared__ __attribute__((aligned(1024))) char split_lds[];

constexpr int WAVES = 4;

// Four wavefronts of a workgroup share a tile of 32 channels and 32 rows; wavefront g takes the k-blocks g, g + 4, g + 8 ...
template <int MODE>
__global__ __launch_bounds__(WAVES * 64) void requant_split_kernel(const GemmParams p) {
    constexpr int TILE = 32, LOADS = 8, STAGE = LOADS * 1024, QUADS = TILE * TILE / 4;
    static_assert(QUADS == WAVES * 64 && QUADS * 16 <= 2 * STAGE, "a thread finishes four channels; the sums fit the stages");
    const LinearArgs& a = p.a;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const TileOrigin t = tile_of_workgroup<TILE, TILE>(p);
    if (!t.valid) return;
    const uint32_t m0 = t.m0, n0 = t.n0;
    const uint32_t nkb = ((a.k + 31u) / 32u + 3u) / 4u, rounds = (nkb + WAVES - 1u) / WAVES;
    const uint32_t last_chunk = (a.k - 1u) / 16u, my_chunk = (lane & 7) ^ ((lane >> 3) & 7);
    const int8_t* const wp = a.w + (size_t)(n0 / 32u) * a.ksteps * 1024u + lane * 16u;
    uint32_t xrow[4];
#pragma unroll
    for (int i = 0; i < 4; i++) xrow[i] = min(m0 + i * 8u + (lane >> 3), a.rows - 1u) * a.ldx;
    // The stages are the wavefront's own: it waits for its loads and for nobody.  (The images are those of gemm_k64.hip: the weights'
    // blocks as they are packed, rows of 128 bytes with their 16-byte chunks swizzled.)
    char* const mine = split_lds + wave * (2 * STAGE);
    auto issue = [&](uint32_t round, int stage) {
        const uint32_t kb = min(round * WAVES + (uint32_t)wave, nkb - 1u);
        char* base = mine + stage * STAGE;
        static_for<4>([&](auto b) { load_to_lds16(wp + (size_t)(kb * 4u + decltype(b)::value) * 1024u, base + decltype(b)::value * 1024); });
        const uint32_t chunk16 = min(kb * 8u + my_chunk, last_chunk) * 16u;
        static_for<4>([&](auto b) { load_to_lds16(a.x + (xrow[decltype(b)::value] + chunk16), base + (4 + decltype(b)::value) * 1024); });
    };
    issue(0u, 0);
    issue(1u, 1);

    v4i acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = v4i{0, 0, 0, 0};
    const uint32_t a_frag = (lane >> 5) * 1024u + ((lane & 15) + 32 * ((lane >> 4) & 1)) * 16u;
    const uint32_t x_frag = 4096u + (lane & 15) * 128u;
    auto round_of = [&](uint32_t round, auto stage_tag) {
        constexpr int S = decltype(stage_tag)::value;
        const char* stage = mine + S * STAGE;
        wait_vmcnt<LOADS>();
        v4i af[2][2], bf[2][2];
#pragma unroll
        for (int s = 0; s < 2; s++) {
#pragma unroll
            for (int i = 0; i < 2; i++) af[s][i] = *reinterpret_cast<const v4i*>(stage + a_frag + s * 2048 + i * 256);
#pragma unroll
            for (int j = 0; j < 2; j++)
                bf[s][j] = *reinterpret_cast<const v4i*>(stage + x_frag + j * 2048 + (((4u * s + (lane >> 4)) ^ (lane & 7u)) << 4)) ^ (int)a.x_flip_mask;
        }
        wait_lgkm0();  // the stage is in registers
        issue(round + 2u, S);
        if (round * WAVES + (uint32_t)wave < nkb) {  // (scalar: an MFMA is not predicated)
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[s][i], bf[s][j], acc[i][j], 0, 0, 0);
        }
    };
    for (uint32_t round = 0; round < rounds; round += 2u) {
        round_of(round, IC<0>{});
        if (round + 1u < rounds) round_of(round + 1u, IC<1>{});
    }
    // this thread finishes channels n .. n + 3 of row m
    const uint32_t m = m0 + threadIdx.x % TILE, n = n0 + threadIdx.x / TILE * 4u;
    ChannelConsts cc[4];
#pragma unroll
    for (int e = 0; e < 4; e++) cc[e] = channel_consts<MODE>(a, n + e);
    const uint32_t row = min(m, a.rows - 1u);
    const float row_scale = MODE == (int)Epilogue::RequantRow ? a.row_scale[row] : 0.0f;
    const int32_t rsum = a.zw ? a.rowsum[row] : 0;
    wait_vmcnt<0>();  // nothing of this workgroup may still be writing LDS
    wg_barrier();
    v4i* const parts = reinterpret_cast<v4i*>(split_lds);  // [wavefront][channel quad][row]
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
            parts[wave * QUADS + (i * 4 + (lane >> 4)) * TILE + j * 16 + (lane & 15)] = acc[i][j];
    wait_lgkm0();
    wg_barrier();
    int32_t dot[4] = {0, 0, 0, 0};
#pragma unroll
    for (int g = 0; g < WAVES; g++) {
        const v4i v = parts[g * QUADS + threadIdx.x];
#pragma unroll
        for (int e = 0; e < 4; e++) dot[e] += v[e];
    }
    const float none[4] = {0.f, 0.f, 0.f, 0.f};
    store_quad<MODE>(a, m, n, dot, none, row_scale, rsum, cc);
}

template <int MODE>
bool launch(hipStream_t s, const LinearArgs& a) {
    constexpr int LDS = WAVES * 2 * 8192;
    static std::atomic<uint64_t> configured{0};
    auto kern = requant_split_kernel<MODE>;
    if (!raise_lds_limit((const void*)kern, LDS, configured)) return false;
    GemmParams p;
    p.a = a;
    p.tiles_n = (a.n + 31u) / 32u;
    p.tiles_m = (a.rows + 31u) / 32u;
    hipLaunchKernelGGL(kern, dim3((p.tiles_n * p.tiles_m + 7u) / 8u * 8u), dim3(WAVES * 64), LDS, s, p);
    return hipGetLastError() == hipSuccess;
}

}  // namespace

// Which calls: those of no more tiles than compute units, or of up to one and a half and two times as many where K is long enough for a
// walk over all of it to be what the others cost.  us, with the tiles of 64 x 64 that took the calls before (of 128 x 64 the last):
//   rows  K -> N       tiles a compute unit            rows  K -> N       tiles a compute unit
//   256    512 -> 1024  1     3.97 -> 3.87             256   1024 -> 1024  1     4.92 -> 4.35
//   128   2048 -> 2048  1     6.72 -> 4.66              33   4096 ->  512  0.1  10.00 -> 5.42
//   256   4096 -> 1024  1    10.40 -> 6.66              64   4096 -> 4096  1    11.06 -> 6.98
//   256   1536 -> 1536  1.5   5.94 -> 5.72             256   3001 -> 1531  1.5  13.87 -> 12.05 (with its staging launch)
//   128   4096 -> 4096  2    11.29 -> 9.42 taken       256   2048 -> 2048  2     6.88 -> 7.19 not taken
//   512   4096 -> 2048  4    11.46 -> 16.68 not taken
// Two k-blocks are walked as fast by the tiles of 64 x 64, up to half a tile a compute unit by 0.3 us (70 x 256 -> 512 3.44 -> 3.72, 67 x 256 ->
// 256 with per-row scales 4.03 -> 4.33; not 52 x 256 -> 3840 6.5 -> 5.8, nor unsigned bytes, which those tiles want flipped first: 124 x 256 ->
// 512 5.8 -> 3.7).
// From 17 rows on also in place of the streaming kernel: 32 x 2048 -> 2048 6.2 -> 4.6, 32 x 4096 -> 512 7.7 -> 5.4 (16 rows 6.2); 32 x
// 1024 -> 1024 3.9 -> 4.2 and 24 x 1536 -> 1536 4.5 are left there.  (17 to 23 rows of K below 2900 and few channels take it 4.2 or 5.3, by where
// their operands lie, and these tiles 4.6: 18 x 2064 -> 1120, 23 x 2656 -> 448.)  105 calls of 17 to 500 rows, bytes, per-row scales and f32 rows: 0.79 of their
// time before (geometric mean of graph replays).
const char* launch_requant_split(hipStream_t s, const LinearArgs& a, int cu_count, const char* force) {
    if (a.mode == Epilogue::DequantF32 || a.weight_bits != 8u || a.x_f32 || a.x_operand_order || a.ldx < 16u || a.ldx % 16u ||
        (uintptr_t)a.x % 16u || (uint64_t)a.rows * a.ldx > 0xffffffffull)
        return nullptr;
    if (force) {
        if (!strstr(force, "t32x32split")) return nullptr;
    } else {
        const uint64_t tiles = (uint64_t)((a.n + 31u) / 32u) * ((a.rows + 31u) / 32u), cu = cu_count > 0 ? (uint64_t)cu_count : 256u;
        if (a.k <= 256u && tiles * 2u <= cu && !a.x_flip_mask) return nullptr;
        if (tiles > (a.k >= 2560u ? cu * 2u : a.k >= 1536u ? cu * 3u / 2u : cu)) return nullptr;
        if (a.rows <= kMaxGemvRows && (a.rows <= 16u || a.k < 2048u || tiles > cu)) return nullptr;
    }
    return (a.mode == Epilogue::RequantRow ? launch<(int)Epilogue::RequantRow>(s, a) : launch<(int)Epilogue::RequantTensor>(s, a))
               ? "t32x32split"
               : nullptr;
}

}  // namespace vxhip
