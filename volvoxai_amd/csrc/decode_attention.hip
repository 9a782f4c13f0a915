// Attention of few tokens a row (decode) at head sizes 64 and 128: grouped-query attention over the cache in f32, scores scaled
// by 1/sqrt(d), causal visibility slot <= position, softmax, P.V; FUSED with the rotary embedding of its own query heads
// and the cache append in front (native/src/kernels/llm_math.h:256-274).
//
// A launch of many rows is bound by its reads: 32 rows of 8 KV heads at slot 145 are 37.9 MB, 7.6 us for a kernel that does
// nothing else.  Few rows are bound by the latency of a launch (1.7), of the position and behind it of the rows (1.5), and
// by what a compute unit takes in: its address unit needs 16 cycles a load of 1 KiB, a microsecond for the 148 KB of a
// head.  So one walk asks for everything that is in sight, values too, before the query is ready, holds it in registers (256
// slots: 128 of a lane's at head size 128), and up to there asks for nothing else; and scores, sums and outputs cross the
// workgroup twice.  At slot 145, against a kernel that kept its scores in LDS and asked for its values behind them (head size 128)
// and one walk of blocks of 128 slots with their requests clamped (64), 16 query and 8 KV heads of 128: 1 row
// 7.3 -> 4.1 us, 8 rows 8.0 -> 5.2, 16 rows 8.9 -> 6.9, 32 rows 12.3 -> 9.3; 8 and 4 of 64: 1 row 4.6 -> 3.3, 32 rows 5.7 -> 4.9.
// Steps of 28 layers: 1 row 0.625 -> 0.539 ms, 32 rows 1.218 -> 1.118.
#include "common.h"
#include "device_math.h"
#include "gemm_tile.h"
#include "wave_ops.h"

#include <math.h>

#include <type_traits>

namespace vxhip {
namespace {

constexpr int kWaitLoads = 0x0f70;  // s_waitcnt vmcnt(0), the other counters at their largest

// What a grid's x, y and z count: tokens are rows * t, those of a row in turn or, where rows come first, the rows' first ones, then their
// second ones; parts are the workgroups of a KV head, its query heads / REP * VS.
enum class GridOrder : uint32_t { TokensHeadsParts, HeadsPartsTokens, RowsPartsHeads };

// A workgroup has REP query heads of a KV head and 1 / VS of
// their channels (the scores want whole rows of keys, and each share makes them again).  The cache is cut into strips of eight slots, dealt to eight
// wavefronts in turn; two wavefronts are a part.  In a wavefront eight lanes share a slot, key and value row alike: 16-byte
// chunks c = lane % 8 + 8 * n, so a load of the wavefront covers a strip in whole 128-byte lines, and a slot's
// probability is in the lanes that weigh its value row.  A wavefront's probabilities refer to its running maximum; up to 256 slots,
// and behind the last one, it shares it with the other of its part, and the four parts are weighed against each other at the end.
template <int HD, int REP, int VS, bool FUSED, bool STREAM>
__global__ __launch_bounds__(512) void decode_attention_kernel(
    const float* __restrict__ q, float* __restrict__ k_cache, float* __restrict__ v_cache,
    const int64_t* __restrict__ positions, GridOrder order, uint32_t t, uint32_t kv_heads, uint32_t rep, uint32_t max_seq, float scale,
    float* __restrict__ out, const float* __restrict__ cos_table, const float* __restrict__ sin_table, uint32_t* __restrict__ fault) {
    constexpr int KC = HD / 32, OWN = HD / VS, VC = KC / VS, PASSES = 4, PARTS = 4, PART_WAVES = 2, WAVES = PARTS * PART_WAVES, THREADS = WAVES * 64;
    constexpr uint32_t STRIP = 8u, PASS = WAVES * STRIP, BLOCK = PASSES * PASS;
    constexpr int STAGED = (REP + (FUSED ? 2 : 0)) * HD;
    static_assert(STAGED <= THREADS && REP * HD <= THREADS, "an element a thread");
    __shared__ __attribute__((aligned(16))) float staged[STAGED];  // queries; FUSED: the appended key and value
    __shared__ __attribute__((aligned(16))) float partial[WAVES][REP][OWN];
    __shared__ __attribute__((aligned(8))) float maxima[2][REP][WAVES];
    __shared__ float sums[WAVES][REP];
    const uint32_t x = order == GridOrder::HeadsPartsTokens ? blockIdx.z : blockIdx.x;
    const uint32_t kvh = order == GridOrder::TokensHeadsParts   ? blockIdx.y
                         : order == GridOrder::HeadsPartsTokens ? blockIdx.x
                                                                : blockIdx.z;
    const uint32_t part = order == GridOrder::TokensHeadsParts ? blockIdx.z : blockIdx.y;
    // (no division stands in front of the first load of a decode step: three of them take a tenth of a microsecond)
    uint32_t row = x, i = 0u;
    if constexpr (!FUSED) {
        const uint32_t per = order == GridOrder::RowsPartsHeads ? gridDim.x / t : t;
        row = order == GridOrder::RowsPartsHeads ? x % per : x / per;
        i = order == GridOrder::RowsPartsHeads ? x / per : x % per;
    }
    const uint32_t token = FUSED ? row : row * t + i, q_heads = kv_heads * rep;
    const uint32_t head0 = kvh * rep + part / VS * REP, share = part % VS;
    const uint64_t named = (uint64_t)positions[i];
    if (named >= max_seq) {  // (the whole workgroup) outside the caches: touch nothing, say so
        if (threadIdx.x == 0) atomicOr(fault, (uint32_t)kFaultBadPosition);
        return;
    }
    const uint32_t position = (uint32_t)named;
    float* kbase = k_cache + ((size_t)row * kv_heads + kvh) * max_seq * HD;
    float* vbase = v_cache + ((size_t)row * kv_heads + kvh) * max_seq * HD;
    const uint32_t lane8 = threadIdx.x & 7u, group = (threadIdx.x >> 3) & 7u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // operands of the queries (and of the appended row) first: loads return in order
    float own = 0.0f, mate = 0.0f, c = 0.0f, sn = 0.0f;
    const uint32_t which = threadIdx.x / HD, dd = threadIdx.x % HD;
    if (STAGED == THREADS || threadIdx.x < STAGED) {
        if constexpr (FUSED) {
            const uint32_t head = which < REP ? head0 + which : which == REP ? q_heads + kvh : q_heads + kv_heads + kvh;
            const float* src = q + ((size_t)token * (q_heads + 2u * kv_heads) + head) * HD;
            own = src[dd];
            mate = src[dd ^ (HD / 2u)];
            c = cos_table[(size_t)position * HD + dd];
            sn = sin_table[(size_t)position * HD + dd];
        } else {
            own = q[((size_t)token * q_heads + head0 + which) * HD + dd];
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    // Rows past the last cached one are outside the descriptor: nothing is read for them and they are zeros.  (A request
    // under a branch would make the number of loads in flight unknown, and the first use wait for all of them.)
    const uint32_t bytes = (FUSED ? position : position + 1u) * (uint32_t)(HD * sizeof(float));
    const __amdgpu_buffer_rsrc_t k_rows = __builtin_amdgcn_make_buffer_rsrc(kbase, 0, (int)bytes, 0x00027000);
    const __amdgpu_buffer_rsrc_t v_rows = __builtin_amdgcn_make_buffer_rsrc(vbase, 0, (int)bytes, 0x00027000);
    const uint32_t lane_at = (wave * STRIP + group) * (HD * 4u) + lane8 * 16u;
    auto strip_of = [&](uint32_t block, int u) { return block * BLOCK + u * PASS + wave * STRIP; };  // (scalar) its first slot
    auto row_of = [&](__amdgpu_buffer_rsrc_t rows, uint32_t first, uint32_t block, int u, auto& to) {
#pragma unroll
        for (uint32_t n = 0; n < sizeof(to) / sizeof(to[0]); n++)
            to[n] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(
                rows, (int)(first + (block * BLOCK + u * PASS) * (HD * 4u) + n * 128u), 0, STREAM ? 2 : 0));
    };
    auto stage = [&] {
        if (STAGED == THREADS || threadIdx.x < STAGED) {
            float y = own;
            if (FUSED && which <= REP)  // the arithmetic of rope_append_kernel
                y = __fadd_rn(__fmul_rn(own, c), __fmul_rn(dd < HD / 2u ? -mate : mate, sn));
            staged[threadIdx.x] = y;
            if (FUSED && which >= REP && part == 0u) (which == REP ? kbase : vbase)[(size_t)position * HD + dd] = y;
        }
        __syncthreads();
    };
    // Probabilities carry a power of two of at most one over the number of slots (it leaves with the division at the
    // end): the sums of their products with values stay in the values' range.
    const float unit = __uint_as_float((127u - (position ? 32u - (uint32_t)__builtin_clz(position) : 0u)) << 23);
    v4f acc[REP][VC];
    float m[REP], sum[REP];
#pragma unroll
    for (int h = 0; h < REP; h++) {
        m[h] = -INFINITY;
        sum[h] = 0.0f;
#pragma unroll
        for (int n = 0; n < VC; n++) acc[h][n] = v4f{0.f, 0.f, 0.f, 0.f};
    }
    // `strip`: its first slot.  `ends`: it may hold the appended slot; `masked`: and slots out of sight
    auto score = [&](uint32_t strip, bool ends, bool masked, const v4f (&qv)[REP][KC], v4f (&kr)[KC], float (&dot)[REP], float (&top)[REP]) {
        const uint32_t slot = strip + group;
        if (FUSED && ends && slot == position) {
#pragma unroll
            for (int n = 0; n < KC; n++) kr[n] = *reinterpret_cast<const v4f*>(staged + REP * HD + 4u * lane8 + 32 * n);
        }
#pragma unroll
        for (int h = 0; h < REP; h++) {
            float d = 0.0f;
#pragma unroll
            for (int n = 0; n < KC; n++)
#pragma unroll
                for (int e = 0; e < 4; e++) d = __builtin_fmaf(qv[h][n][e], kr[n][e], d);
            d += lane_exchange<kDppXor1>(d);
            d += lane_exchange<kDppXor2>(d);
            d += lane_exchange<kDppHalfMirror>(d);
            d = __fmul_rn(d, scale);
            dot[h] = masked && slot > position ? -INFINITY : d;
            top[h] = fmaxf(top[h], dot[h]);
        }
    };
    auto weigh = [&](uint32_t strip, bool ends, v4f (&vr)[VC], const float (&p)[REP]) {
        if (FUSED && ends && strip + group == position) {
#pragma unroll
            for (int n = 0; n < VC; n++) vr[n] = *reinterpret_cast<const v4f*>(staged + (REP + 1) * HD + share * OWN + 4u * lane8 + 32 * n);
        }
#pragma unroll
        for (int h = 0; h < REP; h++)
#pragma unroll
            for (int n = 0; n < VC; n++)
#pragma unroll
                for (int e = 0; e < 4; e++) acc[h][n][e] = __builtin_fmaf(p[h], vr[n][e], acc[h][n][e]);
    };
    auto queries = [&](v4f (&qv)[REP][KC]) {
#pragma unroll
        for (int h = 0; h < REP; h++)
#pragma unroll
            for (int n = 0; n < KC; n++) qv[h][n] = *reinterpret_cast<const v4f*>(staged + h * HD + 4u * lane8 + 32 * n);
    };
    // the part's maximum over this block and those before: its wavefronts meet
    auto meet = [&](uint32_t block, const float (&top)[REP], float (&grown)[REP]) {
#pragma unroll
        for (int h = 0; h < REP; h++) {
            const float most = wave_max(top[h]);
            if ((threadIdx.x & 63u) == 0u) maxima[block & 1u][h][wave] = most;
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < REP; h++) {
            const float2 both = *reinterpret_cast<const float2*>(&maxima[block & 1u][h][wave / PART_WAVES * PART_WAVES]);
            grown[h] = fmaxf(fmaxf(both.x, both.y), m[h]);
        }
    };
    auto reference = [](float v) { return v == -INFINITY ? 0.0f : v; };  // (only scores of -inf so far: zeros)
    // from scores to probabilities, and what there is so far to the new maximum
    auto settle = [&](auto first_tag, const float (&grown)[REP], auto& dot, auto passes_tag) {
#pragma unroll
        for (int h = 0; h < REP; h++) {
            if constexpr (!decltype(first_tag)::value) {
                const float keep = expf(m[h] - reference(grown[h]));
                sum[h] *= keep;
#pragma unroll
                for (int n = 0; n < VC; n++) acc[h][n] *= keep;
            }
            m[h] = grown[h];
#pragma unroll
            for (int u = 0; u < decltype(passes_tag)::value; u++) {
                dot[u][h] = expf(dot[u][h] - reference(m[h])) * unit;
                sum[h] += dot[u][h];
            }
        }
    };
    const uint32_t blocks = position / BLOCK + 1u;
    if (blocks == 1u) {
        // Up to 256 slots: a copy of the code for each number of strips a wavefront has in sight, so that what is not in sight is
        // not asked for: a load outside the descriptor takes the address unit as long as one inside, 1.7 us for 256 slots.
        auto whole = [&](auto passes_tag) {
            constexpr int P = decltype(passes_tag)::value, N = P > 0 ? P : 1;
            v4f kb[N][KC], vb[N][VC];
#pragma unroll
            for (int u = 0; u < P; u++) row_of(k_rows, lane_at, 0u, u, kb[u]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < P; u++) row_of(v_rows, lane_at + share * (OWN * 4u), 0u, u, vb[u]);
            __builtin_amdgcn_sched_barrier(0);
            stage();
            float dot[N][REP], top[REP], grown[REP];
#pragma unroll
            for (int h = 0; h < REP; h++) top[h] = -INFINITY;
            if constexpr (P > 0) {
                v4f qv[REP][KC];
                queries(qv);
#pragma unroll
                for (int u = 0; u < P; u++) score(strip_of(0u, u), u == P - 1, u == P - 1, qv, kb[u], dot[u], top);
            }
            meet(0u, top, grown);
            settle(std::true_type{}, grown, dot, passes_tag);
#pragma unroll
            for (int u = 0; u < P; u++) weigh(strip_of(0u, u), u == P - 1, vb[u], dot[u]);
        };
        const uint32_t passes = position >= wave * STRIP ? (position - wave * STRIP) / PASS + 1u : 0u;
        switch (passes) {
            case 0: whole(std::integral_constant<int, 0>{}); break;
            case 1: whole(std::integral_constant<int, 1>{}); break;
            case 2: whole(std::integral_constant<int, 2>{}); break;
            case 3: whole(std::integral_constant<int, 3>{}); break;
            default: whole(std::integral_constant<int, 4>{}); break;
        }
    } else {
        // More: a block's rows are requested as soon as the registers of the one before are free, and the wavefronts meet behind
        // the last one only.  The first block is the one that is not whole: its first `missing` rounds of 64 slots would lie in front
        // of slot 0, so that only strips of the last round are asked for out of sight.  (With the last block not whole, all of it
        // asked for, and a meeting a block: 16 heads on 8 of 128 at slot 256 1 row 6.5 -> 5.8 us, 16 rows 13.4 -> 10.6, 32 rows 17.8 -> 15.1;
        // 32 heads on 4, 8 rows, slot 256 9.6 -> 8.6, 1000 21.8 -> 20.5, 2000 39.3 -> 35.6.  Copies of the last two blocks for
        // each number of strips, as above, spill.)
        const uint32_t missing = blocks * PASSES - (position / PASS + 1u), back = missing * PASS;
        const uint32_t lane_back = lane_at - back * (HD * 4u);
        v4f kb[PASSES][KC], vb[PASSES][VC];
        auto request_first = [&](auto whole_tag) {
            constexpr bool WHOLE = decltype(whole_tag)::value;
            auto requested = [&](int u) { return WHOLE || u + 1 == PASSES || (uint32_t)u >= missing; };  // (scalar)
#pragma unroll
            for (int u = 0; u < PASSES; u++) {
                if (requested(u)) row_of(k_rows, lane_back, 0u, u, kb[u]);
                else for (auto& chunk : kb[u]) chunk = v4f{0.f, 0.f, 0.f, 0.f};
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < PASSES; u++) {
                if (requested(u)) row_of(v_rows, lane_back + share * (OWN * 4u), 0u, u, vb[u]);
                else for (auto& chunk : vb[u]) chunk = v4f{0.f, 0.f, 0.f, 0.f};
            }
            __builtin_amdgcn_sched_barrier(0);
            stage();
            // Requests under a condition make the number in flight unknown, and the first use would wait for all of them, in either
            // case: here is that wait, so that the other has none.
            if constexpr (!WHOLE) __builtin_amdgcn_s_waitcnt(kWaitLoads);
        };
        if (missing == 0u) request_first(std::true_type{});
        else request_first(std::false_type{});
        v4f qv[REP][KC];
        queries(qv);
        uint32_t block = 0u;
        auto one = [&](auto ends_tag) {
            constexpr bool ENDS = decltype(ends_tag)::value;
            float dot[PASSES][REP], top[REP], grown[REP];
#pragma unroll
            for (int h = 0; h < REP; h++) top[h] = -INFINITY;
#pragma unroll
            for (int u = 0; u < PASSES; u++) {
                score(strip_of(block, u) - back, ENDS && u + 1 == PASSES, true, qv, kb[u], dot[u], top);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (!ENDS) row_of(k_rows, lane_back, block + 1u, u, kb[u]);
            }
#pragma unroll
            for (int h = 0; h < REP; h++) grown[h] = fmaxf(m[h], wave_max(top[h]));
            settle(std::false_type{}, grown, dot, std::integral_constant<int, PASSES>{});
#pragma unroll
            for (int u = 0; u < PASSES; u++) {
                weigh(strip_of(block, u) - back, ENDS && u + 1 == PASSES, vb[u], dot[u]);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (!ENDS) row_of(v_rows, lane_back + share * (OWN * 4u), block + 1u, u, vb[u]);
            }
        };
#pragma clang loop unroll(disable)
        for (; block + 1u < blocks; block++) one(std::false_type{});
        one(std::true_type{});
        float common[REP];
        meet(block, m, common);
#pragma unroll
        for (int h = 0; h < REP; h++) {
            const float keep = expf(m[h] - reference(common[h]));
            sum[h] *= keep;
#pragma unroll
            for (int n = 0; n < VC; n++) acc[h][n] *= keep;
            m[h] = common[h];
        }
    }
    // The groups of a wavefront meet: lanes 32, then 16, then 8 apart.  A step that can exchanges one half of the channels
    // for the other, so a lane is left with one chunk.
    constexpr int kDppRor8 = 0x128;  // lane ^ 8 within a row of 16
    auto halves = [](float a, float b) {  // lower half: a summed over both, upper half: b
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        return __uint_as_float(r[0]) + __uint_as_float(r[1]);
    };
    auto rows16 = [](float a, float b) {  // even rows of sixteen: a summed over a pair of rows, odd rows: b
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        return __uint_as_float(r[0]) + __uint_as_float(r[1]);
    };
#pragma unroll
    for (int h = 0; h < REP; h++) {
        float total = halves(sum[h], sum[h]);
        total = rows16(total, total);
        total += lane_exchange<kDppRor8>(total);
        v4f mine;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float lo = halves(acc[h][0][e], acc[h][VC / 2][e]), hi = VC == 4 ? halves(acc[h][VC / 4][e], acc[h][VC - 1][e]) : lo;
            mine[e] = rows16(lo, hi);
            mine[e] += lane_exchange<kDppRor8>(mine[e]);
        }
        // (four chunks: the upper half of the lanes has 2 and 3, odd rows 1 and 3; two: the upper half has 1)
        const uint32_t upper = (threadIdx.x >> 5) & 1u, odd = (threadIdx.x >> 4) & 1u, chunk = VC == 4 ? upper * 2u + odd : VC == 2 ? upper : 0u;
        const bool leads = (threadIdx.x & 8u) == 0u && (VC == 4 || odd == 0u) && (VC >= 2 || upper == 0u);
        if (leads) *reinterpret_cast<v4f*>(&partial[wave][h][4u * lane8 + 32u * chunk]) = mine;
        if ((threadIdx.x & 63u) == 0u) {
            sums[wave][h] = total;
            maxima[blocks & 1u][h][wave] = m[h];
        }
    }
    __syncthreads();
    if (threadIdx.x < REP * OWN) {
        const uint32_t h = threadIdx.x / OWN, at = threadIdx.x % OWN;
        float top[PARTS], most = -INFINITY, total = 0.0f, y = 0.0f;
#pragma unroll
        for (int p = 0; p < PARTS; p++) {
            top[p] = maxima[blocks & 1u][h][PART_WAVES * p];
            most = fmaxf(most, top[p]);
        }
#pragma unroll
        for (int p = 0; p < PARTS; p++) {
            const float weight = expf(top[p] - reference(most));
            total = __builtin_fmaf(sums[PART_WAVES * p][h] + sums[PART_WAVES * p + 1][h], weight, total);
            y = __builtin_fmaf(partial[PART_WAVES * p][h][at] + partial[PART_WAVES * p + 1][h][at], weight, y);
        }
        out[((size_t)token * q_heads + head0 + h) * HD + share * OWN + at] = __fdiv_rn(y, total);
    }
}

}  // namespace

// How a launch is split.  Few heads: a workgroup a head, and two or four workgroups a head as long as no compute unit has
// two of them; each scores all slots and weighs its share of the channels.  More: two heads that share their rows a
// workgroup, which at head size 64, where the rows are half as long, pays from one workgroup a head and compute unit on
// only.  us a launch at slot 145, a head a workgroup whole | in two | in four | two heads a workgroup (16 query and 8 KV
// heads of 128, then 8 and 4 of 64):
//   128   1 row  4.6 | 4.2 | 4.1 | 5.5    8 rows  5.8 | 5.2 | 6.2 | 6.4    16 rows  6.9 | 8.6 | 10.3 | 6.9    32 rows  14.0 | 16.5 | 19.4 | 9.5
//         (steps of 28 layers, ms: 12 rows 1.027 | 1.077 | 1.098 | 1.017, 16 rows 1.046 | 1.094 | 1.147 | 1.019)
//    64   1 row  3.9 | 3.3 | - | 4.2      8 rows  4.2 | 4.0 | - | 4.8      16 rows  4.5 | 4.2 | - | 5.0         32 rows  4.8 | 5.6 | - | 5.3
// Four heads a workgroup read their rows half as often.  At head size 64, in groups of four heads, from two heads a compute
// unit on (two heads a workgroup | four: 32 heads on 4, 16 rows, slot 145 4.6 | 5.8 us, 20 rows 6.7 | 6.0, slot 2000 38.7 | 30.5; 32 on 8,
// 24 rows, slot 145 8.6 | 7.3, 2000 48.5 | 39.3).  At head size 128 their registers do not fit this kernel: false, and the caller launches
// the one that keeps its scores, in groups of eight heads: more than four heads a compute unit (64 rows of 32 heads on 4 at slot
// 255 47 | 23.3), and from two and a half on where the cache may hold more than 256 slots (32 on 4, 24 rows, slot 145 10.6 | 13.2, 256
// 17.2 | 15.3, 2000 79.6 | 65.3; 32 rows, slot 145 11.4 | 13.6, 256 19.0 | 15.8, 2000 89 | 68; 17 rows, slot 256 16.9 | 15.7, 300 17.2 | 18.2,
// 2000 63.6 | 64.1).
// Workgroups that read the same rows -- the parts of a KV head, the tokens of a row -- share them where they run on one XCD (of
// consecutive workgroups every eighth) and soon after each other.  With the parts last, a device's worth of workgroups and more
// apart, each read its rows from HBM again: 24 heads on 8 of 128, 32 rows, slot 255 34.3 us against 20.7, 2000 259 against 125 (the kernel
// that this one replaced 22.3 and 132); 32 on 8, 32 rows, slot 2000 179 against 98.  Below one and a half workgroups a compute
// unit they run at once (32 on 8, 17 rows 10.8 against 12.0), and eight heads a KV head gain only past the lengths that the
// four-heads kernels have (32 on 4, 24 rows 14.3 against 15.6).  Several tokens a row: 16 heads on 8 of 128, 32 rows of 4 at
// slot 255 47 us against 30.
// Non-temporal loads where a row's reader is alone: 32 rows 9.3 against 10.4 us; where two workgroups read it, plain ones
// (17 rows of 16 heads on 2: 6.8 against 7.2), and where several tokens do (8 heads on 8 of 128, 32 rows of 7 at slot 600 86.5
// against 79.8; 4 on 4 of 64 27.1 against 21.0; two tokens gain and lose up to a tenth).
bool launch_decode_attention(hipStream_t s, int cu_count, uint32_t tokens, const float* q, float* k_cache, float* v_cache,
                             const int64_t* positions, uint32_t t, uint32_t q_heads, uint32_t kv_heads, uint32_t head_dim,
                             uint32_t max_seq, float scale, float* out, const float* cos_table, const float* sin_table,
                             uint32_t* fault) {
    const uint32_t rep = q_heads / kv_heads;
    const uint64_t cu = cu_count > 0 ? (uint64_t)cu_count : 256u, heads = (uint64_t)tokens * q_heads;
    const bool four = rep % 4u == 0u && (head_dim == 64u ? heads > 2u * cu
                                                         : rep >= 8u && (heads > 4u * cu || (max_seq > 256u && heads * 2u >= cu * 5u)));
    GridOrder order = GridOrder::TokensHeadsParts;
    auto grid_of = [&](uint32_t parts) {
        const bool shared = t > 1u || (parts > 1u && !(rep >= 8u && rep % 4u == 0u) && (uint64_t)tokens * kv_heads * parts * 2u >= cu * 3u);
        if (shared && kv_heads % 8u == 0u && tokens <= 0xffffu) {
            order = GridOrder::HeadsPartsTokens;
            return dim3(kv_heads, parts, tokens);
        }
        if (shared && tokens / t % 8u == 0u) {
            order = GridOrder::RowsPartsHeads;
            return dim3(tokens, parts, kv_heads);
        }
        return dim3(tokens, kv_heads, parts);
    };
#define VXHIP_DECODE_AS(HD, REP, VS, FUSED, STREAM)                                                                            \
    do {                                                                                                                       \
        const dim3 grid = grid_of(rep / REP * VS);                                                                             \
        hipLaunchKernelGGL((decode_attention_kernel<HD, REP, VS, FUSED, STREAM>), grid, dim3(512), 0, s, q, k_cache, v_cache,  \
                           positions, order, t, kv_heads, rep, max_seq, scale, out, cos_table, sin_table, fault);              \
    } while (0)
#define VXHIP_DECODE(HD, REP, VS)                                                            \
    do {                                                                                     \
        constexpr bool kAlone = VS == 1 && REP < 4; /* (may be) */                           \
        if (kAlone && rep == REP && t == 1u) {                                               \
            if (cos_table) VXHIP_DECODE_AS(HD, REP, VS, true, kAlone);                       \
            else VXHIP_DECODE_AS(HD, REP, VS, false, kAlone);                                \
        } else {                                                                             \
            if (cos_table) VXHIP_DECODE_AS(HD, REP, VS, true, false);                        \
            else VXHIP_DECODE_AS(HD, REP, VS, false, false);                                 \
        }                                                                                    \
    } while (0)
    if (head_dim == 128u) {
        if (four) return false;
        if (heads * 4u <= cu) VXHIP_DECODE(128, 1, 4);
        else if (heads * 2u <= cu) VXHIP_DECODE(128, 1, 2);
        else if (rep % 2u == 0u) VXHIP_DECODE(128, 2, 1);
        else VXHIP_DECODE(128, 1, 1);
        return true;
    }
    if (head_dim == 64u) {
        if (four) VXHIP_DECODE(64, 4, 1);
        else if (heads * 2u <= cu) VXHIP_DECODE(64, 1, 2);
        else if (heads > cu && rep % 2u == 0u) VXHIP_DECODE(64, 2, 1);
        else VXHIP_DECODE(64, 1, 1);
        return true;
    }
    return false;
#undef VXHIP_DECODE
#undef VXHIP_DECODE_AS
}

}  // namespace vxhip
