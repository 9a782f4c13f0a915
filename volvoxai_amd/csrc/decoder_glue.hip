// The steps either side of the W8A8 linears in a decoder layer, fused so that a decode step
// is a dozen launches per layer instead of several dozen elementwise ones:
//
//   rmsnorm_prepare, swiglu_prepare   row_prepare.hip
//   rope_append       non-interleaved rotary embedding of q and k
//                     (native/src/kernels/llm_math.h:256-274) and the KV-cache append
//   gqa_attention     grouped-query attention of the new tokens over the cache: f32 scores
//                     scaled by 1/sqrt(d), causal visibility slot <= position, softmax, P.V
//                     (of few tokens at head sizes 64 and 128: decode_attention.hip)
//
// All are row-sized, latency-bound kernels; none of them is on the int8 roofline.
#include "common.h"
#include "device_math.h"
#include "gemm_tile.h"
#include "row_math.h"
#include "wave_ops.h"

#include <math.h>

namespace vxhip {
namespace {

extern __shared__ __attribute__((aligned(16))) char glue_lds[];

// grid rows * t, one workgroup per token walking the elements of all its heads (a workgroup per head
// is a launch of a hundred thousand workgroups that move 512 bytes each).  Token (row, i) sits at cache
// slot positions[i]; cos/sin are [max_seq][head_dim] tables indexed by that slot.
__global__ __launch_bounds__(256) void rope_append_kernel(const float* __restrict__ qkv, const float* __restrict__ cos_table,
                                                          const float* __restrict__ sin_table,
                                                          const int64_t* __restrict__ positions, uint32_t t, uint32_t q_heads,
                                                          uint32_t kv_heads, uint32_t head_dim, uint32_t max_seq,
                                                          float* __restrict__ q_out, float* __restrict__ k_cache,
                                                          float* __restrict__ v_cache, uint32_t* __restrict__ fault) {
    const uint32_t token = blockIdx.x;
    const uint32_t row = token / t, i = token % t;
    const uint32_t width = (q_heads + 2u * kv_heads) * head_dim;
    const uint64_t named = (uint64_t)positions[i];
    if (named >= max_seq) {  // outside the caches and the tables: touch nothing, say so
        if (threadIdx.x == 0) atomicOr(fault, (uint32_t)kFaultBadPosition);
        return;
    }
    const uint32_t slot = (uint32_t)named;
    const uint32_t half = head_dim / 2u;
    for (uint32_t j = threadIdx.x; j < width; j += blockDim.x) {
        const uint32_t head = j / head_dim, dd = j % head_dim;
        const float* src = qkv + (size_t)token * width + (size_t)head * head_dim;
        const float v = src[dd];
        if (head >= q_heads + kv_heads) {  // value head: plain append
            const uint32_t h = head - q_heads - kv_heads;
            v_cache[(((size_t)row * kv_heads + h) * max_seq + slot) * head_dim + dd] = v;
            continue;
        }
        const float partner = dd < half ? -src[dd + half] : src[dd - half];
        const float c = cos_table[(size_t)slot * head_dim + dd], s = sin_table[(size_t)slot * head_dim + dd];
        const float y = __fadd_rn(__fmul_rn(v, c), __fmul_rn(partner, s));
        if (head < q_heads) q_out[((size_t)token * q_heads + head) * head_dim + dd] = y;
        else k_cache[(((size_t)row * kv_heads + (head - q_heads)) * max_seq + slot) * head_dim + dd] = y;
    }
}

// The same for head sizes that are powers of two (8 to 1024) and 16-byte aligned operands: a thread takes four
// channels of a head's first half and their partners of the second, so every value is loaded once and all
// accesses are 16 bytes.  The workgroup's size is a multiple of a head's chunks: a thread keeps its channels
// from head to head, and with them its cosines and sines.  Two chunks are requested before the first is used.
// Bound by memory: 134 MB for 32 prompts of 128 tokens with 16 query and 8 KV heads of 128, 21.4 us
// (one channel a thread, its partner loaded again and the tables once per head: 42.9).
__global__ __launch_bounds__(256) void rope_append_chunks_kernel(const float* __restrict__ qkv,
                                                                 const float* __restrict__ cos_table,
                                                                 const float* __restrict__ sin_table,
                                                                 const int64_t* __restrict__ positions, uint32_t t,
                                                                 uint32_t q_heads, uint32_t kv_heads, uint32_t head_dim,
                                                                 uint32_t max_seq, float* __restrict__ q_out,
                                                                 float* __restrict__ k_cache, float* __restrict__ v_cache,
                                                                 uint32_t* __restrict__ fault) {
    typedef float v4 __attribute__((ext_vector_type(4)));
    struct Pair {
        v4 low, high;
    };
    const uint32_t token = blockIdx.x, row = token / t, i = token % t;
    const uint64_t named = (uint64_t)positions[i];
    if (named >= max_seq) {  // outside the caches and the tables: touch nothing, say so
        if (threadIdx.x == 0) atomicOr(fault, (uint32_t)kFaultBadPosition);
        return;
    }
    const uint32_t slot = (uint32_t)named, half = head_dim / 2u;
    const uint32_t shift = 31u - (uint32_t)__builtin_clz(half / 4u);  // log2 of the chunks of a head
    const uint32_t heads = q_heads + 2u * kv_heads, units = heads << shift;
    const uint32_t dd = (threadIdx.x & ((1u << shift) - 1u)) * 4u;
    const float* src = qkv + (size_t)token * heads * head_dim + dd;
    auto pair_at = [&](const float* at) {
        return Pair{*reinterpret_cast<const v4*>(at), *reinterpret_cast<const v4*>(at + half)};
    };
    auto take = [&](uint32_t u) { return pair_at(src + (size_t)(min(u, units - 1u) >> shift) * head_dim); };
    const Pair c = pair_at(cos_table + (size_t)slot * head_dim + dd), s = pair_at(sin_table + (size_t)slot * head_dim + dd);
    auto put = [&](uint32_t u, const Pair& in) {
        const uint32_t head = u >> shift;
        Pair y = in;  // value head: plain append
        if (head < q_heads + kv_heads) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                y.low[e] = __fadd_rn(__fmul_rn(in.low[e], c.low[e]), __fmul_rn(-in.high[e], s.low[e]));
                y.high[e] = __fadd_rn(__fmul_rn(in.high[e], c.high[e]), __fmul_rn(in.low[e], s.high[e]));
            }
        }
        float* dst = head < q_heads ? q_out + ((size_t)token * q_heads + head) * head_dim
                     : head < q_heads + kv_heads
                         ? k_cache + (((size_t)row * kv_heads + (head - q_heads)) * max_seq + slot) * head_dim
                         : v_cache + (((size_t)row * kv_heads + (head - q_heads - kv_heads)) * max_seq + slot) * head_dim;
        *reinterpret_cast<v4*>(dst + dd) = y.low;
        *reinterpret_cast<v4*>(dst + dd + half) = y.high;
    };
    for (uint32_t u = threadIdx.x; u < units; u += 2u * blockDim.x) {
        const Pair a = take(u), b = take(u + blockDim.x);
        put(u, a);
        if (u + blockDim.x < units) put(u + blockDim.x, b);
    }
}

// grid (rows * t, q_heads / REP), block 256: a workgroup takes REP query heads that share one KV
// head, so every K and V row is read once for all of them.  LDS per head: q[head_dim] +
// scores[max_seq] + partial[8][head_dim] floats.  Scores: one thread per visible slot (its whole
// dot products, 16-byte loads, all independent); P.V: the slots split over eight groups of
// 32 threads, a thread four channels.
//
// FUSED (decode, t = 1): q is the qkv row as the linear wrote it.  The workgroup rotates its own
// query heads and the new key of its KV head itself (the arithmetic of rope_append_kernel), uses
// that key and the new value from LDS for the slot being appended, and the first workgroup of
// each KV group also stores them in the caches for later steps; slots before the new one come
// from the caches, so workgroups do not depend on each other.  Every slot is still handled by
// the thread, and in the order, that the unfused kernel gives it: the results are the same bits.
//
// Scores, NC = head_dim / 32 in {1, 4, 8}: eight lanes share a key row, each loading the 16-byte
// chunks c = lane%8 + 8*i, so one load instruction of a wavefront covers eight rows with whole
// 128-byte lines (a thread per row touches 64 lines with every load and refetches each of them
// eight times once the rows outgrow the L1); the eight partial dots meet in three xor-shuffles.
// Rows of four passes (128 slots) are requested before the first is used.  NC = 0 keeps the
// thread-per-row loop for other head sizes.
template <int REP, bool FUSED, int NC>
__global__ __launch_bounds__(256) void gqa_attention_kernel(const float* __restrict__ q,
                                                            float* __restrict__ k_cache,
                                                            float* __restrict__ v_cache,
                                                            const int64_t* __restrict__ positions, uint32_t t,
                                                            uint32_t q_heads, uint32_t kv_heads, uint32_t head_dim,
                                                            uint32_t max_seq, float scale, float* __restrict__ out,
                                                            const float* __restrict__ cos_table,
                                                            const float* __restrict__ sin_table,
                                                            uint32_t* __restrict__ fault) {
    const uint32_t per_head = 9u * head_dim + max_seq;
    float* lds = reinterpret_cast<float*>(glue_lds);
    float* k_new = lds + REP * per_head;  // FUSED: the appended key and value, head_dim floats each
    float* v_new = k_new + head_dim;
    const uint32_t token = blockIdx.x;
    const uint32_t head0 = blockIdx.y * REP;
    const uint32_t row = token / t, i = token % t;
    const uint32_t kvh = head0 / (q_heads / kv_heads);
    const uint64_t named = (uint64_t)positions[i];
    if (named >= max_seq) {  // (the whole workgroup) outside the caches: touch nothing, say so
        if (threadIdx.x == 0) atomicOr(fault, (uint32_t)kFaultBadPosition);
        return;
    }
    const uint32_t position = (uint32_t)named;
    const uint32_t visible = position + 1u;  // slots 0 .. position
    // slots read from the caches: all visible ones, or all before the one being appended
    const uint32_t cached = FUSED ? position : visible;
    float* kbase = k_cache + ((size_t)row * kv_heads + kvh) * max_seq * head_dim;
    float* vbase = v_cache + ((size_t)row * kv_heads + kvh) * max_seq * head_dim;
    // Cached rows arrive in blocks that are requested two blocks ahead of their use, the first
    // two before the query is ready: every workgroup of the launch is resident at once and in the
    // same phase, each dependent request costs all of them a round trip to a loaded memory
    // (2-3 us), and up to 256 slots this way cost one for the keys and one for the values.  A
    // request never depends on a branch: rows past the end are clamped to the last cached one
    // (row 0 of the cache when there is none), so they cost no memory traffic and the waits
    // stay exact.
    // rows of PASSES passes of 32 are in a block (fewer at head size 256, whose rows are twice as
    // long: the two blocks must leave room for three wavefronts per SIMD where they can)
    constexpr int PASSES = NC > 4 ? 2 : 4, KC = NC > 0 ? NC : 1;
    const uint32_t last_cached = max(cached, 1u) - 1u;
    const uint32_t lane8 = threadIdx.x & 7u, rowg = threadIdx.x >> 3;
    float4 kv_a[PASSES][KC], kv_b[PASSES][KC];
    auto request_keys = [&](float4 (&buf)[PASSES][KC], uint32_t s0) {
#pragma unroll
        for (int u = 0; u < PASSES; u++) {
            const uint32_t srow = min(s0 + u * 32u + rowg, last_cached);
            const float4* kr = reinterpret_cast<const float4*>(kbase + (size_t)srow * head_dim);
#pragma unroll
            for (int c = 0; c < KC; c++) buf[u][c] = kr[lane8 + 8u * c];
        }
    };
    if constexpr (FUSED && NC > 0) {
        // (head sizes up to 256: a thread rotates at most one channel)  The operands of the rotation
        // are requested before the keys: loads return in order, so requested after them they
        // would hold the query back until every key of both blocks had arrived.
        const uint32_t width = (q_heads + 2u * kv_heads) * head_dim, half = head_dim / 2u;
        const float* src = q + (size_t)token * width;
        const bool writer = head0 % (q_heads / kv_heads) == 0u;
        const uint32_t dd = threadIdx.x, mate = dd < half ? dd + half : dd - half;
        const bool rotates = dd < head_dim;
        float in_q[REP], in_q_mate[REP], in_k = 0.0f, in_k_mate = 0.0f, in_v = 0.0f, in_cos = 0.0f, in_sin = 0.0f;
#pragma unroll
        for (int h = 0; h < REP; h++) in_q[h] = in_q_mate[h] = 0.0f;
        if (rotates) {
#pragma unroll
            for (int h = 0; h < REP; h++) {
                in_q[h] = src[(size_t)(head0 + h) * head_dim + dd];
                in_q_mate[h] = src[(size_t)(head0 + h) * head_dim + mate];
            }
            in_k = src[(size_t)(q_heads + kvh) * head_dim + dd];
            in_k_mate = src[(size_t)(q_heads + kvh) * head_dim + mate];
            in_v = src[(size_t)(q_heads + kv_heads + kvh) * head_dim + dd];
            in_cos = cos_table[(size_t)position * head_dim + dd];
            in_sin = sin_table[(size_t)position * head_dim + dd];
        }
        request_keys(kv_a, 0u);
        request_keys(kv_b, 32u * PASSES);
        if (rotates) {
            auto rotated = [&](float own, float other) {  // the arithmetic of rope_append_kernel
                return __fadd_rn(__fmul_rn(own, in_cos), __fmul_rn(dd < half ? -other : other, in_sin));
            };
#pragma unroll
            for (int h = 0; h < REP; h++) lds[h * per_head + dd] = rotated(in_q[h], in_q_mate[h]);
            const float kn = rotated(in_k, in_k_mate);
            k_new[dd] = kn;
            v_new[dd] = in_v;
            if (writer) {
                kbase[(size_t)position * head_dim + dd] = kn;
                vbase[(size_t)position * head_dim + dd] = in_v;
            }
        }
    } else if constexpr (FUSED) {
        const uint32_t width = (q_heads + 2u * kv_heads) * head_dim, half = head_dim / 2u;
        const float* src = q + (size_t)token * width;
        const bool writer = head0 % (q_heads / kv_heads) == 0u;
        auto rotated = [&](const float* head, uint32_t dd) {
            const float partner = dd < half ? -head[dd + half] : head[dd - half];
            const float c = cos_table[(size_t)position * head_dim + dd], sn = sin_table[(size_t)position * head_dim + dd];
            return __fadd_rn(__fmul_rn(head[dd], c), __fmul_rn(partner, sn));
        };
        for (uint32_t dd = threadIdx.x; dd < head_dim; dd += 256u) {
#pragma unroll
            for (int h = 0; h < REP; h++) lds[h * per_head + dd] = rotated(src + (size_t)(head0 + h) * head_dim, dd);
            const float kn = rotated(src + (size_t)(q_heads + kvh) * head_dim, dd);
            const float vn = src[(size_t)(q_heads + kv_heads + kvh) * head_dim + dd];
            k_new[dd] = kn;
            v_new[dd] = vn;
            if (writer) {
                kbase[(size_t)position * head_dim + dd] = kn;
                vbase[(size_t)position * head_dim + dd] = vn;
            }
        }
    } else {
        float in_q[REP];
#pragma unroll
        for (int h = 0; h < REP; h++)
            in_q[h] = threadIdx.x < head_dim ? q[((size_t)token * q_heads + head0 + h) * head_dim + threadIdx.x] : 0.0f;
        if constexpr (NC > 0) {
            request_keys(kv_a, 0u);
            request_keys(kv_b, 32u * PASSES);
        }
#pragma unroll
        for (int h = 0; h < REP; h++) {
            if (threadIdx.x < head_dim) lds[h * per_head + threadIdx.x] = in_q[h];
            for (uint32_t dd = threadIdx.x + 256u; dd < head_dim; dd += 256u)
                lds[h * per_head + dd] = q[((size_t)token * q_heads + head0 + h) * head_dim + dd];
        }
    }
    __syncthreads();
    // P.V: group g of 32 threads takes slots g, g + 8, ..., a thread four channels of each; the
    // values come in batches of eight rows, requested two batches ahead like the keys, the first
    // two before the softmax.  (Requesting them while key blocks are still alive takes more than
    // 256 registers, which halves the workgroups a compute unit holds and was slower.)
    const uint32_t group = threadIdx.x >> 5, chunk = threadIdx.x & 31u;
    constexpr int VROWS = 8;
    float4 vv_a[VROWS], vv_b[VROWS];
    auto request_values = [&](float4 (&buf)[VROWS], uint32_t s0, uint32_t c4) {
#pragma unroll
        for (int u = 0; u < VROWS; u++) {
            const uint32_t s = min(s0 + group + 8u * u, last_cached);
            buf[u] = *reinterpret_cast<const float4*>(vbase + (size_t)s * head_dim + min(c4, head_dim - 4u));
        }
    };
    constexpr uint32_t BATCH = 8u * VROWS;  // slots per batch over the eight groups
    float m[REP];
#pragma unroll
    for (int h = 0; h < REP; h++) m[h] = -INFINITY;
    if constexpr (NC > 0) {
        // this lane's share of a row's dot with each query head, then the sum over the eight lanes
        auto finish = [&](float (&dot)[REP], uint32_t slot) {
#pragma unroll
            for (int h = 0; h < REP; h++) {
                float d = dot[h];
                // the eight lanes' sum as a butterfly of lane exchanges inside the register file
                // (an exchange through the LDS crossbar costs a round trip, and the three of a
                // row depend on each other): partners lane^1, lane^2, then the mirrored lane of
                // the other quad, whose four lanes all hold that quad's sum by then
                d += lane_exchange<kDppXor1>(d);
                d += lane_exchange<kDppXor2>(d);
                d += lane_exchange<kDppHalfMirror>(d);
                d = __fmul_rn(d, scale);
                if (lane8 == 0u) lds[h * per_head + head_dim + slot] = d;
                m[h] = fmaxf(m[h], d);
            }
        };
        // this lane's chunks of the query heads: registers when they are few (a read from LDS
        // cannot be hoisted over the score writes by the compiler and would repeat per row)
        constexpr bool Q_HELD = REP * KC <= 8;
        float4 q_held[Q_HELD ? REP : 1][Q_HELD ? KC : 1];
        if constexpr (Q_HELD) {
#pragma unroll
            for (int h = 0; h < REP; h++)
#pragma unroll
                for (int c = 0; c < KC; c++)
                    q_held[h][c] = *reinterpret_cast<const float4*>(lds + h * per_head + 4u * (lane8 + 8u * c));
        }
        auto accumulate = [&](float (&dot)[REP], const float4& kv, int c) {
#pragma unroll
            for (int h = 0; h < REP; h++) {
                float4 qv;
                if constexpr (Q_HELD) qv = q_held[h][c];
                else qv = *reinterpret_cast<const float4*>(lds + h * per_head + 4u * (lane8 + 8u * c));
                // fused multiply-adds: the score phase is bound by vector instruction issue (two
                // wavefronts per SIMD, each a few hundred instructions), and this halves it
                dot[h] = __builtin_fmaf(qv.x, kv.x, dot[h]);
                dot[h] = __builtin_fmaf(qv.y, kv.y, dot[h]);
                dot[h] = __builtin_fmaf(qv.z, kv.z, dot[h]);
                dot[h] = __builtin_fmaf(qv.w, kv.w, dot[h]);
            }
        };
        constexpr uint32_t BLOCK = 32u * PASSES;  // slots per block
        auto score_block = [&](float4 (&buf)[PASSES][KC], uint32_t s0) {
#pragma unroll
            for (int u = 0; u < PASSES; u++) {
                const uint32_t srow = s0 + u * 32u + rowg;
                float dot[REP];
#pragma unroll
                for (int h = 0; h < REP; h++) dot[h] = 0.0f;
#pragma unroll
                for (int c = 0; c < NC; c++) accumulate(dot, buf[u][c], c);
                // (all 64 lanes take part in the shuffles; a row past the end repeats the last
                // cached one, rewrites its score with the same value and is dropped from the
                // maximum here)
                float keep[REP];
#pragma unroll
                for (int h = 0; h < REP; h++) keep[h] = m[h];
                finish(dot, min(srow, last_cached));
                if (srow >= cached) {
#pragma unroll
                    for (int h = 0; h < REP; h++) m[h] = keep[h];
                }
            }
        };
        for (uint32_t s0 = 0; s0 < cached; s0 += 2u * BLOCK) {
            score_block(kv_a, s0);
            request_keys(kv_a, s0 + 2u * BLOCK);
            if (s0 + BLOCK < cached) score_block(kv_b, s0 + BLOCK);  // (a scalar branch)
            request_keys(kv_b, s0 + 3u * BLOCK);
        }
        if constexpr (FUSED) {
            // the appended slot, from LDS, by the eight lanes that own it in the unfused kernel and in
            // the same order of operations
            if (rowg == position % 32u) {
                float dot[REP];
#pragma unroll
                for (int h = 0; h < REP; h++) dot[h] = 0.0f;
#pragma unroll
                for (int c = 0; c < NC; c++)
                    accumulate(dot, *reinterpret_cast<const float4*>(k_new + 4u * (lane8 + 8u * c)), c);
                finish(dot, position);
            }
        }
    } else {
        if constexpr (FUSED) {
            // the appended slot, from LDS; it is the last slot of the thread that owns it
            if (threadIdx.x == position % 256u) {
                float dot[REP];
#pragma unroll
                for (int h = 0; h < REP; h++) dot[h] = 0.0f;
                for (uint32_t c = 0; c < head_dim / 4u; c++) {
#pragma unroll
                    for (int h = 0; h < REP; h++) {
                        const float* qs = lds + h * per_head;
                        dot[h] += qs[4 * c] * k_new[4 * c] + qs[4 * c + 1] * k_new[4 * c + 1] +
                                  qs[4 * c + 2] * k_new[4 * c + 2] + qs[4 * c + 3] * k_new[4 * c + 3];
                    }
                }
#pragma unroll
                for (int h = 0; h < REP; h++) {
                    dot[h] = __fmul_rn(dot[h], scale);
                    lds[h * per_head + head_dim + position] = dot[h];
                    m[h] = fmaxf(m[h], dot[h]);
                }
            }
        }
        for (uint32_t s = threadIdx.x; s < cached; s += 256u) {
            const float4* kr = reinterpret_cast<const float4*>(kbase + (size_t)s * head_dim);
            float dot[REP];
#pragma unroll
            for (int h = 0; h < REP; h++) dot[h] = 0.0f;
#pragma unroll 8
            for (uint32_t c = 0; c < head_dim / 4u; c++) {
                const float4 kv = kr[c];
#pragma unroll
                for (int h = 0; h < REP; h++) {
                    const float* qs = lds + h * per_head;
                    dot[h] += qs[4 * c] * kv.x + qs[4 * c + 1] * kv.y + qs[4 * c + 2] * kv.z + qs[4 * c + 3] * kv.w;
                }
            }
#pragma unroll
            for (int h = 0; h < REP; h++) {
                dot[h] = __fmul_rn(dot[h], scale);
                lds[h * per_head + head_dim + s] = dot[h];
                m[h] = fmaxf(m[h], dot[h]);
            }
        }
    }
    if constexpr (NC > 0) {
        request_values(vv_a, 0u, chunk * 4u);
        request_values(vv_b, BATCH, chunk * 4u);
    }
    // Softmax.  The heads' maxima cross the workgroup in one exchange (every thread scored slots
    // of every head); after that the 4 / REP wavefronts of a group own one head each, so the heads'
    // exponentials, sums and divisions run side by side instead of one head after the other.
    {
        constexpr uint32_t GROUP = 256u / REP, GROUP_WAVES = 4u / REP;
        __shared__ float wave_maxima[4 * REP], wave_sums[4];
        const uint32_t wave = threadIdx.x >> 6, own = threadIdx.x / GROUP, at = threadIdx.x % GROUP;
#pragma unroll
        for (int h = 0; h < REP; h++) {
            const float mw = wave_max(m[h]);
            if ((threadIdx.x & 63u) == 0u) wave_maxima[wave * REP + h] = mw;
        }
        __syncthreads();  // (also: the scores of a slot are read below by other threads than wrote them)
        float mh = wave_maxima[own];
#pragma unroll
        for (uint32_t w = 1; w < 4u; w++) mh = fmaxf(mh, wave_maxima[w * REP + own]);
        float* scores = lds + own * per_head + head_dim;
        float sum = 0.0f;
        for (uint32_t s = at; s < visible; s += GROUP) {
            const float e = expf(scores[s] - mh);
            scores[s] = e;
            sum += e;
        }
        sum = wave_sum_to_lane0(sum);
        if ((threadIdx.x & 63u) == 0u) wave_sums[wave] = sum;
        __syncthreads();
        float total = wave_sums[own * GROUP_WAVES];
#pragma unroll
        for (uint32_t w = 1; w < GROUP_WAVES; w++) total += wave_sums[own * GROUP_WAVES + w];
        for (uint32_t s = at; s < visible; s += GROUP) scores[s] = __fdiv_rn(scores[s], total);
    }
    __syncthreads();
    for (uint32_t c4 = chunk * 4u; c4 < head_dim; c4 += 128u) {
        float4 acc[REP];
#pragma unroll
        for (int h = 0; h < REP; h++) acc[h] = make_float4(0.f, 0.f, 0.f, 0.f);
        auto weigh = [&](const float4& vv, uint32_t s) {
#pragma unroll
            for (int h = 0; h < REP; h++) {
                const float p = lds[h * per_head + head_dim + s];
                acc[h].x = __builtin_fmaf(p, vv.x, acc[h].x);
                acc[h].y = __builtin_fmaf(p, vv.y, acc[h].y);
                acc[h].z = __builtin_fmaf(p, vv.z, acc[h].z);
                acc[h].w = __builtin_fmaf(p, vv.w, acc[h].w);
            }
        };
        if constexpr (NC > 0) {
            auto weigh_batch = [&](float4 (&buf)[VROWS], uint32_t s0) {
#pragma unroll
                for (int u = 0; u < VROWS; u++) {
                    const uint32_t s = s0 + group + 8u * u;
                    if (s < cached) weigh(buf[u], s);
                }
            };
            if (c4 != chunk * 4u) {  // head sizes above 128: a later pass
                request_values(vv_a, 0u, c4);
                request_values(vv_b, BATCH, c4);
            }
            for (uint32_t s0 = 0; s0 < cached; s0 += 2u * BATCH) {
                weigh_batch(vv_a, s0);
                request_values(vv_a, s0 + 2u * BATCH, c4);
                if (s0 + BATCH < cached) weigh_batch(vv_b, s0 + BATCH);
                request_values(vv_b, s0 + 3u * BATCH, c4);
            }
        } else {
#pragma unroll 8
            for (uint32_t s = group; s < cached; s += 8u)
                weigh(*reinterpret_cast<const float4*>(vbase + (size_t)s * head_dim + c4), s);
        }
        if constexpr (FUSED) {
            if (group == position % 8u) {  // the appended slot closes its group's sum
                const float4 vv = *reinterpret_cast<const float4*>(v_new + c4);
#pragma unroll
                for (int h = 0; h < REP; h++) {
                    const float p = lds[h * per_head + head_dim + position];
                    acc[h].x = __builtin_fmaf(p, vv.x, acc[h].x);
                    acc[h].y = __builtin_fmaf(p, vv.y, acc[h].y);
                    acc[h].z = __builtin_fmaf(p, vv.z, acc[h].z);
                    acc[h].w = __builtin_fmaf(p, vv.w, acc[h].w);
                }
            }
        }
#pragma unroll
        for (int h = 0; h < REP; h++)
            *reinterpret_cast<float4*>(lds + h * per_head + head_dim + max_seq + group * head_dim + c4) = acc[h];
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < REP; h++) {
        const float* partial = lds + h * per_head + head_dim + max_seq;
        for (uint32_t dd = threadIdx.x; dd < head_dim; dd += 256u) {
            float total = 0.0f;
#pragma unroll
            for (uint32_t g = 0; g < 8u; g++) total += partial[g * head_dim + dd];
            out[((size_t)token * q_heads + head0 + h) * head_dim + dd] = total;
        }
    }
}

// Prompt attention (t > 1 tokens per row).  The kernels above give every (token, head) its own
// workgroup, so a prompt of t tokens reads each key and value row t times.  Here a workgroup takes
// `tq` consecutive tokens of one row and the `rep` query heads of one KV head, qw = tq * rep <= 32
// queries, and walks that KV head's rows once for all of them, 64 slots at a time through LDS:
//   scores   thread (slot = tid % 64, wavefront) holds eight queries' dots with one staged key row;
//            the eight queries are the same for the whole wavefront, so they are read through the
//            scalar cache straight from global memory and cost no LDS bandwidth (as LDS broadcast
//            reads they took nine tenths of it and bounded the kernel)
//   softmax  a wavefront per query, over the slots that query may see (slot <= its position)
//   P.V      thread (four channels, tid / 32) holds four queries' sums over the staged value rows
// The arithmetic is that of the kernel above (f32, scores scaled after the dot, exp(x - max),
// a true division by the sum) with fused multiply-adds and its own summation order.
// grid (rows * ceil(t / tq), kv_heads), block 256.
// LDS: scores [qw][max_seq rounded up to 64], staged rows [64][head_dim + 4].
constexpr uint32_t kPrefillQueries = 32u, kPrefillSlots = 64u;

__global__ __launch_bounds__(256) void gqa_prefill_kernel(const float* __restrict__ q,
                                                          const float* __restrict__ k_cache,
                                                          const float* __restrict__ v_cache,
                                                          const int64_t* __restrict__ positions, uint32_t t,
                                                          uint32_t tq, uint32_t q_heads, uint32_t kv_heads,
                                                          uint32_t head_dim, uint32_t max_seq, float scale,
                                                          float* __restrict__ out, uint32_t* __restrict__ fault) {
    __shared__ uint32_t visible[kPrefillQueries];  // slots query i may see; 0: no such query
    const uint32_t rep = q_heads / kv_heads, qw = tq * rep;
    const uint32_t blocks = (t + tq - 1u) / tq;
    const uint32_t row = blockIdx.x / blocks, i0 = (blockIdx.x % blocks) * tq, kvh = blockIdx.y;
    // (a score row is a whole number of 64-slot blocks, so that P.V never has to guard a slot)
    const uint32_t hd4 = head_dim / 4u, pitch = head_dim + 4u, score_pitch = (max_seq + 63u) & ~63u;
    float* sc = reinterpret_cast<float*>(glue_lds);
    float* stage = sc + (size_t)qw * score_pitch;
    const float* kbase = k_cache + ((size_t)row * kv_heads + kvh) * max_seq * head_dim;
    const float* vbase = v_cache + ((size_t)row * kv_heads + kvh) * max_seq * head_dim;
    auto token_of = [&](uint32_t qi) { return i0 + qi / rep; };
    auto head_of = [&](uint32_t qi) { return kvh * rep + qi % rep; };

    if (threadIdx.x < kPrefillQueries) {
        const uint32_t qi = threadIdx.x;
        uint32_t v = 0u;
        if (qi < qw && token_of(qi) < t) {
            const uint64_t named = (uint64_t)positions[token_of(qi)];
            if (named >= max_seq) atomicOr(fault, (uint32_t)kFaultBadPosition);  // (its output row is left as it is)
            else v = (uint32_t)named + 1u;
        }
        visible[qi] = v;
    }
    __syncthreads();
    uint32_t span = 0u;  // slots any query of the workgroup sees
    for (uint32_t qi = 0; qi < qw; qi++) span = max(span, visible[qi]);

    // Rows s0 .. s0+63 of a cache (zeros past the span) go to the stage in two steps: requested
    // into registers, stored to LDS a block later -- the request of the next block is in flight
    // while this one is being used.
    constexpr int kStageRegs = 16;  // 64 rows x 256 floats over 256 threads, as 16-byte words
    const uint32_t stage_words = kPrefillSlots * hd4;
    auto fetch_rows = [&](const float* base, uint32_t s0, float4 (&v)[kStageRegs]) {
#pragma unroll
        for (int u = 0; u < kStageRegs; u++) {
            const uint32_t e = threadIdx.x + u * 256u, srow = s0 + e / hd4;
            v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (e < stage_words && srow < span)
                v[u] = *reinterpret_cast<const float4*>(base + (size_t)srow * head_dim + 4u * (e % hd4));
        }
    };
    auto commit_rows = [&](const float4 (&v)[kStageRegs]) {
#pragma unroll
        for (int u = 0; u < kStageRegs; u++) {
            const uint32_t e = threadIdx.x + u * 256u;
            if (e < stage_words) *reinterpret_cast<float4*>(stage + (size_t)(e / hd4) * pitch + 4u * (e % hd4)) = v[u];
        }
    };
    float4 ahead[kStageRegs];
    fetch_rows(kbase, 0u, ahead);

    {   // scores
        const uint32_t slot = threadIdx.x & 63u;
        const uint32_t first = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) * 8u);  // wave-uniform
        // (queries past qw, or of tokens past t, repeat a valid one; their dots are dropped below)
        const float* qrow[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint32_t qi = min(first + j, qw - 1u);
            qrow[j] = q + ((size_t)(row * t + min(token_of(qi), t - 1u)) * q_heads + head_of(qi)) * head_dim;
        }
        for (uint32_t s0 = 0; s0 < span; s0 += kPrefillSlots) {
            commit_rows(ahead);
            __syncthreads();
            // the next block of keys, or after the last one the first block of values
            if (s0 + kPrefillSlots < span) fetch_rows(kbase, s0 + kPrefillSlots, ahead);
            else fetch_rows(vbase, 0u, ahead);
            float dot[8];
#pragma unroll
            for (int j = 0; j < 8; j++) dot[j] = 0.0f;
            const float* krow = stage + (size_t)slot * pitch;
#pragma unroll 4
            for (uint32_t c = 0; c < hd4; c++) {  // (unrolled: the loads of four steps go out together)
                const float4 kv = *reinterpret_cast<const float4*>(krow + 4u * c);
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const float4 qv = *reinterpret_cast<const float4*>(qrow[j] + 4u * c);
                    dot[j] = __builtin_fmaf(qv.x, kv.x, dot[j]);
                    dot[j] = __builtin_fmaf(qv.y, kv.y, dot[j]);
                    dot[j] = __builtin_fmaf(qv.z, kv.z, dot[j]);
                    dot[j] = __builtin_fmaf(qv.w, kv.w, dot[j]);
                }
            }
            const uint32_t s = s0 + slot;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const uint32_t qi = first + j;
                if (qi < qw && s < visible[qi]) sc[(size_t)qi * score_pitch + s] = __fmul_rn(dot[j], scale);
            }
            __syncthreads();
        }
    }
    {   // softmax: probabilities over the visible slots, zeros from there to the span
        const uint32_t lane = threadIdx.x & 63u;
        for (uint32_t qi = threadIdx.x >> 6; qi < qw; qi += 4u) {  // (uniform per wavefront)
            float* mine = sc + (size_t)qi * score_pitch;
            const uint32_t seen = visible[qi];
            if (seen != 0u) {
                float m = -INFINITY;
                for (uint32_t s = lane; s < seen; s += 64u) m = fmaxf(m, mine[s]);
                m = wave_max(m);
                float sum = 0.0f;
                for (uint32_t s = lane; s < seen; s += 64u) {
                    const float e = expf(mine[s] - m);
                    mine[s] = e;
                    sum += e;
                }
                sum = wave_sum(sum);
                for (uint32_t s = lane; s < seen; s += 64u) mine[s] = __fdiv_rn(mine[s], sum);
            }
            const uint32_t span_blocks = (span + kPrefillSlots - 1u) / kPrefillSlots * kPrefillSlots;
            for (uint32_t s = seen + lane; s < span_blocks; s += 64u) mine[s] = 0.0f;
        }
    }
    __syncthreads();
    {   // P.V
        const uint32_t c4 = (threadIdx.x & 31u) * 4u, first = (threadIdx.x >> 5) * 4u;
        float4 acc[2][4];  // channel passes c4 and c4 + 128 (head sizes up to 256) x four queries
#pragma unroll
        for (int pass = 0; pass < 2; pass++)
#pragma unroll
            for (int j = 0; j < 4; j++) acc[pass][j] = make_float4(0.f, 0.f, 0.f, 0.f);
        for (uint32_t s0 = 0; s0 < span; s0 += kPrefillSlots) {
            commit_rows(ahead);
            __syncthreads();
            if (s0 + kPrefillSlots < span) fetch_rows(vbase, s0 + kPrefillSlots, ahead);
            // (every row of the block: the staged rows past the span are zeros and so are their
            // probabilities, and a fixed count lets the reads of eight rows go out together)
#pragma unroll 8
            for (uint32_t r = 0; r < kPrefillSlots; r++) {
                float p[4];
#pragma unroll
                for (int j = 0; j < 4; j++) p[j] = sc[(size_t)min(first + j, qw - 1u) * score_pitch + s0 + r];
#pragma unroll
                for (int pass = 0; pass < 2; pass++) {
                    const uint32_t cc = c4 + pass * 128u;
                    if (cc < head_dim) {
                        const float4 vv = *reinterpret_cast<const float4*>(stage + (size_t)r * pitch + cc);
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            acc[pass][j].x = __builtin_fmaf(p[j], vv.x, acc[pass][j].x);
                            acc[pass][j].y = __builtin_fmaf(p[j], vv.y, acc[pass][j].y);
                            acc[pass][j].z = __builtin_fmaf(p[j], vv.z, acc[pass][j].z);
                            acc[pass][j].w = __builtin_fmaf(p[j], vv.w, acc[pass][j].w);
                        }
                    }
                }
            }
            __syncthreads();
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t qi = first + j;
            if (qi >= qw || token_of(qi) >= t || visible[qi] == 0u) continue;
            float* dst = out + ((size_t)(row * t + token_of(qi)) * q_heads + head_of(qi)) * head_dim;
#pragma unroll
            for (int pass = 0; pass < 2; pass++) {
                const uint32_t cc = c4 + pass * 128u;
                if (cc < head_dim) *reinterpret_cast<float4*>(dst + cc) = acc[pass][j];
            }
        }
    }
}

// The same prompt attention for head sizes 64 and 128 on the f32 matrix pipes (v_mfma_f32_32x32x2f32:
// full f32 products and sums, not a reduced-precision format), every wavefront by itself: no LDS stage,
// no barrier, nothing but matrix instructions with loads between them.  A wavefront takes `tq`
// consecutive tokens of one row and the query heads of one KV head, up to 32 queries, and walks the
// visible slots 32 at a time with a running maximum and sum (softmax rescaled as the maximum grows).
// Lane l is r = l % 32, h = l / 32:
//   scores  transposed, keys as the A operand: MFMA (j, e) adds channels 8j + e (h = 0) and 8j + 4 + e
//           (h = 1) of key row r and query r, so lane l ends with query r's scores of the 16 slots
//           8 * (v / 4) + 4h + v % 4
//   P.V     transposed, values as the A operand: MFMA v adds just those two slots (one per h), so the
//           probabilities are the B operand from the registers where they already are.  Row r of
//           channel tile c is channel VW * r + c (VW = head size / 32): a value load is VW consecutive
//           floats a lane, and the output leaves the same way.
// Bound by the matrix pipes (128 MFMAs of 64 cycles per 32 slots and 128 channels: 17 us for 32 prompts of
// 128 tokens, 16 query and 8 KV heads) and by 100 MB of queries, cache and outputs (20 us); measured 41.5 us.
// With keys and values staged through LDS by four wavefronts and the scores kept there, three barriers per
// 64 slots, the same launch took 99.7 us; heads of 64 on the vector kernel above 76.6, here 17.2.  The loads are a ring of RING 16-byte
// registers, RING * 256 cycles of MFMAs ahead of their use; the fence behind each refill keeps the
// scheduler from collecting them.
// SPLIT wavefronts of a workgroup share their queries and take the 32-slot tiles in turn, then merge
// their sums through LDS; 1: the four take the queries of four neighbouring token blocks.
typedef float v16f __attribute__((ext_vector_type(16)));

template <int HD, int SPLIT>
__global__ __launch_bounds__(256, 2) void gqa_prefill_mfma_kernel(const float* __restrict__ q,
                                                                  const float* __restrict__ k_cache,
                                                                  const float* __restrict__ v_cache,
                                                                  const int64_t* __restrict__ positions, uint32_t rows,
                                                                  uint32_t t, uint32_t tq, uint32_t q_heads,
                                                                  uint32_t kv_heads, uint32_t max_seq, float scale,
                                                                  float* __restrict__ out, uint32_t* __restrict__ fault) {
    static_assert((HD == 64 || HD == 128) && (SPLIT == 1 || SPLIT == 4), "see the launch");
    constexpr int RING = 8, KE = HD / 8, VE = HD / 8, VW = HD / 32;  // 16-byte loads of keys and values per tile
    static_assert((KE + VE) % RING == 0 && RING <= KE, "a ring register keeps its place from tile to tile");
    typedef float out_vec __attribute__((ext_vector_type(VW), aligned(4)));  // (`out` may start at any float)
    const uint32_t lane = threadIdx.x & 63u, r = lane & 31u, h = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t rep = q_heads / kv_heads, qw = tq * rep, blocks = (t + tq - 1u) / tq;
    // The workgroups of the last tokens, which see the most slots, come first, and every other one has
    // its wavefronts in reverse: a SIMD that holds one of the long and one of the short ones is even.
    const uint32_t pairs = rows * kv_heads, pair = blockIdx.x % pairs, turn = blockIdx.x / pairs;
    const uint32_t row = pair / kv_heads, kvh = pair % kv_heads;
    uint32_t block;
    if constexpr (SPLIT > 1) {
        block = blocks - 1u - turn;
    } else {
        const uint32_t from_end = turn * 4u + ((turn & 1u) ? 3u - wave : wave);
        if (from_end >= blocks) return;
        block = blocks - 1u - from_end;
    }
    const float* kbase = k_cache + ((size_t)row * kv_heads + kvh) * max_seq * HD;
    const float* vbase = v_cache + ((size_t)row * kv_heads + kvh) * max_seq * HD;

    const uint32_t token = block * tq + r / rep, head = kvh * rep + r % rep;
    const bool exists = r < qw && token < t;
    uint32_t visible = 0u;  // slots query r may see
    if (exists) {
        const uint64_t named = (uint64_t)positions[token];
        if (named >= max_seq) atomicOr(fault, (uint32_t)kFaultBadPosition);  // (its output row is left as it is)
        else visible = (uint32_t)named + 1u;
    }
    uint32_t span = visible;
#pragma unroll
    for (int d = 1; d < 32; d <<= 1) span = max(span, (uint32_t)__shfl_xor((int)span, d));
    span = __builtin_amdgcn_readfirstlane(span);
    if (span == 0u) return;  // (the same in every wavefront that shares these queries)

    float4 qreg[KE];  // channels 8j + 4h .. +3 of query r (zeros for a query that does not exist)
    {
        const float* src = q + ((size_t)(row * t + (exists ? token : 0u)) * q_heads + (exists ? head : 0u)) * HD + 4u * h;
#pragma unroll
        for (int j = 0; j < KE; j++)
            qreg[j] = exists ? *reinterpret_cast<const float4*>(src + 8 * j) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    // Load e of the tile at s0: key chunks first, then value slots.  Slots past the span repeat its last
    // (their probabilities are zero, and what the cache holds there is nobody's).
    float4 ring[RING];
    auto fetch = [&](auto e_tag, uint32_t s0) {
        constexpr int e = decltype(e_tag)::value;
        if constexpr (e < KE) {
            ring[e % RING] = *reinterpret_cast<const float4*>(kbase + (size_t)min(s0 + r, span - 1u) * HD + 8 * e + 4u * h);
        } else if constexpr (VW == 4) {
            constexpr int v = e - KE;
            const uint32_t slot = min(s0 + 8u * (v / 4) + 4u * h + v % 4, span - 1u);
            ring[e % RING] = *reinterpret_cast<const float4*>(vbase + (size_t)slot * HD + 4u * r);
        } else {
            constexpr int v = 2 * (e - KE);
            const uint32_t slot = s0 + 8u * (v / 4) + 4u * h + v % 4;
            const float2 a = *reinterpret_cast<const float2*>(vbase + (size_t)min(slot, span - 1u) * HD + 2u * r);
            const float2 b = *reinterpret_cast<const float2*>(vbase + (size_t)min(slot + 1u, span - 1u) * HD + 2u * r);
            ring[e % RING] = make_float4(a.x, a.y, b.x, b.y);
        }
    };
    constexpr uint32_t STEP = 32u * SPLIT;
    const uint32_t first = SPLIT > 1 ? 32u * wave : 0u;
    static_for<RING>([&](auto e_tag) { fetch(e_tag, first); });

    float m = -INFINITY, sum = 0.0f;  // of query r, the same in both lanes that hold it
    v16f o[VW];
#pragma unroll
    for (int c = 0; c < VW; c++)
#pragma unroll
        for (int v = 0; v < 16; v++) o[c][v] = 0.0f;
    for (uint32_t s0 = first; s0 < span; s0 += STEP) {
        auto refill = [&](auto e_tag) {  // the ring register of load e takes load e + RING
            constexpr int e = decltype(e_tag)::value + RING;
            if constexpr (e < KE + VE) fetch(IC<e>{}, s0);
            else fetch(IC<e - KE - VE>{}, s0 + STEP);
            __builtin_amdgcn_sched_barrier(0);
        };
        // A dot's error grows with the length of its chain of sums: a chain for every 32 channels, joined in pairs.
        v16f chain[HD / 32];
#pragma unroll
        for (int n = 0; n < HD / 32; n++)
#pragma unroll
            for (int v = 0; v < 16; v++) chain[n][v] = 0.0f;
        auto join = [&](int to, int from) {
#pragma unroll
            for (int v = 0; v < 16; v++) chain[to][v] = __fadd_rn(chain[to][v], chain[from][v]);
        };
        static_for<KE>([&](auto e_tag) {
            constexpr int e = decltype(e_tag)::value, n = e / 4;
            const float4 kv = ring[e % RING];
            chain[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.x, qreg[e].x, chain[n], 0, 0, 0);
            chain[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.y, qreg[e].y, chain[n], 0, 0, 0);
            chain[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.z, qreg[e].z, chain[n], 0, 0, 0);
            chain[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.w, qreg[e].w, chain[n], 0, 0, 0);
            if constexpr (HD == 128 && e == 9) join(0, 1);  // (their last sums are out of the pipe by now)
            refill(e_tag);
        });
        if constexpr (HD == 128) {
            join(2, 3);
            join(0, 2);
        } else {
            join(0, 1);
        }
        v16f s = chain[0];
        auto both_halves = [&](float x) {  // the values of the two lanes that hold a query
            return __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
        };
        float top = -INFINITY;
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const uint32_t slot = s0 + 8u * (v / 4) + 4u * h + v % 4;
            s[v] = slot < visible ? __fmul_rn(s[v], scale) : -INFINITY;
            top = fmaxf(top, s[v]);
        }
        const auto tops = both_halves(top);
        const float grown = fmaxf(m, fmaxf(__uint_as_float(tops[0]), __uint_as_float(tops[1])));
        // (nothing visible yet, or only scores of -inf: any finite reference gives zeros)
        const float reference = grown == -INFINITY ? 0.0f : grown;
        const float keep = expf(m - reference);
        m = grown;
        float part = 0.0f;
#pragma unroll
        for (int v = 0; v < 16; v++) {
            s[v] = expf(s[v] - reference);  // (the reference is no NaN: a maximum passes them over)
            part += s[v];
        }
        const auto parts = both_halves(part);
        sum = __builtin_fmaf(sum, keep, __uint_as_float(parts[0]) + __uint_as_float(parts[1]));
#pragma unroll
        for (int c = 0; c < VW; c++)
#pragma unroll
            for (int v = 0; v < 16; v++) o[c][v] *= keep;
        static_for<VE>([&](auto e_tag) {
            constexpr int e = decltype(e_tag)::value;
            const float4 vv = ring[(KE + e) % RING];
            if constexpr (VW == 4) {
                o[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv.x, s[e], o[0], 0, 0, 0);
                o[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv.y, s[e], o[1], 0, 0, 0);
                o[2] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv.z, s[e], o[2], 0, 0, 0);
                o[3] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv.w, s[e], o[3], 0, 0, 0);
            } else {
                o[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv.x, s[2 * e], o[0], 0, 0, 0);
                o[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv.y, s[2 * e], o[1], 0, 0, 0);
                o[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv.z, s[2 * e + 1], o[0], 0, 0, 0);
                o[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv.w, s[2 * e + 1], o[1], 0, 0, 0);
            }
            refill(IC<KE + e>{});
        });
    }

    // Outputs that are not finite: a value that is not, of a slot that only others of the wavefront's queries see, was
    // multiplied by the zero probability of a query that does not, or the sums over probabilities up to 1 have
    // overflowed.  Such queries (a bit each) are computed once more over the slots they see, with the probabilities
    // divided first; channels ch0 .. ch0 + CH - 1, by the wavefront that stores them.
    auto recompute = [&](uint32_t queries, uint32_t ch0, auto channels_tag) {
        constexpr uint32_t CH = decltype(channels_tag)::value;
        __threadfence_block();  // (other lanes have stored these outputs)
        __builtin_amdgcn_s_waitcnt(0);
        for (; queries; queries &= queries - 1u) {
            const uint32_t qi = __builtin_ctz(queries), seen = __builtin_amdgcn_readlane(visible, qi);
            const size_t at = ((size_t)(row * t + block * tq + qi / rep) * q_heads + kvh * rep + qi % rep) * HD;
            auto score = [&](uint32_t slot) {
                float dot[2] = {};
                for (uint32_t c = 0; c < HD / 2u; c++)
#pragma unroll
                    for (uint32_t n = 0; n < 2u; n++)
                        dot[n] = __builtin_fmaf(q[at + HD / 2u * n + c], kbase[(size_t)slot * HD + HD / 2u * n + c], dot[n]);
                return __fmul_rn(__fadd_rn(dot[0], dot[1]), scale);
            };
            float best = -INFINITY, part = 0.0f;
            for (uint32_t slot = lane; slot < seen; slot += 64u) best = fmaxf(best, score(slot));
            best = wave_max(best);
            for (uint32_t slot = lane; slot < seen; slot += 64u) part += expf(score(slot) - best);
            const float total = wave_sum(part);
            constexpr int YS = (CH + 63u) / 64u;  // channels a lane
            float y[YS] = {};
            for (uint32_t s0 = 0; s0 < seen; s0 += 64u) {
                const float p = s0 + lane < seen ? __fdiv_rn(expf(score(s0 + lane) - best), total) : 0.0f;
                for (uint32_t j = 0; j < min(64u, seen - s0); j++) {
                    const float weight = lane_value(p, (int)j);
                    const float* value = vbase + (size_t)(s0 + j) * HD + ch0 + lane;
#pragma unroll
                    for (int i = 0; i < YS; i++)
                        if (lane + 64u * i < CH) y[i] = __builtin_fmaf(weight, value[64 * i], y[i]);
                }
            }
#pragma unroll
            for (int i = 0; i < YS; i++)
                if (lane + 64u * i < CH) out[at + ch0 + lane + 64u * i] = y[i];
        }
    };
    auto queries_of = [](bool lanes) {  // one bit a query from the two lanes that hold it
        const uint64_t both = __builtin_amdgcn_ballot_w64(lanes);
        return (uint32_t)both | (uint32_t)(both >> 32);
    };

    float* dst = out + ((size_t)(row * t + token) * q_heads + head) * HD;
    float any = 0.0f;  // stays zero while the outputs are finite
    if constexpr (SPLIT == 1) {
#pragma unroll
        for (int v = 0; v < 16; v++) {
            out_vec y;
#pragma unroll
            for (int c = 0; c < VW; c++) {
                y[c] = __fdiv_rn(o[c][v], sum);
                any = __builtin_fmaf(y[c], 0.0f, any);
            }
            if (visible != 0u) *reinterpret_cast<out_vec*>(dst + VW * (8u * (v / 4) + 4u * h + v % 4)) = y;
        }
        const uint32_t again = queries_of(visible != 0u && any != 0.0f);
        if (again) recompute(again, 0u, IC<HD>{});
    } else {
        // [wavefront][2 + 16 * VW][64]: maximum, sum, then the outputs; wavefront w merges the registers
        // 4w .. 4w + 3 of every channel tile
        constexpr uint32_t PART = (2u + 16u * VW) * 64u;
        float* mine = reinterpret_cast<float*>(glue_lds) + wave * PART + lane;
        mine[0] = m;
        mine[64] = sum;
#pragma unroll
        for (int c = 0; c < VW; c++)
#pragma unroll
            for (int v = 0; v < 16; v++) mine[(2 + v * VW + c) * 64] = o[c][v];
        __syncthreads();
        const float* parts = reinterpret_cast<const float*>(glue_lds) + lane;
        float top = -INFINITY, weight[SPLIT], total = 0.0f;
#pragma unroll
        for (int w = 0; w < SPLIT; w++) top = fmaxf(top, parts[w * PART]);
        const float reference = top == -INFINITY ? 0.0f : top;
#pragma unroll
        for (int w = 0; w < SPLIT; w++) {
            weight[w] = expf(parts[w * PART] - reference);
            total = __builtin_fmaf(parts[w * PART + 64], weight[w], total);
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            out_vec y;
#pragma unroll
            for (int c = 0; c < VW; c++) {
                float x = 0.0f;
#pragma unroll
                for (int w = 0; w < SPLIT; w++)
                    x = __builtin_fmaf(parts[w * PART + (2u + (4u * wave + u) * VW + c) * 64u], weight[w], x);
                y[c] = __fdiv_rn(x, total);
                any = __builtin_fmaf(y[c], 0.0f, any);
            }
            if (visible != 0u) *reinterpret_cast<out_vec*>(dst + VW * (8u * wave + 4u * h + u)) = y;
        }
        const uint32_t again = queries_of(visible != 0u && any != 0.0f);
        if (again) recompute(again, 8u * VW * wave, IC<8 * VW>{});
    }
}

// Whether the wavefronts of a workgroup share their queries and split the slots (see the kernel above): while
// the launch has not one wavefront for every SIMD, and more than one tile to split.  Measured, shared against
// apart (16 query / 8 KV heads of 128): 128 tokens of 1 row 10.6 / 24.6 us, of 8 rows (512 query blocks)
// 18.5 / 26.3, of 16 rows (1024) 33.1 / 28.2, of 32 rows 55.9 / 41.5; 190 tokens of 8 rows (768) 34.1 / 36.0;
// 64 tokens of 16 rows (512) 17.9 / 17.0.  Heads of 64, 128 tokens: 512 blocks 11.6 / 16.4, 1024 20.1 / 17.2.
bool split_prompt_slots(uint32_t query_blocks, uint32_t t, int compute_units) {
    return t > 32u && query_blocks < 4u * (uint32_t)(compute_units > 0 ? compute_units : 256);
}

// Query heads that share a workgroup (and with it every key and value row of their KV head):
// four for wide groups, two for any even group, else one.  With the key and value rows requested
// ahead of their use the kernel is bound by those reads, and two heads per workgroup (half the
// requests, half the workgroups) run a 32-row decode step of 16 heads 3 % faster than one; before
// that rewrite the kernel was latency bound and one head per workgroup was the faster choice.
// Few rows: while one head per workgroup still leaves no compute unit with two workgroups the launch
// is latency bound again, and the heads are faster apart (28 layers of 16 query / 8 KV heads of 128,
// per decode step: 1 row 1.13 -> 1.10 ms, 16 rows 1.385 -> 1.348; 32 rows 1.49 with two heads
// together, 1.55 apart).  (Measured at head size 128, which decode_attention.hip has since taken over but for the launches
// of four; the other sizes keep these lines.)
uint32_t heads_per_workgroup(uint32_t rep, uint32_t query_heads_in_launch, int compute_units) {
    if (query_heads_in_launch <= (uint32_t)(compute_units > 0 ? compute_units : 256)) return 1u;
    return rep >= 8u && rep % 4u == 0u ? 4u : rep % 2u == 0u ? 2u : 1u;
}

bool device_ready(VxHipContext* ctx) {
    return ctx && hipSetDevice(ctx->device) == hipSuccess;
}

// What a prepare entry point writes: row-major rows of d codes, or, on a context set to
// VXHIP_ACTIVATIONS_OPERAND32 and for at most 32 rows, operand order.
ActivationLayout prepared_layout(const VxHipContext* ctx, uint32_t rows, uint32_t d) {
    if (ctx->activation_layout == VXHIP_ACTIVATIONS_OPERAND32 && rows <= kOperandOrderRows)
        return ActivationLayout{(d + 15u) / 16u * 16u, 1u};
    return ActivationLayout{d, 0u};
}

// Which kernel an attention over the caches runs on, and what it needs.
enum class GqaRoute { None, PromptMfma, PromptScores, Token };
struct GqaPlan {
    GqaRoute route;
    uint32_t tokens;    // of a workgroup's walk (prompt kernels)
    uint32_t together;  // query heads a workgroup (per-token kernel)
    size_t lds;         // (dynamic) of the kernels that keep their scores
};

GqaPlan plan_gqa(const VxHipContext* ctx, uint32_t rows, uint32_t t, uint32_t q_heads, uint32_t kv_heads, uint32_t head_dim,
                 uint32_t max_seq) {
    const uint32_t rep = q_heads / kv_heads;
    const uint32_t together = heads_per_workgroup(rep, rows * t * q_heads, ctx->cu_count);
    const size_t token_lds = (size_t)together * (9u * head_dim + max_seq) * sizeof(float);  // of the per-token kernel
    auto prompt_lds = [&](uint32_t tokens) {  // of the prompt kernel that keeps its scores
        const size_t qw = (size_t)tokens * rep;
        return (qw * ((max_seq + 63u) & ~63u) + (size_t)kPrefillSlots * (head_dim + 4u)) * sizeof(float);
    };
    constexpr size_t kTokenLds = 60u * 1024u, kPromptLds = 150u * 1024u;
    // A prompt at the common head sizes: the matrix-pipe kernel.  (It holds no scores and would take any cache; those
    // that neither the prompt kernel with scores nor the per-token kernel could hold are refused as before it.)
    if (t >= 8u && rep <= kPrefillQueries && (head_dim == 128u || head_dim == 64u) &&
        (prompt_lds(1u) <= kPromptLds || token_lds <= kTokenLds))
        return {GqaRoute::PromptMfma, kPrefillQueries / rep, together, 0u};
    if (t >= 8u && rep <= kPrefillQueries && head_dim <= 256u) {
        // a prompt: tokens share the walk over the cache, as many per workgroup as the LDS holds
        uint32_t tq = kPrefillQueries / rep;
        while (tq > 1u && prompt_lds(tq) > kPromptLds) tq /= 2u;
        // two workgroups per compute unit hide each other's staging, if four tokens or more still
        // share a walk then
        if (prompt_lds(tq) > 78u * 1024u) {
            uint32_t fewer = tq;
            while (fewer > 4u && prompt_lds(fewer) > 78u * 1024u) fewer /= 2u;
            if (prompt_lds(fewer) <= 78u * 1024u) tq = fewer;
        }
        if (prompt_lds(tq) <= kPromptLds) return {GqaRoute::PromptScores, tq, together, prompt_lds(tq)};
    }
    return {token_lds > kTokenLds ? GqaRoute::None : GqaRoute::Token, 0u, together, token_lds};
}

// The query heads per workgroup (4, 2 or 1) and the head size pick the instance.
template <bool FUSED>
void launch_attention(VxHipContext* ctx, uint32_t together, dim3 grid, size_t lds, const float* q, float* k_cache,
                      float* v_cache, const int64_t* positions, uint32_t t, uint32_t q_heads, uint32_t kv_heads,
                      uint32_t head_dim, uint32_t max_seq, float scale, float* out, const float* cos_table,
                      const float* sin_table) {
    if (launch_decode_attention(ctx->stream, ctx->cu_count, grid.x, q, k_cache, v_cache, positions, t, q_heads, kv_heads,
                                head_dim, max_seq, scale, out, cos_table, sin_table, ctx->fault_dev))
        return;
#define VXHIP_ATTENTION(R, NC)                                                                                       \
    hipLaunchKernelGGL((gqa_attention_kernel<R, FUSED, NC>), grid, dim3(256), lds, ctx->stream, q, k_cache, v_cache, \
                       positions, t, q_heads, kv_heads, head_dim, max_seq, scale, out, cos_table, sin_table, ctx->fault_dev)
#define VXHIP_ATTENTION_HEADS(NC)     \
    do {                              \
        if (together == 4u) VXHIP_ATTENTION(4, NC); \
        else if (together == 2u) VXHIP_ATTENTION(2, NC); \
        else VXHIP_ATTENTION(1, NC);  \
    } while (0)
    switch (head_dim) {
        case 32: VXHIP_ATTENTION_HEADS(1); break;
        case 128: VXHIP_ATTENTION(4, 4); break;  // (the only ones that are not taken above)
        case 256: VXHIP_ATTENTION_HEADS(8); break;
        default: VXHIP_ATTENTION_HEADS(0); break;
    }
#undef VXHIP_ATTENTION_HEADS
#undef VXHIP_ATTENTION
}

// Embedding lookup (embedding.inc:5-16): out[i] = table[tokens[i]], one workgroup per token.
// The reference reads whatever an id outside the table points at; here such a row is zeros and
// a fault bit is raised.
__global__ __launch_bounds__(256) void embedding_gather_kernel(const int32_t* __restrict__ tokens,
                                                               const float* __restrict__ table,
                                                               float* __restrict__ out, uint32_t d, uint32_t vocab,
                                                               uint32_t* fault) {
    const int32_t id = tokens[blockIdx.x];
    const bool ok = id >= 0 && (uint32_t)id < vocab;
    const float* src = table + (size_t)(ok ? id : 0) * d;
    float* dst = out + (size_t)blockIdx.x * d;
    if (!ok && threadIdx.x == 0) atomicOr(fault, (uint32_t)kFaultBadToken);
    if ((d & 3u) == 0u) {
        for (uint32_t j = threadIdx.x * 4u; j < d; j += blockDim.x * 4u) {
            const float4 v = ok ? *reinterpret_cast<const float4*>(src + j) : make_float4(0.f, 0.f, 0.f, 0.f);
            *reinterpret_cast<float4*>(dst + j) = v;
        }
    } else {
        for (uint32_t j = threadIdx.x; j < d; j += blockDim.x) dst[j] = ok ? src[j] : 0.0f;
    }
}

// ArgMax over the last axis (reduction_argmax.inc:211-235): a scan in index order that replaces
// the best only on a strictly greater value, so ties keep the first index, a NaN is never
// chosen, and a NaN in element 0 wins the row (nothing compares greater than it).  A candidate
// (v, i) beats (bv, bi) if v > bv, or v == bv and i < bi, which gives the same answer in any
// evaluation order.  One workgroup per row; `advance` (optional) are counters the first
// workgroup increments, e.g. the decode position.
__global__ __launch_bounds__(1024) void argmax_rows_kernel(const float* __restrict__ x, uint32_t n,
                                                           int32_t* __restrict__ out, int64_t* advance,
                                                           uint32_t advance_count) {
    const float* row = x + (size_t)blockIdx.x * n;
    const float first = row[0];  // (requested with the row, not after the reduction)
    float bv = -INFINITY;
    uint32_t bi = 0xffffffffu;
    auto offer = [&](float v, uint32_t i) {
        if (v > bv || (v == bv && i < bi)) {
            bv = v;
            bi = i;
        }
    };
    if ((n & 3u) == 0u && ((uintptr_t)row & 15u) == 0u) {
        // eight loads go out together: one round trip for 32 elements a thread instead of eight (the
        // branches of `offer` keep the compiler from overlapping the loads of a plain loop)
        constexpr uint32_t U = 8;
        const uint32_t pitch = blockDim.x * 4u;
        for (uint32_t j0 = threadIdx.x * 4u; j0 < n; j0 += pitch * U) {
            float4 v[U];
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
                const uint32_t j = j0 + u * pitch;
                v[u] = j < n ? *reinterpret_cast<const float4*>(row + j) : float4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
                const uint32_t j = j0 + u * pitch;
                if (j < n) {
                    offer(v[u].x, j);
                    offer(v[u].y, j + 1u);
                    offer(v[u].z, j + 2u);
                    offer(v[u].w, j + 3u);
                }
            }
        }
    } else {
        for (uint32_t j = threadIdx.x; j < n; j += blockDim.x) offer(row[j], j);
    }
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_down(bv, off, 64);
        const uint32_t oi = __shfl_down(bi, off, 64);
        offer(ov, oi);
    }
    __shared__ float wave_v[16];
    __shared__ uint32_t wave_i[16];
    const uint32_t wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    if ((threadIdx.x & 63u) == 0u) {
        wave_v[wave] = bv;
        wave_i[wave] = bi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (uint32_t w = 1; w < waves; w++) offer(wave_v[w], wave_i[w]);
        out[blockIdx.x] = (first != first || bi == 0xffffffffu) ? 0 : (int32_t)bi;
    }
    if (blockIdx.x == 0 && advance && threadIdx.x < advance_count) advance[threadIdx.x] += 1;
}

}  // namespace

bool gqa_takes(const VxHipContext* ctx, uint32_t rows, uint32_t t, uint32_t q_heads, uint32_t kv_heads, uint32_t head_dim,
               uint32_t max_seq) {
    return head_dim % 4u == 0u && plan_gqa(ctx, rows, t, q_heads, kv_heads, head_dim, max_seq).route != GqaRoute::None;
}

}  // namespace vxhip

using namespace vxhip;

extern "C" {

VxHipStatus vxhip_rmsnorm_prepare_i8(VxHipContext* ctx, const float* input_dev, const float* gain_dev, uint32_t rows,
                                     uint32_t d, double eps, int8_t* prepared_dev, float* row_scales_dev,
                                     float* normalized_dev) {
    if (!ctx || !input_dev || !gain_dev || !prepared_dev || !row_scales_dev || !d || d > kMaxRowOpLength) {
        set_error("rmsnorm_prepare_i8: null argument or row length outside 1..%u", kMaxRowOpLength);
        return VXHIP_INVALID_ARGUMENT;
    }
    if (!rows) return VXHIP_OK;
    if (!device_ready(ctx)) return VXHIP_BACKEND_UNAVAILABLE;
    return launch_row_prepare(ctx->stream, RowOp::Norm, const_cast<float*>(input_dev), nullptr, gain_dev, eps, rows, d,
                              prepared_dev, prepared_layout(ctx, rows, d), row_scales_dev, normalized_dev);
}

VxHipStatus vxhip_add_rmsnorm_prepare_i8(VxHipContext* ctx, float* residual_dev, const float* delta_dev,
                                         const float* gain_dev, uint32_t rows, uint32_t d, double eps,
                                         int8_t* prepared_dev, float* row_scales_dev) {
    if (!ctx || !residual_dev || !delta_dev || !gain_dev || !prepared_dev || !row_scales_dev || !d ||
        d > kMaxRowOpLength) {
        set_error("add_rmsnorm_prepare_i8: null argument or row length outside 1..%u", kMaxRowOpLength);
        return VXHIP_INVALID_ARGUMENT;
    }
    if (!rows) return VXHIP_OK;
    if (!device_ready(ctx)) return VXHIP_BACKEND_UNAVAILABLE;
    return launch_row_prepare(ctx->stream, RowOp::Norm, residual_dev, delta_dev, gain_dev, eps, rows, d, prepared_dev,
                              prepared_layout(ctx, rows, d), row_scales_dev, nullptr);
}

VxHipStatus vxhip_swiglu_prepare_i8(VxHipContext* ctx, const float* gate_up_dev, uint32_t rows, uint32_t inter,
                                    int8_t* prepared_dev, float* row_scales_dev, float* activated_dev) {
    if (!ctx || !gate_up_dev || !prepared_dev || !row_scales_dev || !inter || inter > kMaxRowOpLength) {
        set_error("swiglu_prepare_i8: null argument or row length outside 1..%u", kMaxRowOpLength);
        return VXHIP_INVALID_ARGUMENT;
    }
    if (!rows) return VXHIP_OK;
    if (!device_ready(ctx)) return VXHIP_BACKEND_UNAVAILABLE;
    return launch_row_prepare(ctx->stream, RowOp::Swiglu, const_cast<float*>(gate_up_dev), nullptr, nullptr, 0.0, rows,
                              inter, prepared_dev, prepared_layout(ctx, rows, inter), row_scales_dev, activated_dev);
}

VxHipStatus vxhip_rope_append_kv(VxHipContext* ctx, const float* qkv_dev, const float* cos_dev, const float* sin_dev,
                                 const int64_t* positions_dev, uint32_t rows, uint32_t t, uint32_t q_heads,
                                 uint32_t kv_heads, uint32_t head_dim, uint32_t max_seq, float* q_out_dev,
                                 float* k_cache_dev, float* v_cache_dev) {
    if (!ctx || !qkv_dev || !cos_dev || !sin_dev || !positions_dev || !q_out_dev || !k_cache_dev || !v_cache_dev ||
        !q_heads || !kv_heads || q_heads % kv_heads || !head_dim || head_dim % 2u || head_dim > kMaxRopeHead || !max_seq) {
        set_error("rope_append_kv: null argument or unsupported head geometry");
        return VXHIP_INVALID_ARGUMENT;
    }
    if (!rows || !t) return VXHIP_OK;
    if (!device_ready(ctx)) return VXHIP_BACKEND_UNAVAILABLE;
    const uintptr_t operands = (uintptr_t)qkv_dev | (uintptr_t)cos_dev | (uintptr_t)sin_dev | (uintptr_t)q_out_dev |
                               (uintptr_t)k_cache_dev | (uintptr_t)v_cache_dev;
    const bool chunks = head_dim >= 8u && (head_dim & (head_dim - 1u)) == 0u && operands % 16u == 0u;
    const uint32_t threads = chunks && (q_heads + 2u * kv_heads) * (head_dim / 8u) <= 128u ? 128u : 256u;
    hipLaunchKernelGGL(chunks ? rope_append_chunks_kernel : rope_append_kernel, dim3(rows * t), dim3(threads), 0,
                       ctx->stream, qkv_dev, cos_dev, sin_dev, positions_dev, t, q_heads, kv_heads, head_dim, max_seq,
                       q_out_dev, k_cache_dev, v_cache_dev, ctx->fault_dev);
    VXHIP_TRY(hipGetLastError());
    return VXHIP_OK;
}

VxHipStatus vxhip_gqa_attention(VxHipContext* ctx, const float* q_dev, const float* k_cache_dev,
                                const float* v_cache_dev, const int64_t* positions_dev, uint32_t rows, uint32_t t,
                                uint32_t q_heads, uint32_t kv_heads, uint32_t head_dim, uint32_t max_seq,
                                float* out_dev) {
    if (!ctx || !q_dev || !k_cache_dev || !v_cache_dev || !positions_dev || !out_dev || !q_heads || !kv_heads ||
        q_heads % kv_heads || !head_dim || head_dim % 4u || !max_seq) {
        set_error("gqa_attention: null argument or unsupported geometry");
        return VXHIP_INVALID_ARGUMENT;
    }
    if (!rows || !t) return VXHIP_OK;
    if (!device_ready(ctx)) return VXHIP_BACKEND_UNAVAILABLE;
    const float scale = (float)(1.0 / sqrt((double)head_dim));
    const GqaPlan plan = plan_gqa(ctx, rows, t, q_heads, kv_heads, head_dim, max_seq);
    const uint32_t tq = plan.tokens;
    if (plan.route == GqaRoute::PromptMfma) {
        const uint32_t blocks = (t + tq - 1u) / tq, pairs = rows * kv_heads;
        const bool split = split_prompt_slots(pairs * blocks, t, ctx->cu_count);
        const uint32_t grid = pairs * (split ? blocks : (blocks + 3u) / 4u);
        const size_t lds = split ? 4u * (2u + head_dim / 2u) * 64u * sizeof(float) : 0u;
#define VXHIP_PROMPT(HD, SPLIT)                                                                                       \
    do {                                                                                                              \
        static std::atomic<uint64_t> configured{0};                                                                   \
        if (lds > 64u * 1024u && !raise_lds_limit((const void*)gqa_prefill_mfma_kernel<HD, SPLIT>, (int)lds, configured)) { \
            set_error("gqa_attention: the prompt kernel's LDS limit could not be raised");                            \
            return VXHIP_EXECUTION_FAILED;                                                                            \
        }                                                                                                             \
        hipLaunchKernelGGL((gqa_prefill_mfma_kernel<HD, SPLIT>), dim3(grid), dim3(256), lds, ctx->stream, q_dev,      \
                           k_cache_dev, v_cache_dev, positions_dev, rows, t, tq, q_heads, kv_heads, max_seq, scale,   \
                           out_dev, ctx->fault_dev);                                                                  \
    } while (0)
        if (head_dim == 128u && split) VXHIP_PROMPT(128, 4);
        else if (head_dim == 128u) VXHIP_PROMPT(128, 1);
        else if (split) VXHIP_PROMPT(64, 4);
        else VXHIP_PROMPT(64, 1);
#undef VXHIP_PROMPT
        VXHIP_TRY(hipGetLastError());
        return VXHIP_OK;
    }
    if (plan.route == GqaRoute::PromptScores) {
        static std::atomic<uint64_t> configured{0};
        if (!raise_lds_limit((const void*)gqa_prefill_kernel, 152 * 1024, configured)) {  // (plus its static 128 bytes)
            set_error("gqa_attention: the prompt kernel's LDS limit could not be raised");
            return VXHIP_EXECUTION_FAILED;
        }
        const dim3 grid(rows * ((t + tq - 1u) / tq), kv_heads);
        hipLaunchKernelGGL(gqa_prefill_kernel, grid, dim3(256), plan.lds, ctx->stream, q_dev, k_cache_dev,
                           v_cache_dev, positions_dev, t, tq, q_heads, kv_heads, head_dim, max_seq, scale, out_dev,
                           ctx->fault_dev);
        VXHIP_TRY(hipGetLastError());
        return VXHIP_OK;
    }
    if (plan.route == GqaRoute::None) {
        set_error("gqa_attention: head_dim/max_seq too large for the score buffer");
        return VXHIP_INVALID_ARGUMENT;
    }
    const dim3 grid(rows * t, q_heads / plan.together);
    launch_attention<false>(ctx, plan.together, grid, plan.lds, q_dev, const_cast<float*>(k_cache_dev),
                            const_cast<float*>(v_cache_dev), positions_dev, t, q_heads, kv_heads, head_dim, max_seq,
                            scale, out_dev, nullptr, nullptr);
    VXHIP_TRY(hipGetLastError());
    return VXHIP_OK;
}

VxHipStatus vxhip_rope_gqa_attention_decode(VxHipContext* ctx, const float* qkv_dev, const float* cos_dev,
                                            const float* sin_dev, const int64_t* position_dev, uint32_t rows,
                                            uint32_t q_heads, uint32_t kv_heads, uint32_t head_dim,
                                            uint32_t max_seq, float* k_cache_dev, float* v_cache_dev,
                                            float* out_dev) {
    if (!ctx || !qkv_dev || !cos_dev || !sin_dev || !position_dev || !k_cache_dev || !v_cache_dev || !out_dev ||
        !q_heads || !kv_heads || q_heads % kv_heads || !head_dim || head_dim % 4u || head_dim > 1024u || !max_seq) {
        set_error("rope_gqa_attention_decode: null argument or unsupported geometry");
        return VXHIP_INVALID_ARGUMENT;
    }
    if (!rows) return VXHIP_OK;
    if (!device_ready(ctx)) return VXHIP_BACKEND_UNAVAILABLE;
    const float scale = (float)(1.0 / sqrt((double)head_dim));
    const uint32_t rep = q_heads / kv_heads;
    const uint32_t together = heads_per_workgroup(rep, rows * q_heads, ctx->cu_count);
    const size_t lds = ((size_t)together * (9u * head_dim + max_seq) + 2u * head_dim) * sizeof(float);
    if (lds > 60u * 1024u) {
        set_error("rope_gqa_attention_decode: head_dim/max_seq too large for the score buffer");
        return VXHIP_INVALID_ARGUMENT;
    }
    const dim3 grid(rows, q_heads / together);
    launch_attention<true>(ctx, together, grid, lds, qkv_dev, k_cache_dev, v_cache_dev, position_dev, 1u,
                           q_heads, kv_heads, head_dim, max_seq, scale, out_dev, cos_dev, sin_dev);
    VXHIP_TRY(hipGetLastError());
    return VXHIP_OK;
}

VxHipStatus vxhip_embedding_gather_f32(VxHipContext* ctx, const int32_t* tokens_dev, const float* table_dev,
                                       uint32_t count, uint32_t d_model, uint32_t vocab, float* out_dev) {
    if (!ctx || !tokens_dev || !table_dev || !out_dev || !d_model || !vocab) {
        set_error("embedding_gather_f32: null argument or empty table");
        return VXHIP_INVALID_ARGUMENT;
    }
    if (!count) return VXHIP_OK;
    if (!device_ready(ctx)) return VXHIP_BACKEND_UNAVAILABLE;
    hipLaunchKernelGGL(embedding_gather_kernel, dim3(count), dim3(256), 0, ctx->stream, tokens_dev, table_dev,
                       out_dev, d_model, vocab, ctx->fault_dev);
    VXHIP_TRY(hipGetLastError());
    return VXHIP_OK;
}

VxHipStatus vxhip_argmax_rows_f32(VxHipContext* ctx, const float* input_dev, uint32_t rows, uint32_t n,
                                  int32_t* indices_dev, int64_t* advance_dev, uint32_t advance_count) {
    if (!ctx || !input_dev || !indices_dev || !n || (advance_count && !advance_dev) || advance_count > 64u) {
        set_error("argmax_rows_f32: null argument, empty axis or more than 64 counters");
        return VXHIP_INVALID_ARGUMENT;
    }
    if (!rows) return VXHIP_OK;
    if (!device_ready(ctx)) return VXHIP_BACKEND_UNAVAILABLE;
    const uint32_t block = n >= 4096u ? 1024u : n >= 1024u ? 256u : 64u;
    hipLaunchKernelGGL(argmax_rows_kernel, dim3(rows), dim3(block), 0, ctx->stream, input_dev, n, indices_dev,
                       advance_dev, advance_count);
    VXHIP_TRY(hipGetLastError());
    return VXHIP_OK;
}

}  // extern "C"
