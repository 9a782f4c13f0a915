// A small prompt of a pre-norm decoder as one call: the launches of every layer, issued from here.  Such a prompt is bound by the host
// that issues them -- 4 layers of hidden 1024 over 128 tokens take the device 222 us, and took 496 while a wrapper call with its checks
// and an output allocation stood in front of each of the ten launches of a layer.  The work is that of the entry points called
// below, one by one, with one workspace behind them; a larger prompt has linears that take what follows them (gemm_k64.hip).
#include "common.h"

#include <algorithm>

using namespace vxhip;

namespace {

// dst [rows][kept][width] = the last `kept` of src's [rows][t][width]; V: float or four of them
template <class V>
__global__ __launch_bounds__(256) void last_tokens_kernel(const V* __restrict__ src, uint32_t t, uint32_t kept, uint32_t width,
                                                          uint32_t total, V* __restrict__ dst) {
    const uint32_t e = blockIdx.x * 256u + threadIdx.x;
    if (e >= total) return;
    const uint32_t i = e % width, token = e / width, row = token / kept;
    dst[e] = src[((size_t)row * t + (t - kept) + (token - row * kept)) * width + i];
}

bool last_tokens(hipStream_t s, const float* src, uint32_t rows, uint32_t t, uint32_t kept, uint32_t width, float* dst) {
    const bool wide = width % 4u == 0u;  // (every buffer starts on a 256-byte boundary)
    const uint32_t w = wide ? width / 4u : width;
    const uint64_t total = (uint64_t)rows * kept * w;
    if (total > 0xffffffffull - 255u) return false;
    const dim3 grid((uint32_t)((total + 255u) / 256u));
    if (wide)
        hipLaunchKernelGGL(last_tokens_kernel<float4>, grid, dim3(256), 0, s, (const float4*)src, t, kept, w, (uint32_t)total, (float4*)dst);
    else
        hipLaunchKernelGGL(last_tokens_kernel<float>, grid, dim3(256), 0, s, src, t, kept, w, (uint32_t)total, dst);
    return hipGetLastError() == hipSuccess;
}

struct Workspace {
    float *stream, *wide, *q, *attention, *delta, *last_stream, *last_q, *last_attention, *scales;
    int8_t* codes;
    size_t bytes;
};

// `wide` holds a layer's [q | k | v], then its [gate | up]: neither outlives the other.
Workspace carve(const VxHipContext* ctx, const VxHipDecoderPrompt* p, char* base) {
    Workspace w{};
    size_t at = 0;
    auto take = [&](size_t bytes) {
        char* here = base + at;
        at += (bytes + 255u) / 256u * 256u;
        return here;
    };
    const size_t tokens = (size_t)p->rows * p->t;
    const uint32_t q_dim = p->q_heads * p->head_dim, qkv = q_dim + 2u * p->kv_heads * p->head_dim;
    uint32_t widest = qkv, longest = std::max(p->hidden, q_dim);
    for (uint32_t i = 0; i < p->layer_count; i++) {
        widest = std::max(widest, p->layers[i].gate_up->w.n);
        longest = std::max(longest, p->layers[i].gate_up->w.n / 2u);
    }
    w.stream = (float*)take(tokens * p->hidden * 4u);
    w.wide = (float*)take(tokens * widest * 4u);
    w.q = (float*)take(tokens * q_dim * 4u);
    w.attention = (float*)take(tokens * q_dim * 4u);
    w.delta = (float*)take(tokens * p->hidden * 4u);
    w.last_stream = (float*)take((size_t)p->rows * p->hidden * 4u);
    w.last_q = (float*)take((size_t)p->rows * 8u * q_dim * 4u);
    w.last_attention = (float*)take((size_t)p->rows * q_dim * 4u);
    w.scales = (float*)take(tokens * 4u);
    w.codes = (int8_t*)take(std::max(vxhip_context_prepared_bytes(ctx, (uint32_t)tokens, longest),
                                     vxhip_context_prepared_bytes(ctx, p->rows, longest)));
    w.bytes = at;
    return w;
}

// Tokens a row that go through the last layer's attention: the last eight, the fewest that run on the prompt kernels, which take caches
// that the per-token form does not (its limit is 60 KiB of scores, theirs 150).  The rows do not depend on each other: the same bits.
uint32_t tokens_seen_last(uint32_t t) { return t >= 8u ? 8u : 1u; }

// Everything that a step could refuse, so that no launch of a prompt runs where another will not.
bool admitted(const VxHipContext* ctx, const VxHipDecoderPrompt* p) {
    if (!ctx || !p || !p->tokens_dev || !p->embedding_dev || !p->layers || !p->layer_count || !p->final_gain_dev || !p->lm_head ||
        !p->cos_dev || !p->sin_dev || !p->positions_dev || !p->rows || p->t < 2u || !p->hidden || !p->q_heads || !p->kv_heads ||
        p->q_heads % p->kv_heads || !p->head_dim || !p->max_seq || p->t > p->max_seq ||
        (uint64_t)p->rows * p->t > 0xffffffffull || p->lm_head->w.k != p->hidden || !p->vocab || p->hidden > kMaxRowOpLength ||
        p->head_dim > kMaxRopeHead ||
        (p->layer_count > 1u && !gqa_takes(ctx, p->rows, p->t, p->q_heads, p->kv_heads, p->head_dim, p->max_seq)) ||
        !gqa_takes(ctx, p->rows, tokens_seen_last(p->t), p->q_heads, p->kv_heads, p->head_dim, p->max_seq) ||
        p->lm_head->device != ctx->device)
        return false;
    const uint64_t q_dim = (uint64_t)p->q_heads * p->head_dim, qkv = q_dim + 2ull * p->kv_heads * p->head_dim;
    for (uint32_t i = 0; i < p->layer_count; i++) {
        const VxHipDecoderLayer& L = p->layers[i];
        if (!L.gain1_dev || !L.gain2_dev || !L.qkv || !L.output || !L.gate_up || !L.down || !L.k_cache_dev || !L.v_cache_dev ||
            L.qkv->w.k != p->hidden || L.qkv->w.n != qkv || L.output->w.k != q_dim || L.output->w.n != p->hidden ||
            L.gate_up->w.k != p->hidden || L.gate_up->w.n % 2u || L.down->w.k != L.gate_up->w.n / 2u || L.down->w.n != p->hidden ||
            L.down->w.k > kMaxRowOpLength || L.qkv->device != ctx->device || L.output->device != ctx->device ||
            L.gate_up->device != ctx->device || L.down->device != ctx->device)
            return false;
    }
    return true;
}

}  // namespace

extern "C" {

size_t vxhip_decoder_prompt_workspace(const VxHipContext* ctx, const VxHipDecoderPrompt* p) {
    return admitted(ctx, p) ? carve(ctx, p, nullptr).bytes : 0u;
}

VxHipStatus vxhip_decoder_prompt(VxHipContext* ctx, const VxHipDecoderPrompt* p) {
    if (!admitted(ctx, p) || !p->workspace_dev || (uintptr_t)p->workspace_dev % 256u || !p->logits_dev || !p->next_dev) {
        set_error("decoder_prompt: a null argument, extents that do not fit each other or that a step does not take, or a linear of another device");
        return VXHIP_INVALID_ARGUMENT;
    }
    const Workspace w = carve(ctx, p, (char*)p->workspace_dev);
    if (w.bytes > p->workspace_bytes) {
        set_error("decoder_prompt: a workspace of %zu bytes, %zu are needed", p->workspace_bytes, w.bytes);
        return VXHIP_INVALID_ARGUMENT;
    }
    const uint32_t rows = p->rows, t = p->t, hidden = p->hidden, q_dim = p->q_heads * p->head_dim;
    const uint32_t all = rows * t;
#define VXHIP_STEP(expr)                            \
    do {                                            \
        const VxHipStatus s_ = (expr);              \
        if (s_ != VXHIP_OK) return s_;              \
    } while (0)
    // an int result of a linear: 0 is success
#define VXHIP_LINEAR(expr)                              \
    do {                                                \
        if ((expr) != 0) return VXHIP_INTERNAL;         \
    } while (0)
    float* x = w.stream;
    const float* pending = nullptr;  // what the next RMSNorm adds to the residual stream first
    uint32_t n = all;                // rows of the residual stream
    auto norm = [&](const float* gain) {
        return pending ? vxhip_add_rmsnorm_prepare_i8(ctx, x, pending, gain, n, hidden, p->eps, w.codes, w.scales)
                       : vxhip_rmsnorm_prepare_i8(ctx, x, gain, n, hidden, p->eps, w.codes, w.scales, nullptr);
    };
    VXHIP_STEP(vxhip_embedding_gather_f32(ctx, p->tokens_dev, p->embedding_dev, all, hidden, p->vocab, x));
    for (uint32_t li = 0; li < p->layer_count; li++) {
        const VxHipDecoderLayer& L = p->layers[li];
        const bool last = li + 1u == p->layer_count;
        VXHIP_STEP(norm(L.gain1_dev));
        VXHIP_LINEAR(vxhip_packed_linear_forward_a8(ctx, L.qkv, w.codes, w.scales, w.wide, nullptr, n));
        VXHIP_STEP(vxhip_rope_append_kv(ctx, w.wide, p->cos_dev, p->sin_dev, p->positions_dev, rows, t, p->q_heads, p->kv_heads,
                                        p->head_dim, p->max_seq, w.q, L.k_cache_dev, L.v_cache_dev));
        const float *q = w.q, *attention = w.attention;
        uint32_t seen = t;
        // Behind the cache append of the last layer only each row's last token goes on to the logits.
        if (last) {
            seen = tokens_seen_last(t);
            if (seen != t) {
                if (!last_tokens(ctx->stream, w.q, rows, t, seen, q_dim, w.last_q)) return VXHIP_INTERNAL;
                q = w.last_q;
            }
        }
        VXHIP_STEP(vxhip_gqa_attention(ctx, q, L.k_cache_dev, L.v_cache_dev, p->positions_dev + (t - seen), rows, seen, p->q_heads,
                                       p->kv_heads, p->head_dim, p->max_seq, w.attention));
        if (last) {
            if (!last_tokens(ctx->stream, x, rows, t, 1u, hidden, w.last_stream)) return VXHIP_INTERNAL;
            x = w.last_stream;
            if (seen > 1u) {
                if (!last_tokens(ctx->stream, w.attention, rows, seen, 1u, q_dim, w.last_attention)) return VXHIP_INTERNAL;
                attention = w.last_attention;
            }
            n = rows;
        }
        VXHIP_LINEAR(vxhip_packed_linear_forward_f32(ctx, L.output, attention, w.delta, n));
        pending = w.delta;
        VXHIP_STEP(norm(L.gain2_dev));
        VXHIP_LINEAR(vxhip_packed_linear_forward_a8(ctx, L.gate_up, w.codes, w.scales, w.wide, nullptr, n));
        VXHIP_STEP(vxhip_swiglu_prepare_i8(ctx, w.wide, n, L.down->w.k, w.codes, w.scales, nullptr));
        VXHIP_LINEAR(vxhip_packed_linear_forward_a8(ctx, L.down, w.codes, w.scales, w.delta, nullptr, n));
    }
    VXHIP_STEP(norm(p->final_gain_dev));
    VXHIP_LINEAR(vxhip_packed_linear_forward_a8(ctx, p->lm_head, w.codes, w.scales, p->logits_dev, nullptr, n));
#undef VXHIP_STEP
#undef VXHIP_LINEAR
    return vxhip_argmax_rows_f32(ctx, p->logits_dev, n, p->lm_head->w.n, p->next_dev, nullptr, 0u);
}

}  // extern "C"
