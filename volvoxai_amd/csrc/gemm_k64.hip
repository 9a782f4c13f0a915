// int8 MFMA GEMM for large prefill shapes on v_mfma_i32_16x16x64_i8: the requantizing epilogues
// of gemm_mfma.hip (same bytes), the same LDS stages and prepacked weights, but the matrix
// instruction with the long inner dimension.  Fed with random 8-bit operands the device is
// power limited and lowers its clock until the matrix pipes fit the budget; per delivered
// operation the 16x16x64 form moves a quarter of the accumulator registers of the 32x32x32
// form and sustains about 1.16 times its rate (3.7 against 3.2 POP/s in a register-only loop).
// Replaces, on gfx950, what the reference does on the CPU in vx_qgemm_w8a8_avx2
// (native/src/kernels/packed_quant_gemm.c:2411-2600).
//
// Operand roles as in gemm_mfma.hip: weights are the MFMA "A" operand (16 output channels x 64
// k), activations the "B" operand (64 k x 16 rows).  Lane l of an operand holds 16 consecutive
// k-bytes, chunk l/16 of the 64, of channel or row l%16; lane l of a result tile holds row
// l%16 and the four consecutive channels 4*(l/16) .. +3.
//
// One A operand is half of two adjacent 1 KiB blocks of the prepacked weight (common.h): lanes
// 0..31 read block 2t, lanes 32..63 block 2t+1, each its channel's two 16-byte slots.  The B
// operand comes from the row-major, XOR-swizzled activation image gemm_mfma.hip describes.
#include "common.h"
#include "device_math.h"
#include "epilogue.h"
#include "gemm_tile.h"
#include "row_math.h"

#include <stdio.h>
#include <string.h>

namespace vxhip {

namespace {

extern __shared__ __attribute__((aligned(1024))) char lds_raw[];

// WN x WM wavefronts, each owning TN x TM result tiles of 16 channels x 16 rows.  MODE is the
// requantizing Epilogue.  Two LDS stages of 128 k-bytes, i.e. two 64-wide MFMA steps each.
// FLIP: the activation bytes are unsigned; each activation fragment has its top bits flipped (one XOR per
// dword) in front of the first MFMA row of the step that uses it, so that a U8 input needs no pass of its own.
// DQ: the DequantizeLinear behind the QLinear rides in the epilogue -- each byte's value goes out as
// f32((q - dq_zp) * dq_scale) (a.dq_out, 16 bytes a lane and tile), the bytes themselves only if a.y is set.
template <int WN, int WM, int TN, int TM, int MODE, bool FLIP = false, bool DQ = false>
__global__ __launch_bounds__(WN* WM * 64) void gemm_k64_kernel(const GemmParams p) {
    static_assert(MODE != (int)Epilogue::DequantF32, "requantizing epilogues only");
    static_assert(TN % 4 == 0, "the epilogue transposes four channel tiles at a time");
    constexpr int NWAVES = WN * WM;
    constexpr int BN = WN * TN * 16, BM = WM * TM * 16;
    constexpr int KS = 4;  // 32-byte k-steps per stage (the unit of the weight blocks)
    constexpr int WBLK = (BN / 32) * KS, XBLK = BM / 8;  // 1 KiB blocks per stage
    static_assert(WBLK % NWAVES == 0 && XBLK % NWAVES == 0, "blocks must divide over waves");
    constexpr int WLOADS = WBLK / NWAVES, XLOADS = XBLK / NWAVES, NLOADS = WLOADS + XLOADS;
    constexpr int STAGE_BYTES = (WBLK + XBLK) * 1024;
    const LinearArgs& a = p.a;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int wave_n = wave % WN, wave_m = wave / WN;

    uint32_t m0, n0;
    {
        const TileOrigin t = tile_of_workgroup<BN, BM>(p);
        if (!t.valid) return;
        m0 = t.m0;
        n0 = t.n0;
    }

    // ---- operand loads (global -> LDS), as in gemm_mfma.hip ------------------------------
    const uint32_t w_lane = lane * 16u;
    const uint32_t panel_bytes = a.ksteps * 1024u;
    const int8_t* const w_tile = a.w + (size_t)(n0 / 32u) * panel_bytes;
    const uint32_t last_chunk = (a.k - 1u) / 16u;
    const uint32_t my_chunk = (lane & 7) ^ ((lane >> 3) & 7);
    uint32_t xrow[XLOADS];
#pragma unroll
    for (int i = 0; i < XLOADS; i++) {
        const int b = wave + i * NWAVES;
        uint32_t row = m0 + b * 8 + (lane >> 3);
        row = min(row, a.rows - 1u);
        xrow[i] = row * a.ldx;
    }
    const uint32_t ksteps_real = (a.k + 31u) / 32u;
    const uint32_t nkb = (ksteps_real + KS - 1) / KS;
    auto issue_one = [&](auto t_tag, uint32_t kb, int stage) {
        constexpr int t = decltype(t_tag)::value;
        kb = min(kb, nkb - 1u);  // a block past the end refills a stage nobody reads
        char* base = lds_raw + stage * STAGE_BYTES;
        if constexpr (t < WLOADS) {
            const uint32_t b = wave + t * NWAVES;
            const int8_t* src = w_tile + (size_t)(b / KS) * panel_bytes + (size_t)(kb * KS + b % KS) * 1024u;
            load_to_lds16(src + w_lane, base + b * 1024);
        } else {
            const uint32_t chunk16 = min(kb * 8u + my_chunk, last_chunk) * 16u;
            const uint32_t b = wave + (t - WLOADS) * NWAVES;
            load_to_lds16(a.x + (xrow[t - WLOADS] + chunk16), base + (WBLK + b) * 1024);
        }
    };

    v4i acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; i++)
#pragma unroll
        for (int j = 0; j < TM; j++) acc[i][j] = v4i{0, 0, 0, 0};

    float row_scale[TM];
    if constexpr (MODE == (int)Epilogue::RequantRow) {
#pragma unroll
        for (int j = 0; j < TM; j++) {
            const uint32_t m = min(m0 + (wave_m * TM + j) * 16 + (lane & 15), a.rows - 1u);
            row_scale[j] = a.row_scale[m];
        }
    }

    // ---- fragment addressing -----------------------------------------------------------
    // weights: tile i of the wave is half (i%2) of panel wave_n*TN/2 + i/2; MFMA step s of the stage
    // is the block pair (2s, 2s+1).  Lane l reads block 2s + l/32, slot 16*(i%2) + l%16 + 32*((l/16)%2).
    const uint32_t a_frag = (uint32_t)(wave_n * (TN / 2) * KS) * 1024u + (uint32_t)(lane >> 5) * 1024u +
                            (uint32_t)((lane & 15) + 32 * ((lane >> 4) & 1)) * 16u;
    // activations: row (wave_m*TM + j)*16 + l%16 of 128 bytes, chunk 4s + l/16 at slot chunk ^ (row%8)
    const uint32_t x_row = WBLK * 1024u + ((uint32_t)(wave_m * TM * 16) + (lane & 15)) * 128u;
    uint32_t x_slot[2];
#pragma unroll
    for (int s = 0; s < 2; s++) x_slot[s] = (((4u * s + (lane >> 4)) ^ (lane & 7u)) << 4);

    v4i af[TN], bf[2][TM];
    auto read_a = [&](auto i_tag, const char* stage, auto s_tag) {
        constexpr int i = decltype(i_tag)::value, s = decltype(s_tag)::value;
        af[i] = *reinterpret_cast<const v4i*>(stage + a_frag + ((i / 2) * KS + 2 * s) * 1024 + (i & 1) * 256);
    };
    auto read_b = [&](auto j_tag, const char* stage, auto s_tag) {
        constexpr int j = decltype(j_tag)::value, s = decltype(s_tag)::value;
        bf[s][j] = *reinterpret_cast<const v4i*>(stage + x_row + j * 16 * 128 + x_slot[s]);
    };

    // ---- main loop -------------------------------------------------------------------------
    // A k-block is two MFMA steps of TN rows of TM MFMAs (row i: channel tile i against every row
    // tile).  The weight fragment of a row is replaced as soon as the row has issued, by the same
    // row's fragment of the following step; the activation fragments are double buffered by step
    // parity.  Step 0 reads step 1's fragments from the same stage.  Step 1 runs its first RB rows,
    // then waits for its own LDS reads and its loads of the next k-block, passes the barrier,
    // and from there on reads the next stage's step 0 and refills the current stage for k-block
    // kb+2, every request placed behind a fixed MFMA so that LDS reads, global loads and MFMAs
    // issue evenly mixed.
    constexpr int RB = 1;
    static_assert(TN - RB >= TM && TN >= TM, "every activation fragment needs a row to be re-read behind");
    // both stages are requested at once: the second k-block's latency then runs beside the first's
    static_for<NLOADS>([&](auto t) { issue_one(t, 0u, 0); });
    static_for<NLOADS>([&](auto t) { issue_one(t, 1u, 1); });

    float* lds_f0 = reinterpret_cast<float*>(lds_raw + 2 * STAGE_BYTES);
    int32_t* lds_cb = reinterpret_cast<int32_t*>(lds_f0 + BN);
    float* lds_bo = reinterpret_cast<float*>(lds_cb + BN);
    int32_t* lds_zw = reinterpret_cast<int32_t*>(lds_bo + BN);
    for (int t = threadIdx.x; t < BN; t += NWAVES * 64) {
        const ChannelConsts c = channel_consts<MODE>(a, n0 + t);
        lds_f0[t] = c.f0;
        lds_cb[t] = c.cb;
        lds_bo[t] = c.bo;
        lds_zw[t] = c.zw;
    }

    auto mfma_row = [&](auto i_tag, auto s_tag, auto&& after) {
        constexpr int i = decltype(i_tag)::value, s = decltype(s_tag)::value;
        static_for<TM>([&](auto j_tag) {
            constexpr int j = decltype(j_tag)::value;
            if constexpr (FLIP && i == 0) bf[s][j] ^= (int)0x80808080u;
            acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[i], bf[s][j], acc[i][j], 0, 0, 0);
            after(j_tag);
            __builtin_amdgcn_sched_barrier(0);
        });
    };

    wait_vmcnt<0>();
    wg_barrier();
    static_for<TM>([&](auto j) { read_b(j, lds_raw, IC<0>{}); });
    static_for<TN>([&](auto i) { read_a(i, lds_raw, IC<0>{}); });

    auto k_block = [&](uint32_t kb, auto last_tag) {
        constexpr bool LAST = decltype(last_tag)::value;
        const int cur = kb & 1;
        const char* stage = lds_raw + cur * STAGE_BYTES;
        const char* next = lds_raw + (cur ^ 1) * STAGE_BYTES;
        // step 0: behind row i, the same row's weight fragment of step 1; the activation fragments of
        // step 1 go out behind the first MFMAs of rows 0 .. TM-1
        static_for<TN>([&](auto i_tag) {
            constexpr int i = decltype(i_tag)::value;
            mfma_row(i_tag, IC<0>{}, [&](auto j_tag) {
                constexpr int j = decltype(j_tag)::value;
                if constexpr (j == 0 && i < TM) read_b(IC<(i < TM ? i : 0)>{}, stage, IC<1>{});
                if constexpr (j == TM - 1) read_a(i_tag, stage, IC<1>{});
            });
        });
        if constexpr (LAST) {
            static_for<TN>([&](auto i_tag) { mfma_row(i_tag, IC<1>{}, [&](auto) {}); });
        } else {
            static_for<RB>([&](auto i_tag) { mfma_row(i_tag, IC<1>{}, [&](auto) {}); });
            wait_lgkm0();     // my reads of this stage have landed in registers
            wait_vmcnt<0>();  // my loads of the next k-block have landed
            wg_barrier();
            static_for<RB>([&](auto i_tag) { read_a(i_tag, next, IC<0>{}); });
            // (TN - RB) * TM MFMAs carry the NLOADS loads of k-block kb+2 and TM activation reads
            constexpr int REST = (TN - RB) * TM;
            static_for<TN - RB>([&](auto r_tag) {
                constexpr int i = RB + decltype(r_tag)::value;
                mfma_row(IC<i>{}, IC<1>{}, [&](auto j_tag) {
                    constexpr int j = decltype(j_tag)::value;
                    constexpr int m = (i - RB) * TM + j;
                    if constexpr (j == 0 && i - RB < TM) read_b(IC<(i - RB < TM ? i - RB : 0)>{}, next, IC<0>{});
                    if constexpr (j == TM - 1) read_a(IC<i>{}, next, IC<0>{});
                    static_for<NLOADS>([&](auto l_tag) {
                        constexpr int l = decltype(l_tag)::value;
                        if constexpr ((l * REST) / NLOADS == m) issue_one(l_tag, kb + 2u, cur);
                    });
                });
            });
        }
    };
    for (uint32_t kb = 0; kb + 1 < nkb; kb++) k_block(kb, std::false_type{});
    k_block(nkb - 1u, std::true_type{});
    wait_vmcnt<0>();  // nothing of this workgroup may still be writing LDS when the epilogue runs

    // ---- epilogue: requantize, pack, transpose across the four lane groups, 16-byte stores ----
    const float zp_f = (float)a.out_zp, lo_f = (float)a.out_lo, hi_f = (float)a.out_hi;
    const float so = a.output_scale, sr = a.output_scale_recip;
    [[maybe_unused]] const float dq_zp_f = (float)a.dq_zp;
    uint32_t mrow[TM];
    int32_t rsum[TM];
    uint32_t miss1 = 1, miss2 = 1;
    if (MODE == (int)Epilogue::RequantRow && a.div_proof) {
        miss1 = a.div_proof[0];
        miss2 = a.div_proof[1];
    }
    bool lean = a.zw == nullptr;
    if constexpr (MODE == (int)Epilogue::RequantRow) lean = lean && fast_div_in_range(so) && miss2 == 0;
    const bool no_int_terms = a.int_bias_zero && (MODE == (int)Epilogue::RequantRow || a.input_zp == 0);
    const bool bare_ok = no_int_terms && a.out_zp == 0 && (MODE != (int)Epilogue::RequantRow || miss1 == 0);
    bool bad = false;
#pragma unroll
    for (int j = 0; j < TM; j++) {
        mrow[j] = m0 + (wave_m * TM + j) * 16 + (lane & 15);
        rsum[j] = (a.zw && mrow[j] < a.rows) ? a.rowsum[mrow[j]] : 0;
        if constexpr (MODE == (int)Epilogue::RequantRow) {
            const float plo = __fmul_rn(row_scale[j], a.wscale_min), phi = __fmul_rn(row_scale[j], a.wscale_max);
            if (mrow[j] < a.rows) {
                bad |= !scale_valid(__fdiv_rn(plo, so)) || !scale_valid(__fdiv_rn(phi, so));
                lean &= fast_div_in_range(plo) && fast_div_in_range(phi);
            }
        }
    }
    if (bad) atomicOr(a.fault, (uint32_t)kFaultBadMultiplier);
    const bool wave_lean = __builtin_amdgcn_ballot_w64(!lean) == 0ull;
    // LEVEL 0: general.  1: no weight zero points, every quotient in the range of the proved short
    // division.  2: in addition nothing to add to the accumulator or the product (gemm_mfma.hip).
    auto run = [&](auto level_tag, auto streamed_tag) {
        constexpr int LEVEL = decltype(level_tag)::value;
        constexpr bool STREAMED = decltype(streamed_tag)::value;
        constexpr bool LEAN = LEVEL >= 1, BARE = LEVEL == 2;
#pragma unroll
        for (int h = 0; h < TN / 4; h++) {
            v4f f0[4], bo[4];
            v4i cb[4], zw[4];
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const int c0 = (wave_n * TN + h * 4 + t) * 16 + (lane >> 4) * 4;
                f0[t] = *reinterpret_cast<const v4f*>(lds_f0 + c0);
                cb[t] = *reinterpret_cast<const v4i*>(lds_cb + c0);
                bo[t] = v4f{0.f, 0.f, 0.f, 0.f};
                zw[t] = v4i{0, 0, 0, 0};
                if (MODE == (int)Epilogue::RequantRow && (BARE || a.bias_row)) bo[t] = *reinterpret_cast<const v4f*>(lds_bo + c0);
                if (!LEAN && a.zw) zw[t] = *reinterpret_cast<const v4i*>(lds_zw + c0);
            }
#pragma unroll
            for (int j = 0; j < TM; j++) {
                uint32_t pk[4];
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    uint32_t u[4];
                    v4f dq;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        uint32_t total = (uint32_t)acc[h * 4 + t][j][e];
                        if (!BARE) total += (uint32_t)cb[t][e];
                        if (!LEAN) total -= (uint32_t)zw[t][e] * (uint32_t)rsum[j];
                        float mu = f0[t][e];
                        if constexpr (MODE == (int)Epilogue::RequantRow) {
                            const float prod = __fmul_rn(row_scale[j], f0[t][e]);
                            mu = BARE   ? div_by_uniform_once(prod, so, sr)
                                 : LEAN ? div_by_uniform(prod, so, sr)
                                        : __fdiv_rn(prod, so);
                        }
                        float v = __fmul_rn((float)(int32_t)total, mu);
                        if (!BARE) v = __fadd_rn(v, zp_f);
                        if (MODE == (int)Epilogue::RequantRow && (BARE || a.bias_row)) v = __fadd_rn(v, bo[t][e]);
                        // clamp, then ties-to-even by adding 1.5 * 2^23: the low mantissa bits are the integer
                        v = __builtin_amdgcn_fmed3f(v, lo_f, hi_f);
                        const float rounded = __fadd_rn(v, 12582912.0f);
                        u[e] = __float_as_uint(rounded);
                        if constexpr (DQ) {
                            // the byte's value as a float (exact), then the DequantizeLinear's one rounding
                            const float qf = __fsub_rn(rounded, 12582912.0f);
                            dq[e] = __fmul_rn(__fsub_rn(qf, dq_zp_f), a.dq_scale);
                        }
                    }
                    if constexpr (DQ) {
                        const uint32_t nq = n0 + (wave_n * TN + h * 4 + t) * 16 + (lane >> 4) * 4;
                        if (mrow[j] < a.rows && nq < a.n) *reinterpret_cast<v4f*>(a.dq_out + (size_t)mrow[j] * a.n + nq) = dq;
                    }
                    const uint32_t p01 = __builtin_amdgcn_perm(u[1], u[0], 0x0c0c0400u);
                    const uint32_t p23 = __builtin_amdgcn_perm(u[3], u[2], 0x0c0c0400u);
                    pk[t] = __builtin_amdgcn_perm(p23, p01, 0x05040100u);
                }
                // pk[t] in lane group g = channels 4g..4g+3 of tile t.  Transpose the 4 x 4 of (tile, lane
                // group): afterwards lane group g holds the four dwords of tile g, 16 consecutive bytes.
                const auto s02 = __builtin_amdgcn_permlane32_swap(pk[0], pk[2], false, false);
                const auto s13 = __builtin_amdgcn_permlane32_swap(pk[1], pk[3], false, false);
                const auto r01 = __builtin_amdgcn_permlane16_swap(s02[0], s13[0], false, false);
                const auto r23 = __builtin_amdgcn_permlane16_swap(s02[1], s13[1], false, false);
                const uint32_t n16 = n0 + (wave_n * TN + h * 4 + (lane >> 4)) * 16;
                if ((!DQ || a.y) && mrow[j] < a.rows && n16 < a.n) {
                    const v4i v = v4i{(int)r01[0], (int)r01[1], (int)r23[0], (int)r23[1]};
                    store_stream<STREAMED>(reinterpret_cast<v4i*>((uint8_t*)a.y + (size_t)mrow[j] * a.n + n16), v);
                }
            }
        }
    };
    // (the two straight-line levels come in a streamed copy as well; the general one stores plainly)
    const bool streamed = !DQ && a.stream_out != 0u;  // (the dequantizing form's f32 stores are never streamed)
    if (wave_lean && bare_ok) {
        if (streamed) run(IC<2>{}, std::true_type{});
        else run(IC<2>{}, std::false_type{});
    } else if (wave_lean) {
        if (streamed) run(IC<1>{}, std::true_type{});
        else run(IC<1>{}, std::false_type{});
    } else {
        run(IC<0>{}, std::false_type{});
    }
}

// eight codes' low nibbles (two's complement) as four signed bytes, every second one: ((v ^ 8) - 8) without a
// borrow between the bytes
__device__ __forceinline__ uint32_t signed_nibbles(uint32_t v) {
    return (((v & 0x0f0f0f0fu) ^ 0x08080808u) + 0x78787878u) ^ 0x80808080u;
}

// ---- the dequantizing form (PackedLinear under DYNAMIC_I8) ----------------------------------------
// sum += f32(dot_g) * (s_a * s_w[n][g]) in ascending group order with every product and sum rounded
// on its own (packed_linear_ops.inc:1498-1504): four VALU operations per output and group against
// 2 * group_size matrix operations, so the kernel is bound by the vector pipe, not by the MFMAs.
// It therefore runs small wave tiles (16 x TN channels x 16 x TM rows, at most 64 x 32) at four waves per
// SIMD and leaves the overlap of one wave's fold with the other waves' MFMAs to the hardware: two workgroups
// of 128 x 128 per compute unit, each with its own barrier, or more of the narrow tiles that put a small
// launch on every SIMD (see pick_f32_tile).  GK: 64-wide MFMA steps per scale group (1, 2 or 4; 0: two groups
// of 32 per step, on 16x16x32 MFMAs, which take the same cycles).  W4: four-bit weights; a 1 KiB block then holds the block pair of one MFMA step, low
// nibbles for its first 32 k, high nibbles for the rest, and a lane shifts its half into place.
// The scales of the groups that end in a k-block travel as the tail of that k-block's LDS stage.
// UNI: every channel has one scale for all its groups (a per-channel scale replicated, which is what
// per-channel quantization exports); s_a * s_w is then formed once per output instead of once per
// output and group -- the same products, so the same bits -- and the fold is three operations.
//
// AFTER (a decoder's prompt): the workgroup goes on with its outputs instead of storing them for another launch to read.
// Rope and Swiglu combine channels in pairs, d and d + half a head, or gate and up.  So that both of a pair are in the
// same lane and element, a tile of BN channels is BN / 2 first ones and their BN / 2 second ones, each from panels of
// their own (`panel_of`), and of a wavefront's TN channel tiles half are firsts and half the seconds of those.
// 32 prompts of 128 tokens, a layer of hidden 1024 (q/k/v 4096 channels, gate/up 6144), traced: the four linears, rotary, and
// row operations 250 us as launches of their own (167, 24, 59), 203 so (52 with rotary and append, 55 with SwiGLU, 2 x 29 with
// the residual add, 37 of row operations).
template <int GK, bool W4, int WN, int WM, int TN, int TM, int NS, bool UNI, After AFTER>
__device__ __forceinline__ void gemm_f32_body(const GemmParams& p, const LinearTail& tail) {
    constexpr bool PAIRS = AFTER == After::Rope || AFTER == After::Swiglu;
    static_assert(!PAIRS || TN % 2 == 0, "as many first as second tiles");
    constexpr int F = PAIRS ? TN / 2 : TN;  // first tiles of a wavefront
    constexpr int NWAVES = WN * WM;
    constexpr int BN = WN * TN * 16, BM = WM * TM * 16;
    constexpr int KS = 4, KB = W4 ? 2 : 4;  // 32-byte k-steps and 1 KiB weight blocks per panel and stage
    static_assert(BN % 32 == 0 && BM % 8 == 0 && (TN == 1 || TN % 2 == 0), "whole panels, whole loads");
    constexpr int WBLK = (BN / 32) * KB, XBLK = BM / 8;
    constexpr int GPB = GK == 0 ? 4 : GK == 1 ? 2 : 1;  // scale groups that end in a k-block (GK == 4: every second block)
    constexpr int SBLK = UNI ? 0 : (GPB * BN + 63) / 64;  // loads of 64 scales
    constexpr int WLOADS = (WBLK + NWAVES - 1) / NWAVES, XLOADS = (XBLK + NWAVES - 1) / NWAVES;
    // Wide wave tiles: the first SBLK waves load 64 scales each (and wait for one load more than they must), since a
    // repeated load for the others costs more than that: 619 x 9500 -> 9861 in groups of 128 121.9 -> 119.1 us (none to
    // see in groups of 64 and 256).
    constexpr bool SOME_LOAD_SCALES = TN * TM > 4 && SBLK <= NWAVES;
    constexpr int SLOADS = SOME_LOAD_SCALES ? 0 : (SBLK + NWAVES - 1) / NWAVES;
    constexpr int SCALE_OFF = (WBLK + XBLK) * 1024;
    constexpr int STAGE_BYTES = SCALE_OFF + SBLK * 256;
    constexpr int NLOADS = WLOADS + XLOADS + SLOADS;
    const LinearArgs& a = p.a;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int wave_n = wave % WN, wave_m = wave / WN;
    uint32_t m0, n0;
    {
        const TileOrigin t = tile_of_workgroup<BN, BM, 8>(p);
        if (!t.valid) return;
        m0 = t.m0;
        n0 = t.n0;
    }

    // pair panel q: 32 first channels and the 32 second ones behind them, of a head or of the two halves of the row
    const uint32_t pair_panels = PAIRS ? a.n / 64u : 0u, halves = AFTER == After::Rope ? tail.head_dim / 64u : 1u;
    auto pair_panel = [&](uint32_t q, bool second) {
        if constexpr (AFTER == After::Rope) return q / halves * 2u * halves + q % halves + (second ? halves : 0u);
        else return q + (second ? pair_panels : 0u);
    };
    // panel `b` of the tile
    auto panel_of = [&](uint32_t b) {
        if constexpr (PAIRS) {
            constexpr uint32_t P = BN / 64;
            return pair_panel(min(n0 / 64u + b % P, pair_panels - 1u), b >= P);
        } else {
            return n0 / 32u + b;
        }
    };

    const uint32_t w_lane = lane * 16u;
    const uint32_t panel_bytes = a.ksteps * 1024u;
    const uint32_t last_chunk = (a.k - 1u) / 16u;
    const uint32_t my_chunk = (lane & 7) ^ ((lane >> 3) & 7);
    // (a wave without a block of its own in the last round of loads repeats another's: the same bytes to the
    // same place, and every wave has the same number of loads in flight)
    uint32_t xrow[XLOADS];
#pragma unroll
    for (int i = 0; i < XLOADS; i++) {
        const int b = (wave + i * NWAVES) % XBLK;
        uint32_t row = m0 + b * 8 + (lane >> 3);
        row = min(row, a.rows - 1u);
        xrow[i] = row * a.ldx;
    }
    const uint32_t ksteps_real = (a.k + 31u) / 32u;
    const uint32_t nkb = (ksteps_real + KS - 1) / KS;
    auto issue_block = [&](uint32_t kb, int stage) {
        char* base = lds_raw + stage * STAGE_BYTES;
        // the scales of the groups that end in this k-block, [group][channel]: 4 bytes per lane
        auto scales = [&](uint32_t b) {
            const uint32_t e = b * 64u + lane, slot = e / BN;
            const uint32_t g = GK == 0 ? kb * 4u + slot : GK == 1 ? kb * 2u + slot : GK == 2 ? kb : kb / 2u;
            const uint32_t n = PAIRS ? panel_of(e % BN / 32u) * 32u + e % 32u : n0 + e % BN;
            load_to_lds4(a.scales_t + (size_t)min(g, a.groups - 1u) * a.n_pad + n, base + SCALE_OFF + b * 256);
        };
        if constexpr (SOME_LOAD_SCALES) {
            if (wave < SBLK) scales(wave);
        }
        static_for<NLOADS>([&](auto t_tag) {
            constexpr int t = decltype(t_tag)::value;
            if constexpr (t < SLOADS) {
                scales((wave + t * NWAVES) % (SBLK > 0 ? SBLK : 1));
            } else if constexpr (t < SLOADS + WLOADS) {
                const uint32_t b = (wave + (t - SLOADS) * NWAVES) % WBLK;
                const int8_t* src = a.w + (size_t)panel_of(b / KB) * panel_bytes + (size_t)(kb * KB + b % KB) * 1024u;
                load_to_lds16(src + w_lane, base + b * 1024);
            } else {
                constexpr int i = t - SLOADS - WLOADS;
                const uint32_t chunk16 = min(kb * 8u + my_chunk, last_chunk) * 16u;
                const uint32_t b = (wave + i * NWAVES) % XBLK;
                load_to_lds16(a.x + (xrow[i] + chunk16), base + (WBLK + b) * 1024);
            }
        });
    };

    v4i acc[TN][TM];
    v4f fsum[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; i++)
#pragma unroll
        for (int j = 0; j < TM; j++) {
            acc[i][j] = v4i{0, 0, 0, 0};
            fsum[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
        }
    float row_scale[TM];
#pragma unroll
    for (int j = 0; j < TM; j++) {
        const uint32_t m = min(m0 + (wave_m * TM + j) * 16 + (lane & 15), a.rows - 1u);
        row_scale[j] = a.row_scale[m];
    }

    // fragment addressing (see the requantizing kernel); four-bit weights: one block per MFMA step,
    // the lane's 16-byte slot is the same for both halves of the step
    const uint32_t tile0 = (uint32_t)wave_n * F;  // the wave's first 16 channels
    // channel tile i of the wave, from there: its 16 channels, and its bytes of a stage
    constexpr auto tile_channels = [](int i) { return PAIRS ? i % F * 16 + i / F * (BN / 2) : i * 16; };
    constexpr auto tile_bytes = [](int i, int step) {
        return PAIRS ? (i / F * (BN / 64) * KB + step) * 1024 + i % F * 256 : (i / 2 * KB + step) * 1024 + (i & 1) * 256;
    };
    const uint32_t a_tile = (tile0 / 2u) * KB * 1024u + (tile0 & 1u) * 256u;
    // (groups of 32: the MFMA takes eight bytes a lane, of one k-step)
    const uint32_t a_frag = GK == 0 ? a_tile + (uint32_t)((lane & 15) + 32 * (lane >> 5)) * 16u + ((lane >> 4) & 1) * 8u
                            : W4    ? a_tile + (uint32_t)((lane & 15) + 32 * ((lane >> 4) & 1)) * 16u
                                    : a_tile + (uint32_t)(lane >> 5) * 1024u + (uint32_t)((lane & 15) + 32 * ((lane >> 4) & 1)) * 16u;
    const uint32_t nib_shift = lane < 32 ? 4u : 0u;
    const uint32_t x_row = WBLK * 1024u + ((uint32_t)(wave_m * TM * 16) + (lane & 15)) * 128u;
    uint32_t x_slot[GK == 0 ? KS : 2];
    if constexpr (GK == 0) {
#pragma unroll
        for (int s = 0; s < KS; s++) x_slot[s] = (((2u * s + (lane >> 5)) ^ (lane & 7u)) << 4) + ((lane >> 4) & 1) * 8u;
    } else {
#pragma unroll
        for (int s = 0; s < 2; s++) x_slot[s] = (((4u * s + (lane >> 4)) ^ (lane & 7u)) << 4);
    }
    const uint32_t sw_lane = SCALE_OFF + (uint32_t)(wave_n * F * 16 + (lane >> 4) * 4) * 4u;
    // the four channels of tile i that the lane has, as the weights count them
    auto channels_of = [&](int i) {
        if constexpr (PAIRS) {
            const uint32_t at = (wave_n * F + i % F) * 16u;
            return panel_of(at / 32u + i / F * (BN / 64)) * 32u + at % 32u + (lane >> 4) * 4u;
        } else {
            return n0 + (wave_n * TN + i) * 16 + (lane >> 4) * 4;
        }
    };

    // UNI: the products s_a * s_w of the lane's outputs
    float gs_all[UNI ? TN : 1][UNI ? TM : 1][4];
    if constexpr (UNI) {
#pragma unroll
        for (int i = 0; i < TN; i++) {
            const v4f sw = *reinterpret_cast<const v4f*>(a.scales_t + channels_of(i));
#pragma unroll
            for (int j = 0; j < TM; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) gs_all[i][j][e] = __fmul_rn(row_scale[j], sw[e]);
        }
    }
    // fold of scale-group slot `slot` of the stage: every tile of the wave
    constexpr int DOT_SHIFT = W4 && GK != 0 ? 4 : 0;
    auto group_scales = [&](const char* stage, int slot, int i) {
        v4f sw = {0.f, 0.f, 0.f, 0.f};
        if constexpr (!UNI) sw = *reinterpret_cast<const v4f*>(stage + sw_lane + (slot * BN + tile_channels(i)) * 4);
        return sw;
    };
    auto fold_by = [&](auto&& scales_of) {
#pragma unroll
        for (int i = 0; i < TN; i++) {
            const v4f sw = scales_of(i);
#pragma unroll
            for (int j = 0; j < TM; j++) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float gs = UNI ? gs_all[UNI ? i : 0][UNI ? j : 0][e] : __fmul_rn(row_scale[j], sw[e]);
                    // four-bit operands carry a factor 16; the dot is exact, so is the shift
                    const float term = __fmul_rn((float)(acc[i][j][e] >> DOT_SHIFT), gs);
                    fsum[i][j][e] = __fadd_rn(fsum[i][j][e], term);
                }
            }
        }
    };
    auto fold = [&](const char* stage, int slot) { fold_by([&](int i) { return group_scales(stage, slot, i); }); };

    // NS stages: k-blocks kb+1 .. kb+NS-1 are in flight while k-block kb is consumed.  One barrier per
    // k-block, at its top: behind it every wave's loads of the block have landed and every wave is done
    // with the previous block, whose stage is refilled at once.  (Blocks past the end are clamped to the
    // last one, so the count of loads in flight is the same in every iteration.)
    static_for<NS - 1>([&](auto b_tag) { issue_block(min((uint32_t)decltype(b_tag)::value, nkb - 1u), decltype(b_tag)::value); });
    int cur = 0, refill = NS - 1;
    const v4i zero = {0, 0, 0, 0};
    auto k_block = [&](uint32_t kb, auto ends_tag, auto odd_tag) {
        constexpr bool ENDS = decltype(ends_tag)::value;  // may be the last k-block, with fewer groups
        constexpr bool ODD = decltype(odd_tag)::value;    // GK == 4: the second half of a group
        wait_vmcnt<(NS - 2) * NLOADS>();
        wg_barrier();
        issue_block(min(kb + NS - 1u, nkb - 1u), refill);
        const char* stage = lds_raw + cur * STAGE_BYTES;
        if constexpr (GK == 0) {
            // a group per k-step of 32.  Four-bit weights are spread to signed bytes here, which the many outputs
            // of a group are cheaper for than a shift each.  On the 64x64 tile, of which a SIMD has two wavefronts at most, a
            // step's operands and scales are read while the step before is multiplied and folded: 333 x 3000 -> 5001
            // with them read as they were needed | so: 8 bits 36.4 | 34.7 us, 4 bits 37.8 | 37.2.  What is left is issue:
            // some 350 vector instructions a k-block and wavefront, 256 of them the fold.  (Groups of 64 and more, whose
            // steps are longer, gained nothing from it: 0.98 to 1.02.)
            long bf[2][TM], raw[2][TN];
            v4f sw[2][TN];
            auto read = [&](int s) {
#pragma unroll
                for (int j = 0; j < TM; j++) bf[s & 1][j] = *reinterpret_cast<const long*>(stage + x_row + j * 16 * 128 + x_slot[s]);
#pragma unroll
                for (int i = 0; i < TN; i++) raw[s & 1][i] = *reinterpret_cast<const long*>(stage + a_frag + tile_bytes(i, W4 ? s / 2 : s));
#pragma unroll
                for (int i = 0; i < TN; i++) sw[s & 1][i] = group_scales(stage, s, i);
            };
            constexpr bool BEFORE = TN * TM == 4;
            if constexpr (BEFORE) read(0);
#pragma unroll
            for (int s = 0; s < KS; s++) {
                if constexpr (BEFORE) {
                    if (s + 1 < KS) read(s + 1);
                    __builtin_amdgcn_sched_barrier(0);
                } else {
                    read(s);
                }
                long af[TN];
#pragma unroll
                for (int i = 0; i < TN; i++) {
                    if constexpr (W4) {
                        const uint32_t lo = signed_nibbles((uint32_t)raw[s & 1][i] >> (s & 1) * 4);
                        const uint32_t hi = signed_nibbles((uint32_t)((uint64_t)raw[s & 1][i] >> 32) >> (s & 1) * 4);
                        af[i] = (long)(((uint64_t)hi << 32) | lo);
                    } else {
                        af[i] = raw[s & 1][i];
                    }
                }
#pragma unroll
                for (int i = 0; i < TN; i++)
#pragma unroll
                    for (int j = 0; j < TM; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x32_i8(af[i], bf[s & 1][j], zero, 0, 0, 0);
                if (!ENDS || kb * 4u + s < a.groups) fold_by([&](int i) { return sw[s & 1][i]; });
            }
        } else {
#pragma unroll
            for (int s = 0; s < 2; s++) {
                v4i af[TN], bf[TM];
#pragma unroll
                for (int j = 0; j < TM; j++) bf[j] = *reinterpret_cast<const v4i*>(stage + x_row + j * 16 * 128 + x_slot[s]);
#pragma unroll
                for (int i = 0; i < TN; i++) {
                    if constexpr (W4) {
                        const v4i raw = *reinterpret_cast<const v4i*>(stage + a_frag + tile_bytes(i, s));
#pragma unroll
                        for (int d = 0; d < 4; d++) af[i][d] = (raw[d] << nib_shift) & (int)0xf0f0f0f0u;
                    } else {
                        af[i] = *reinterpret_cast<const v4i*>(stage + a_frag + tile_bytes(i, 2 * s));
                    }
                }
                // first MFMA step of a scale group: accumulate onto zero instead of clearing registers
                const bool fresh = GK == 1 || (GK == 2 && s == 0) || (GK == 4 && s == 0 && !ODD);
#pragma unroll
                for (int i = 0; i < TN; i++)
#pragma unroll
                    for (int j = 0; j < TM; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[i], bf[j], fresh ? zero : acc[i][j], 0, 0, 0);
                // last MFMA step of a scale group (or of the row): fold it.  A group that starts past the
                // end of k does not exist (its dot would be zero, but adding +0.0 can flip a -0.0 sum).
                if constexpr (GK == 1) {
                    if (!ENDS || kb * 2u + s < a.groups) fold(stage, s);
                } else if constexpr (GK == 2) {
                    if (s == 1) fold(stage, 0);
                } else {
                    if (s == 1 && (ODD || ENDS)) fold(stage, 0);
                }
            }
        }
        refill = cur;
        cur = cur + 1 == NS ? 0 : cur + 1;
    };
    // (narrow wave tiles take the last k-block by itself, so that nothing in the others is conditional; the wide
    // ones would spill.  Groups of 256 take two k-blocks a round: with the half of the group as a condition of the loop
    // 995 x 4224 -> 3168 takes 45.0 us, so 37.8; 1137 x 6912 -> 2752 65.9 and 55.0.)
    constexpr bool PEEL = TN * TM <= 4;
    uint32_t kb = 0;
    if constexpr (GK == 4) {
        for (; kb + 1u < nkb; kb += 2u) {
            k_block(kb, std::false_type{}, std::false_type{});
            k_block(kb + 1u, std::false_type{}, std::true_type{});
        }
        if (kb < nkb) k_block(kb, std::true_type{}, std::false_type{});
    } else {
        if constexpr (PEEL) {
            for (; kb + 1u < nkb; kb++) k_block(kb, std::false_type{}, std::false_type{});
        }
        for (; kb < nkb; kb++) k_block(kb, std::true_type{}, std::false_type{});
    }
    wait_vmcnt<0>();

    // ---- epilogue: + bias, 16-byte stores (a lane owns row l%16 and four consecutive channels) ----
    // (streamed stores, as in the requantizing kernel, were measured here too: config 5's 32 MiB of f32 output
    // 0.7 % faster, the second copy of the epilogue 1.3 % slower where it is not used; left out)
    if constexpr (PAIRS) {
#pragma unroll
        for (int j = 0; j < TM; j++) {
            const uint32_t m = m0 + (wave_m * TM + j) * 16 + (lane & 15);
            if (m >= a.rows) continue;
            uint32_t slot = 0u, sequence = 0u;
            if constexpr (AFTER == After::Rope) {
                sequence = m / tail.t;
                const uint64_t named = (uint64_t)tail.positions[m - sequence * tail.t];
                if (named >= tail.max_seq) {  // outside the caches and the tables: touch nothing, say so
                    atomicOr(a.fault, (uint32_t)kFaultBadPosition);
                    continue;
                }
                slot = (uint32_t)named;
            }
#pragma unroll
            for (int i = 0; i < F; i++) {
                const uint32_t at = (wave_n * F + i) * 16u, q = n0 / 64u + at / 32u;
                if (q >= pair_panels) continue;
                const uint32_t n = channels_of(i), mate = channels_of(i + F);
                const v4f b_lo = *reinterpret_cast<const v4f*>(a.bias_f32 + n), b_hi = *reinterpret_cast<const v4f*>(a.bias_f32 + mate);
                v4f lo, hi;
#pragma unroll
                for (int e = 0; e < 4; e++) lo[e] = __fadd_rn(fsum[i][j][e], b_lo[e]), hi[e] = __fadd_rn(fsum[i + F][j][e], b_hi[e]);
                if constexpr (AFTER == After::Swiglu) {
                    v4f out;
#pragma unroll
                    for (int e = 0; e < 4; e++) out[e] = swiglu_value(lo[e], hi[e]);
                    *reinterpret_cast<v4f*>((float*)a.y + (size_t)m * (a.n / 2u) + n) = out;
                } else {
                    const uint32_t hd = tail.head_dim, half = hd / 2u, head = n / hd, dd = n % hd;
                    if (head < tail.q_heads + tail.kv_heads) {
                        const float* c = tail.cos_table + (size_t)slot * hd + dd;
                        const float* sn = tail.sin_table + (size_t)slot * hd + dd;
                        const v4f c_lo = *reinterpret_cast<const v4f*>(c), c_hi = *reinterpret_cast<const v4f*>(c + half);
                        const v4f s_lo = *reinterpret_cast<const v4f*>(sn), s_hi = *reinterpret_cast<const v4f*>(sn + half);
#pragma unroll
                        for (int e = 0; e < 4; e++) {  // the arithmetic of rope_append_kernel
                            const float l = lo[e], h = hi[e];
                            lo[e] = __fadd_rn(__fmul_rn(l, c_lo[e]), __fmul_rn(-h, s_lo[e]));
                            hi[e] = __fadd_rn(__fmul_rn(h, c_hi[e]), __fmul_rn(l, s_hi[e]));
                        }
                    }
                    const uint32_t kv = head - tail.q_heads;  // (of a key or value head)
                    float* dst = head < tail.q_heads ? tail.q_out + ((size_t)m * tail.q_heads + head) * hd
                                 : kv < tail.kv_heads
                                     ? tail.k_cache + (((size_t)sequence * tail.kv_heads + kv) * tail.max_seq + slot) * hd
                                     : tail.v_cache + (((size_t)sequence * tail.kv_heads + kv - tail.kv_heads) * tail.max_seq + slot) * hd;
                    *reinterpret_cast<v4f*>(dst + dd) = lo;
                    *reinterpret_cast<v4f*>(dst + dd + half) = hi;
                }
            }
        }
        return;
    }
    const bool vec_ok = (a.n % 4u) == 0u;
#pragma unroll
    for (int j = 0; j < TM; j++) {
        const uint32_t m = m0 + (wave_m * TM + j) * 16 + (lane & 15);
        if (m >= a.rows) continue;
#pragma unroll
        for (int i = 0; i < TN; i++) {
            const uint32_t n = n0 + (wave_n * TN + i) * 16 + (lane >> 4) * 4;
            if (n >= a.n) continue;
            const v4f b = *reinterpret_cast<const v4f*>(a.bias_f32 + n);
            v4f out;
#pragma unroll
            for (int e = 0; e < 4; e++) out[e] = __fadd_rn(fsum[i][j][e], b[e]);
            float* y = (float*)a.y + (size_t)m * a.n + n;
            if constexpr (AFTER == After::Add) {  // (whole groups of four channels)
                const v4f r = *reinterpret_cast<const v4f*>(y);
#pragma unroll
                for (int e = 0; e < 4; e++) out[e] = __fadd_rn(r[e], out[e]);
            }
            if (vec_ok) {
                *reinterpret_cast<v4f*>(y) = out;
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (n + e < a.n) y[e] = out[e];
            }
        }
    }
}

template <int GK, bool W4, int WN, int WM, int TN, int TM, int NS, bool UNI>
__global__ __launch_bounds__(WN * WM * 64, 4) void gemm_k64_f32_kernel(const GemmParams p) {
    gemm_f32_body<GK, W4, WN, WM, TN, TM, NS, UNI, After::Store>(p, LinearTail{});
}
template <After AFTER, int GK, int WN, int WM, int TN, int TM, int NS, bool UNI>
__global__ __launch_bounds__(WN * WM * 64, 4) void gemm_k64_followed_kernel(const FollowedParams p) {
    gemm_f32_body<GK, false, WN, WM, TN, TM, NS, UNI, AFTER>(p.g, p.tail);
}

template <int GK, bool W4, int WN, int WM, int TN, int TM, int NS, bool UNI>
bool launch_f32_as(hipStream_t s, const LinearArgs& a) {
    constexpr int BN = WN * TN * 16, BM = WM * TM * 16, GPB = GK == 0 ? 4 : GK == 1 ? 2 : 1;
    constexpr int LDS = NS * (((BN / 32) * (W4 ? 2 : 4) + BM / 8) * 1024 + (UNI ? 0 : (GPB * BN + 63) / 64 * 256));
    static_assert(LDS <= 160 * 1024, "stages do not fit the LDS");
    static std::atomic<uint64_t> configured{0};
    auto kern = gemm_k64_f32_kernel<GK, W4, WN, WM, TN, TM, NS, UNI>;
    if (!raise_lds_limit((const void*)kern, LDS, configured)) return false;
    GemmParams p;
    p.a = a;
    p.tiles_n = (a.n + BN - 1) / BN;
    p.tiles_m = (a.rows + BM - 1) / BM;
    const uint32_t total = p.tiles_n * p.tiles_m;
    const uint32_t grid = ((total + 7u) / 8u) * 8u;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(WN * WM * 64), LDS, s, p);
    return hipGetLastError() == hipSuccess;
}

template <int GK, bool W4, int WN, int WM, int TN, int TM, int NS>
bool launch_f32(hipStream_t s, const LinearArgs& a) {
    // (the instances listed keep the products in registers without spilling at four waves per SIMD;
    // the others would lose more to scratch traffic than the fourth operation costs)
    constexpr bool kUniformFits = TN * TM <= 4 || GK == 1 || (GK == 2 && (W4 || WM == 8));
    if constexpr (kUniformFits) {
        if (a.uniform_group_scales) return launch_f32_as<GK, W4, WN, WM, TN, TM, NS, true>(s, a);
    }
    return launch_f32_as<GK, W4, WN, WM, TN, TM, NS, false>(s, a);
}

template <bool W4, int WN, int WM, int TN, int TM, int NS>
bool launch_f32_group(hipStream_t s, const LinearArgs& a) {
    switch (a.group_size) {
        case 32:
            // (only narrow wave tiles: the wide ones have no registers left)
            if constexpr (TN * TM <= 4) return launch_f32<0, W4, WN, WM, TN, TM, NS>(s, a);
            else return false;
        case 64: return launch_f32<1, W4, WN, WM, TN, TM, NS>(s, a);
        case 128: return launch_f32<2, W4, WN, WM, TN, TM, NS>(s, a);
        case 256: return launch_f32<4, W4, WN, WM, TN, TM, NS>(s, a);
        default: return false;
    }
}

template <int WN, int WM, int TN, int TM, int NS>
bool launch_f32_bits(hipStream_t s, const LinearArgs& a) {
    return a.weight_bits == 4u ? launch_f32_group<true, WN, WM, TN, TM, NS>(s, a)
                               : launch_f32_group<false, WN, WM, TN, TM, NS>(s, a);
}

template <int WN, int WM, int TN, int TM, int MODE, bool FLIP = false, bool DQ = false>
bool launch_one(hipStream_t s, const LinearArgs& a) {
    constexpr int BN = WN * TN * 16, BM = WM * TM * 16;
    constexpr int LDS = 2 * ((BN / 32) * 4 + BM / 8) * 1024 + BN * 16;
    static_assert(LDS <= 160 * 1024, "stages do not fit the LDS");
    static std::atomic<uint64_t> configured{0};
    auto kern = gemm_k64_kernel<WN, WM, TN, TM, MODE, FLIP, DQ>;
    if (!raise_lds_limit((const void*)kern, LDS, configured)) return false;
    GemmParams p;
    p.a = a;
    p.a.stream_out = (size_t)a.rows * a.n >= (12u << 20) ? 1u : 0u;  // (see store_stream: the byte output only)
    p.tiles_n = (a.n + BN - 1) / BN;
    p.tiles_m = (a.rows + BM - 1) / BM;
    const uint32_t total = p.tiles_n * p.tiles_m;
    const uint32_t grid = ((total + 7u) / 8u) * 8u;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(WN * WM * 64), LDS, s, p);
    return hipGetLastError() == hipSuccess;
}

}  // namespace

namespace {

template <After AFTER, int GK, int WN, int WM, int TN, int TM, int NS, bool UNI>
bool launch_followed_as(hipStream_t s, const LinearArgs& a, const LinearTail& tail) {
    constexpr int BN = WN * TN * 16, BM = WM * TM * 16, GPB = GK == 1 ? 2 : 1;
    constexpr int LDS = NS * (((BN / 32) * 4 + BM / 8) * 1024 + (UNI ? 0 : (GPB * BN + 63) / 64 * 256));
    static_assert(LDS <= 160 * 1024, "stages do not fit the LDS");
    static std::atomic<uint64_t> configured{0};
    auto kern = gemm_k64_followed_kernel<AFTER, GK, WN, WM, TN, TM, NS, UNI>;
    if (!raise_lds_limit((const void*)kern, LDS, configured)) return false;
    FollowedParams p;
    p.g.a = a;
    p.g.tiles_n = (a.n + BN - 1) / BN;
    p.g.tiles_m = (a.rows + BM - 1) / BM;
    p.tail = tail;
    const uint32_t grid = (p.g.tiles_n * p.g.tiles_m + 7u) / 8u * 8u;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(WN * WM * 64), LDS, s, p);
    return hipGetLastError() == hipSuccess;
}
template <After AFTER, int GK>
bool launch_followed_tile(hipStream_t s, const LinearArgs& a, const LinearTail& tail, bool wide) {
    if (wide) {
        if constexpr (GK == 1) {  // (where the products s_a * s_w fit the registers: launch_f32)
            if (a.uniform_group_scales) return launch_followed_as<AFTER, GK, 2, 4, 4, 2, 2, true>(s, a, tail);
        }
        return launch_followed_as<AFTER, GK, 2, 4, 4, 2, 2, false>(s, a, tail);
    }
    return a.uniform_group_scales ? launch_followed_as<AFTER, GK, 2, 2, 2, 2, 3, true>(s, a, tail)
                                  : launch_followed_as<AFTER, GK, 2, 2, 2, 2, 3, false>(s, a, tail);
}
template <After AFTER>
bool launch_followed_group(hipStream_t s, const LinearArgs& a, const LinearTail& tail, bool wide) {
    switch (a.group_size) {
        case 64: return launch_followed_tile<AFTER, 1>(s, a, tail, wide);
        case 128: return launch_followed_tile<AFTER, 2>(s, a, tail, wide);
        case 256: return launch_followed_tile<AFTER, 4>(s, a, tail, wide);
        default: return false;
    }
}

}  // namespace

// Taken: eight-bit weights in groups of 64 and more, rows that read as they are, and launches that run on the 128x128 or
// the 64x64 tile anyway (a launch of fewer tiles wants the narrow ones, which hold no pairs).
const char* launch_gemm_followed(hipStream_t s, const LinearArgs& a, After after, const LinearTail& tail, int cu_count) {
    if (a.mode != Epilogue::DequantF32 || a.weight_bits != 8u || a.group_size < 64u || a.rows <= kMaxGemvRows || a.acc_out ||
        a.ldx < 16u || a.ldx % 16u || (uintptr_t)a.x % 16u || (uint64_t)a.rows * a.ldx > 0xffffffffull)
        return nullptr;
    const F32Tile tile = pick_f32_tile(a, cu_count > 0 ? cu_count : 256);
    if (tile != F32Tile::T128x128 && tile != F32Tile::T64x64) return nullptr;
    const bool wide = tile == F32Tile::T128x128;
    bool ok = false;
    switch (after) {
        case After::Rope:
            // (16-byte accesses of whole groups of four channels)
            if ((tail.head_dim != 64u && tail.head_dim != 128u) || a.n != (tail.q_heads + 2u * tail.kv_heads) * tail.head_dim ||
                (((uintptr_t)tail.cos_table | (uintptr_t)tail.sin_table | (uintptr_t)tail.q_out | (uintptr_t)tail.k_cache |
                  (uintptr_t)tail.v_cache) % 16u) != 0u)
                return nullptr;
            ok = launch_followed_group<After::Rope>(s, a, tail, wide);
            break;
        case After::Swiglu:
            if (a.n % 64u || (uintptr_t)a.y % 16u) return nullptr;
            ok = launch_followed_group<After::Swiglu>(s, a, tail, wide);
            break;
        case After::Add:
            if (a.n % 4u || (uintptr_t)a.y % 16u) return nullptr;
            ok = launch_followed_group<After::Add>(s, a, tail, wide);
            break;
        case After::Store: return nullptr;
    }
    if (!ok) return nullptr;
    static const char* const names[3][2] = {{"hip.packed-linear.a8-mfma.t64x64k64-rope", "hip.packed-linear.a8-mfma.t128x128k64-rope"},
                                            {"hip.packed-linear.a8-mfma.t64x64k64-swiglu", "hip.packed-linear.a8-mfma.t128x128k64-swiglu"},
                                            {"hip.packed-linear.a8-mfma.t64x64k64-add", "hip.packed-linear.a8-mfma.t128x128k64-add"}};
    return names[(int)after - 1][wide ? 1 : 0];
}

// The requantizing GEMM on 16x16x64 MFMAs.  tile 0: 256 channels x 256 rows per workgroup; 1: 256 x
// 128.  The caller has checked what the straight-line epilogue needs (n % 16 == 0, a 16-byte
// aligned byte output, no accumulator dump).  Returns the tile's name, or null if nothing ran.
const char* launch_gemm_k64(hipStream_t s, const LinearArgs& a, int tile) {
    const bool row = a.mode == Epilogue::RequantRow;
    if (a.mode == Epilogue::DequantF32) return nullptr;
    constexpr int T = (int)Epilogue::RequantTensor, R = (int)Epilogue::RequantRow;
    const bool dq = a.dq_out != nullptr;
    bool ok = false;
    if (a.x_flip_mask) {
        // unsigned activation bytes, flipped in the kernel (the per-tensor form only: per-token scales come with I8 rows)
        if (row) return nullptr;
        if (tile == 0) ok = dq ? launch_one<2, 4, 8, 4, T, true, true>(s, a) : launch_one<2, 4, 8, 4, T, true>(s, a);
        else ok = dq ? launch_one<2, 4, 8, 2, T, true, true>(s, a) : launch_one<2, 4, 8, 2, T, true>(s, a);
    } else if (tile == 0) {
        ok = row ? (dq ? launch_one<2, 4, 8, 4, R, false, true>(s, a) : launch_one<2, 4, 8, 4, R>(s, a))
                 : (dq ? launch_one<2, 4, 8, 4, T, false, true>(s, a) : launch_one<2, 4, 8, 4, T>(s, a));
    } else {
        ok = row ? (dq ? launch_one<2, 4, 8, 2, R, false, true>(s, a) : launch_one<2, 4, 8, 2, R>(s, a))
                 : (dq ? launch_one<2, 4, 8, 2, T, false, true>(s, a) : launch_one<2, 4, 8, 2, T>(s, a));
    }
    if (!ok) return nullptr;
    return tile == 0 ? (dq ? "t256x256k64-dq" : "t256x256k64") : (dq ? "t256x128k64-dq" : "t256x128k64");
}

// The dequantizing GEMM on 16x16x64 MFMAs (16x16x32 for groups of 32, on the three narrow tiles only).
const char* launch_gemm_k64_f32(hipStream_t s, const LinearArgs& a, F32Tile tile) {
    if (a.mode != Epilogue::DequantF32 || a.acc_out || !a.y) return nullptr;
    switch (tile) {
        case F32Tile::T128x256: return launch_f32_group<false, 2, 8, 4, 2, 3>(s, a) ? "t128x256k64s3" : nullptr;
        case F32Tile::T128x128: return launch_f32_bits<2, 4, 4, 2, 2>(s, a) ? "t128x128k64" : nullptr;
        case F32Tile::T64x64: return launch_f32_bits<2, 2, 2, 2, 3>(s, a) ? "t64x64k64" : nullptr;
        case F32Tile::T64x32: return launch_f32_bits<2, 2, 2, 1, 4>(s, a) ? "t64x32k64" : nullptr;
        case F32Tile::T32x32: return launch_f32_bits<2, 2, 1, 1, 4>(s, a) ? "t32x32k64" : nullptr;
    }
    return nullptr;
}

// Which tile.  Few rows or channels: the narrow tiles, which put the outputs on more wavefronts -- a wavefront
// walks all of K with a barrier, the fragments and a fold per group in its way, so what counts first is that no
// SIMD is without one, then that it has two.  us with 64x64 | 64x32 | 32x32 tiles, preparation included
// (and with the 32x32x32 kernels of gemm_mfma.hip that these launches took before):
//   8 bits, groups of 128   64 x 4096 -> 4096     18.1 | 15.0 | 12.3 (21.6)   200 x 4096 -> 4096   19.8 | 18.2 | 18.4 (23.2)
//                           512 x 4096 -> 4096    26.2 | 32.2 | 34.9 (32.7)   333 x 3000 -> 5001   22.7 | 27.8 | 27.1 (29.6)
//                           1000 x 8192 -> 1024   40.2 | 37.2 | 40.7 (46.4)   128 x 3000 -> 5001   16.5 | 15.3 | 13.8 (19.7)
//   4 bits, groups of 32    64 x 4096 -> 4096     40.8 | 27.1 | 19.1 (54.9)   333 x 3000 -> 5001   41.0 | 40.0 | 39.2 (67.1)
//                           512 x 4096 -> 4096    52.1 | 51.1 | 54.2 (94.2)   1024 x 3000 -> 5001  82.3 | 88.6 | 94.4 (227)
// The lines: 1.5 workgroups of a tile per compute unit; 2.5 of 64x32 with four-bit weights in groups of up to 128, whose
// operands take longest to spread (235 x 2048 -> 5120 16.2 | 15.3 | 14.8, 302 x 9728 -> 3584 51.7 | 50.9 | 47.5).
// Past them groups of 32, whose fold is most of their time: 64x32 tiles where a compute unit's share of them, 0.595 of a 64x64 tile each,
// is the smaller one: three against two and five against three, and where rows end in a tile's first half up to ten against six (64x64 | 64x32, 8 bits and then 4: 1000 x 2000 ->
// 1531 28.0 | 24.4 and 29.6 | 25.5, 640 x 1500 -> 4096 27.2 | 27.6 and 28.7 | 28.0; where they are not, 720 x 1500 -> 4500 34.8 | 34.8
// and 33.7 | 34.3, 1500 x 1000 -> 3000 30.7 | 33.1 and 31.6 | 32.2, 2048 x 1024 -> 5184 56.8 | 67.8 and 55.6 | 63.0, -> 13888 130 | 160 and
// 129 | 154).  The other groups: the 128-channel tiles against 64x64, by how many a compute unit gets, in units of one 128x128 tile (an odd
// one of those has no second workgroup to take turns with).  What a 64x64 tile costs of it depends on the fold:
// where both have the products s_a * s_w or neither, 0.345; one scale per channel in groups of 128, whose products
// fit the registers beside the narrow tile alone, 0.3; four-bit weights 0.29.  64x64 | 128x128 | 128x256, 8 bits,
// one scale per channel, groups of 128:
//   1024 x 3000 -> 5001  43.8 | 52.7         700 x 1024 -> 4096   14.0 | 16.9 | 21.0   4096 x 1024 -> 4096  47.0 | 43.7 | 48.0
//   333 x 4096 -> 14336  48.9 | 55.9 | 53.4  700 x 4096 -> 14336  77.7 | 81.4 | 89.9   2048 x 14336 -> 4096  211 | 195 | 172
// scales of their own for every group: 1323 x 1536 -> 12800  68.8 | 62.4, 670 x 7072 -> 8832  98.5 | 91.1; groups of 256:
// 1582 x 4768 -> 3616  68.9 | 59.9.  4 bits, groups of 128:  4096 x 2048 -> 1024  33.1 | 36.9
//   700 x 4096 -> 14336  88.5 | 96.5   2048 x 4096 -> 14336  230 | 214   806 x 1024 -> 13824  34.4 | 33.8
// A 128x256 tile costs 1.75 of a 128x128 one where its products fit the registers and that one's do not: groups of
// 128.  (Groups of 64, where both have them: 2044 x 7040 -> 7616  233 | 197 | 207, 874 x 4288 -> 5920  65.7 | 64.4 | 68.8.)
F32Tile pick_f32_tile(const LinearArgs& a, int cu_count) {
    const auto tiles = [&](uint32_t bn, uint32_t bm) { return (uint64_t)((a.n + bn - 1) / bn) * ((a.rows + bm - 1) / bm); };
    const uint64_t cu = (uint64_t)cu_count, busy = cu * 3 / 2;
    const bool four = a.weight_bits == 4u;
    if (tiles(64, 64) < busy)
        return tiles(64, 32) < (four && a.group_size <= 128u ? cu * 5 / 2 + 1u : busy) ? F32Tile::T32x32 : F32Tile::T64x32;
    const auto per_cu = [&](uint64_t t) { return (t + cu - 1) / cu; };
    if (a.group_size < 64u) return 0.595f * (float)per_cu(tiles(64, 32)) < (float)per_cu(tiles(64, 64)) ? F32Tile::T64x32 : F32Tile::T64x64;
    const uint64_t c128 = per_cu(tiles(128, 128));
    const bool narrow_products = !four && a.uniform_group_scales && a.group_size == 128u;
    const float narrow = (float)per_cu(tiles(64, 64)) * (four ? 0.29f : narrow_products ? 0.3f : 0.345f);
    const float wide = (float)c128 + (c128 % 2 ? (four ? 0.2f : 0.1f) : 0.0f);
    if (a.uniform_group_scales && a.weight_bits == 8u && a.group_size == 128u && a.k >= 4096u) {
        const float deep = 1.75f * (float)per_cu(tiles(128, 256));
        if (deep < wide && deep < narrow) return F32Tile::T128x256;
    }
    return narrow < wide ? F32Tile::T64x64 : F32Tile::T128x128;
}

}  // namespace vxhip
