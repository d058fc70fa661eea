// Fused gated-attention kernels for gfx950 (CDNA4), bf16 storage, head_size 32.
//
// Two kernels compute the gated weighted average avg = softmax(q.k^T/sqrt(d) + bias + pair_bias).v *
// sigmoid(gate) for one (batch row b, head h) unit at a time; everything the reference materialises
// in memory between its GEMMs -- q, k, v, gate, the [bs, S] logits block, the probabilities
// (reference src/attention/gating_attention.cpp:47-66, 97-147) -- stays in LDS and registers:
//
//   persistent_head_kernel  seq_len <= 384 (C=128) / 256 (C=256).  One workgroup per CU keeps one head
//       for its lifetime (its four weight matrices staged once in LDS as MFMA fragments) and walks
//       batch rows; wave j owns sequence block j: it projects the block's K, V, Q and gate, then
//       attends its 32 queries against all keys of the row.
//   fused_head_kernel       any seq_len <= 1024.  One workgroup per unit; projections first (weights
//       staged through LDS in groups), then attention, up to four query blocks per wave.
//
// Both run the same attention blocks.  attend_block_l2 is the fast one (logits in log2 units, no running
// maximum, pair bias from a fragment-major copy made by pair_bias_fragments_kernel, row sums on the
// matrix core); attend_block and attend_block_direct are the general ones (running maximum with lazy
// rescale, pair bias read in place) for calls whose pair bias cannot be copied.
// The final GEMM with fp32 bias (reference :152-157) is output_projection_tile_kernel, or output_projection_kernel.
//
// All contractions are v_mfma_f32_32x32x16_bf16 (fp32 accumulate); fragment and accumulator layouts
// are described in mfma_tiles.h.  Two consequences of those layouts are used everywhere below:
//   * a contraction index may be permuted freely as long as both operands agree, so an accumulator
//     can be fed back as the k-dimension of the next MFMA without any cross-lane movement: Q^T and
//     K^T share their head-dim order, and the probabilities share their key order with V;
//   * the sequence position handled by "row r" of a 32-row block is pi(r) = 16*((r>>2)&1) +
//     4*(r>>3) + (r&3), chosen so that the 16 logits a lane holds for its query are 16 CONSECUTIVE
//     keys (pair-bias row loads become two 16-byte loads).
#include <hip/hip_runtime.h>

#include <atomic>
#include <climits>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <type_traits>
#include <vector>

#include "api_internal.h"
#include "attention_util.h"
#include "device_util.h"
#include "launch_internal.h"
#include "mfma_tiles.h"
#include "profiler.h"

using namespace kutacc_dev;

namespace {

constexpr int HEAD = 32;            // head_size the MFMA kernels are written for
constexpr int MAX_WAVES = 12;       // fused_head_kernel: 768 threads, 3 waves per SIMD, 168 VGPRs each
constexpr int FAIR_SLICE_SHIFT = 11;  // log2 of the clocks a wave keeps one issue priority (timeslice_priority); 2^8 to 2^13 measured alike
constexpr float RESCALE_GAP = 5.5f; // running max may lag the true max by this much (natural log units, ~8 octaves)

// Waves per workgroup a given fused_head_kernel instantiation may be launched with.  One query block
// per wave needs about 140 VGPRs at C=128, which fits three waves per SIMD; the variants that hold
// more state (more query blocks per wave, or 256 input channels in registers) get two per SIMD.
__host__ __device__ constexpr int max_waves(int C, int BPW) { return (C == 128 && BPW <= 2) ? MAX_WAVES : 8; }

enum Proj { PROJ_K = 0, PROJ_V = 1, PROJ_Q = 2, PROJ_G = 3 };

struct FusedParams {
    const bf16_t *x;
    const bf16_t *w[4]; // indexed by Proj
    const float *bg;
    const bf16_t *bias;
    const bf16_t *nb;
    bf16_t *avg;
    int64_t x_ld, x_sb, bias_sb, bias_sk, nb_sh, nb_sq, avg_sb, avg_ss, avg_sh; // x_sb: from one batch row of x to the next
    const float *ln_gamma, *ln_beta; // fused LayerNorm of the input rows (persistent kernel), else nullptr
    float ln_eps;
    int bias_is_mask; // bias holds the 0/1 mask; the kernels form 1e9*(mask-1) themselves
    int B, S, H, NB, NW, GW;
    int nb_vec;   // pair-bias rows may be read with 16-byte loads
    float qscale; // 1 / sqrt(head_size)
    int ngrp;     // persistent kernel: batch-row groups per XCD
    const uint4 *nbf; // pair bias * log2(e): fp16, in fragment-major order (pair_bias_fragments_kernel), or fp32 tiles, or nullptr
    int NT;           // key tiles the LDS arrays are laid out for: NB rounded up to an even number (the log2-unit
                      // loop walks tile pairs; the phantom tile's K and V are zeros, its mask is -inf, and in the copies
                      // of the pair bias it holds what keys past the end hold: PAST_THE_END_F16 or LOWEST_BIAS)
    int l2mode;       // logits in log2 units (attend_block_l2); needs nbf when there is a pair bias
};

// 0/1 selection fragments that scatter the pair-bias words a lane loads (16 consecutive keys, 8 per
// MFMA) onto the logits rows: row i of a tile is key pi(i); k-slot 8*g+e of the first MFMA carries
// key 16*g+e, of the second key 16*g+8+e.
__device__ __forceinline__ void make_selectors(int lane, bf16x8 &sel0, bf16x8 &sel1)
{
    const int r = lane & 31, g = lane >> 5;
    const int gi = (r >> 2) & 1;          // which 16-key half row r belongs to
    const int w = 4 * (r >> 3) + (r & 3); // position of row r's key inside that half
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        sel0[e] = (bf16_t)((gi == g && w == e) ? 1.0f : 0.0f);
        sel1[e] = (bf16_t)((gi == g && w == e + 8) ? 1.0f : 0.0f);
    }
}

// Pair-bias words on their way into a selector MFMA: -inf (and any negative NaN pattern) becomes the most negative power of
// two in bf16, since the MFMA multiplies every word by 0 or 1 and 0 x inf is a NaN.  As 16-bit unsigned numbers the negative
// values sort by magnitude, so this is one packed minimum per word; what the logit then holds is absorbed like a -inf, and finite with a mask as low
// (finite_bias).
__device__ __forceinline__ uint4 finite_bias_words(uint4 w)
{
    typedef __attribute__((ext_vector_type(2))) unsigned short u16x2;
    union {
        uint4 u;
        u16x2 h[4];
    } c;
    c.u = w;
    const u16x2 bound = {0xff00, 0xff00};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        c.h[i] = __builtin_elementwise_min(c.h[i], bound);
    }
    return c.u;
}

// The same selectors with fp16 ones, for the log2-unit loop, whose pair-bias fragments are fp16.
__device__ __forceinline__ void make_selectors_f16(int lane, f16x8 &sel0, f16x8 &sel1)
{
    const int r = lane & 31, g = lane >> 5;
    const int gi = (r >> 2) & 1;
    const int w = 4 * (r >> 3) + (r & 3);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        sel0[e] = (_Float16)((gi == g && w == e) ? 1.0f : 0.0f);
        sel1[e] = (_Float16)((gi == g && w == e + 8) ? 1.0f : 0.0f);
    }
}

// The mask that all S keys of a row have, as it was staged; 0 if they differ
__device__ __forceinline__ float one_mask_of(const float *mask, int S, int lane)
{
    const float first = mask[0];
    bool differ = false;
    for (int k = lane; k < S; k += 64) {
        differ |= mask[k] != first;
    }
    return __any(differ) ? 0.f : first;
}

// Mask bias of one batch row -> LDS as fp32 (keys past S get -inf), plus one flag bit per 32-key tile
// saying "this tile needs the mask added" (non-zero bias or ragged tail; keys from `flagged` on set none).  Wave w covers keys
// [64w, 64w+64); *flag_word must have been zeroed before, with a barrier in between.
// bias_row[k * stride_k] is the mask bias itself, or (from_mask) the 0/1 mask, turned into 1e9*(mask-1) here with the
// same multiply-add and bf16 rounding as the stand-alone mask-bias pass.
template <bool NEAR = false> // NEAR: S * stride_k < 2^31 and stride_k < 2^24 (checked on the host), 32-bit offsets
__device__ __forceinline__ void stage_mask_part(const bf16_t *bias_row, float *mask, uint32_t *flag_word, int S, int NB,
                                                int flagged, int wave, int lane, float scale, int64_t stride_k, bool from_mask)
{
    const int k = wave * 64 + lane;
    if (wave * 64 < NB * 32) {
        float mv = -INFINITY;
        if (k < S) {
            mv = to_f32(bias_row[NEAR ? (int64_t)__umul24((uint32_t)k, (uint32_t)stride_k) : k * stride_k]);
            if (from_mask) {
                mv = to_f32((bf16_t)fmaf(mv, 1e9f, -1e9f));
            }
            mv = finite_bias(mv * scale);
        }
        if (k < NB * 32) {
            mask[k] = mv;
        }
        const unsigned long long nz = __ballot(k < flagged && mv != 0.f);
        const uint32_t bits = (((uint32_t)nz != 0u ? 1u : 0u) | ((uint32_t)(nz >> 32) != 0u ? 2u : 0u)) << (2 * wave);
        if (lane == 0 && bits != 0u) {
            atomicOr(flag_word, bits);
        }
    }
}

// stage_mask_part for the two-row kernel, which adds a row's mask bias to its logits with one more MFMA (a rank-one
// product of the per-key values with ones) instead of sixteen vector additions per tile: the value of key k is stored
// as two bf16, v = hi + lo to 2^-17 of |v|, the k-slots 0 and 1 of that MFMA's A operand.  -inf (keys past S): hi = -inf,
// lo = 0.  Keys from `flagged` on set no flag: those past S need no mask where the tiles of the pair bias have them at LOWEST_BIAS, so that rows of a ragged
// length without a mask take the loop without one (the operator, us: 199 residues 38.0 -> 36.2, 255 43.5 -> 42.1, 352 80.5 -> 75.6, 383 90.9 -> 86.2; MSA
// rows of 255, whole block, 119.6 -> 116.9).
template <bool NEAR = false>
__device__ __forceinline__ void stage_mask_words(const bf16_t *bias_row, uint32_t *words, uint32_t *flag_word, int S, int NB,
                                                 int flagged, int wave, int lane, float scale, int64_t stride_k, bool from_mask)
{
    const int k = wave * 64 + lane;
    if (wave * 64 < NB * 32) {
        float mv = -INFINITY;
        if (k < S) {
            mv = to_f32(bias_row[NEAR ? (int64_t)__umul24((uint32_t)k, (uint32_t)stride_k) : k * stride_k]);
            if (from_mask) {
                mv = to_f32((bf16_t)fmaf(mv, 1e9f, -1e9f));
            }
            mv = finite_bias(mv * scale);
        }
        if (k < NB * 32) {
            words[k] = mask_word(mv);
        }
        const unsigned long long nz = __ballot(k < flagged && mv != 0.f);
        const uint32_t bits = (((uint32_t)nz != 0u ? 1u : 0u) | ((uint32_t)(nz >> 32) != 0u ? 2u : 0u)) << (2 * wave);
        if (lane == 0 && bits != 0u) {
            atomicOr(flag_word, bits);
        }
    }
}

// The value stage_mask_part would store for key k, in two steps for kernels that fetch the mask early and store it
// later, so that nothing waits for the load where it is issued: the raw element of key min(k, S - 1) ...
__device__ __forceinline__ bf16_t mask_bias_fetch(const bf16_t *bias_row, int S, int k, int64_t stride_k)
{
    return bias_row[(k < S ? k : S - 1) * stride_k];
}

// ... and the value made of it where it is stored.
__device__ __forceinline__ float mask_bias_finish(bf16_t raw, bool in_range, float scale, bool from_mask)
{
    float mv = to_f32(raw);
    if (from_mask) {
        mv = to_f32((bf16_t)fmaf(mv, 1e9f, -1e9f));
    }
    return in_range ? finite_bias(mv * scale) : -INFINITY;
}

// Flash-style attention of one 32-query block against all keys of the unit.
//   lds_k / lds_v : K and V fragments of the unit, [tile][kstep][lane] in 16-byte units
//   mask4         : fp32 mask bias in LDS, already offset by 16*g floats; flags: one bit per tile
//   nb_head       : pair bias of this head, [S, S] with row stride nb_sq (HAS_NB only); q0row = first
//                   query of the block
//   panel         : wave-private 4 KB staging panel, or nullptr to load the pair bias directly
//   q0, q1        : Q^T fragments scaled by 1/sqrt(d)
// Returns the unnormalised O^T accumulator and the row sum (identical in both lane halves).
// Per key tile: the logits accumulator starts at the mask bias (or 0); two MFMAs with the 0/1 selectors
// add the pair bias straight from its bf16 words (exact), two add q.k; the running maximum is
// refreshed only when some row's tile maximum exceeds it by RESCALE_GAP; probabilities go from the
// accumulator registers into the B operand of the P.V MFMAs without touching LDS.  The logits of
// tile t+1 are issued before the softmax of tile t so that the matrix core works under the VALU.
// Pair bias arrives two key tiles (64 keys = one 128-byte line per query) at a time through the
// staging panel, prefetched one pair ahead into registers; tiles of a ragged or unaligned tail are
// read directly.
template <bool HAS_NB>
__device__ __forceinline__ void attend_block(const uint4 *lds_k, const uint4 *lds_v, const f32x4 *mask4, uint32_t flags,
                                             const bf16_t *nb_head, int64_t nb_sq, int q0row, bool nb_vec, uint4 *panel,
                                             bf16x8 q0, bf16x8 q1, bf16x8 sel0, bf16x8 sel1, int NB, int S, int lane,
                                             f32x16 &o_out, float &l_out)
{
    const int r = lane & 31, g = lane >> 5;
    const int prow = pi_row(r);
    f32x16 o = zero16();
    float m_run = -1e30f; // finite, so the first rescale factor is exp2(-huge) = 0, never NaN
    float lsum = 0.f;     // this lane's share of the row sum; the two halves are added at the end
    bf16x2 one2;
    one2[0] = (bf16_t)1.0f, one2[1] = (bf16_t)1.0f;

    const int qrow = q0row + prow < S ? q0row + prow : S - 1;
    const bf16_t *nbrow = HAS_NB ? nb_head + (int64_t)qrow * nb_sq + 16 * g : nullptr;
    // number of leading tile pairs that go through the staging panel
    const int staged_pairs = (HAS_NB && panel != nullptr && nb_vec) ? S / 64 : 0;
    PanelRegs pf; // the next staged pair, in flight from global memory
    if (HAS_NB && staged_pairs > 0) {
        pf = panel_load(nb_head, nb_sq, q0row, S - 1, 0, lane);
    }

    // pair-bias words of key tile t for this lane (16 consecutive keys): B operands of the selector MFMAs
    auto nb_words = [&](int t, uint4 &w0, uint4 &w1) {
        const int pair = t >> 1;
        if (pair < staged_pairs) {
            if ((t & 1) == 0) {
                panel_store(panel, lane, pf); // the previous pair's reads were issued earlier in program order
                if (pair + 1 < staged_pairs) {
                    pf = panel_load(nb_head, nb_sq, q0row, S - 1, (pair + 1) * 64, lane);
                }
            }
            const int c = 4 * (t & 1) + 2 * g;
            w0 = panel[panel_slot(prow, c)];
            w1 = panel[panel_slot(prow, c + 1)];
        } else if (nb_vec && (t + 1) * 32 <= S) {
            w0 = *reinterpret_cast<const uint4 *>(nbrow + t * 32);
            w1 = *reinterpret_cast<const uint4 *>(nbrow + t * 32 + 8);
        } else {
            const uint16_t *s16 = reinterpret_cast<const uint16_t *>(nbrow + t * 32);
            const int key0 = t * 32 + 16 * g;
            uint32_t wds[8];
#pragma unroll
            for (int v = 0; v < 8; ++v) {
                const uint32_t a0 = key0 + 2 * v < S ? s16[2 * v] : 0u;
                const uint32_t a1 = key0 + 2 * v + 1 < S ? s16[2 * v + 1] : 0u;
                wds[v] = a0 | (a1 << 16);
            }
            w0.x = wds[0], w0.y = wds[1], w0.z = wds[2], w0.w = wds[3];
            w1.x = wds[4], w1.y = wds[5], w1.z = wds[6], w1.w = wds[7];
        }
    };
    // logits^T of key tile t (rows = keys, columns = this wave's 32 queries), natural-log units
    auto logits = [&](int t, f32x16 &x) {
        if ((flags >> t) & 1u) {
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const f32x4 mv = mask4[t * 8 + a];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    x[4 * a + c] = mv[c];
                }
            }
        } else {
            x = zero16();
        }
        if (HAS_NB) {
            uint4 w0, w1;
            nb_words(t, w0, w1);
            x = mfma(sel0, as_bf16x8(finite_bias_words(w0)), x);
            x = mfma(sel1, as_bf16x8(finite_bias_words(w1)), x);
        }
        x = mfma(as_bf16x8(lds_k[(t * 2 + 0) * 64 + lane]), q0, x);
        x = mfma(as_bf16x8(lds_k[(t * 2 + 1) * 64 + lane]), q1, x);
    };
    // online softmax of tile t held in xc, then O^T += V^T . P; before that, start tile t+1 into xn
    auto step = [&](int t, f32x16 &xc, f32x16 &xn) {
        if (t + 1 < NB) {
            logits(t + 1, xn);
        }
        float mx = xc[0];
#pragma unroll
        for (int v = 1; v < 16; ++v) {
            mx = fmaxf(mx, xc[v]);
        }
        mx = half_swap_max(mx);
        if (__any(mx > m_run + RESCALE_GAP)) {
            const float m_new = fmaxf(m_run, mx);
            const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * LOG2E);
            lsum *= alpha;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                o[v] *= alpha;
            }
            m_run = m_new;
        }
        const float ml = -m_run * LOG2E;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            xc[v] = __builtin_amdgcn_exp2f(fmaf(xc[v], LOG2E, ml));
        }
        // the row sum is taken over the bf16-rounded probabilities, two per dot2 instruction
        const bf16x8 p0 = pack8(xc, 0), p1 = pack8(xc, 8);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            bf16x2 a, c;
            a[0] = p0[2 * v], a[1] = p0[2 * v + 1];
            c[0] = p1[2 * v], c[1] = p1[2 * v + 1];
            lsum = __builtin_amdgcn_fdot2_f32_bf16(a, one2, lsum, false);
            lsum = __builtin_amdgcn_fdot2_f32_bf16(c, one2, lsum, false);
        }
        o = mfma(as_bf16x8(lds_v[(t * 2 + 0) * 64 + lane]), p0, o);
        o = mfma(as_bf16x8(lds_v[(t * 2 + 1) * 64 + lane]), p1, o);
    };

    // softmax of a finished logits tile and its P.V accumulation (the part of `step` after the lookahead)
    auto softmax_pv = [&](int t, f32x16 &xc) {
        float mx = xc[0];
#pragma unroll
        for (int v = 1; v < 16; ++v) {
            mx = fmaxf(mx, xc[v]);
        }
        mx = half_swap_max(mx);
        if (__any(mx > m_run + RESCALE_GAP)) {
            const float m_new = fmaxf(m_run, mx);
            const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * LOG2E);
            lsum *= alpha;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                o[v] *= alpha;
            }
            m_run = m_new;
        }
        const float ml = -m_run * LOG2E;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            xc[v] = __builtin_amdgcn_exp2f(fmaf(xc[v], LOG2E, ml));
        }
        const bf16x8 p0 = pack8(xc, 0), p1 = pack8(xc, 8);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            bf16x2 a, c;
            a[0] = p0[2 * v], a[1] = p0[2 * v + 1];
            c[0] = p1[2 * v], c[1] = p1[2 * v + 1];
            lsum = __builtin_amdgcn_fdot2_f32_bf16(a, one2, lsum, false);
            lsum = __builtin_amdgcn_fdot2_f32_bf16(c, one2, lsum, false);
        }
        o = mfma(as_bf16x8(lds_v[(t * 2 + 0) * 64 + lane]), p0, o);
        o = mfma(as_bf16x8(lds_v[(t * 2 + 1) * 64 + lane]), p1, o);
    };
    // logits of a tile whose pair bias sits in the staging panel; no branches, so that the scheduler
    // can spread the LDS reads, MFMAs and the neighbouring softmax over each other
    auto logits_staged = [&](int t, f32x16 &x, auto with_mask) {
        if (decltype(with_mask)::value) {
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const f32x4 mv = mask4[t * 8 + a];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    x[4 * a + c] = mv[c];
                }
            }
        } else {
            x = zero16();
        }
        const int c0 = 4 * (t & 1) + 2 * g;
        x = mfma(sel0, as_bf16x8(finite_bias_words(panel[panel_slot(prow, c0)])), x);
        x = mfma(sel1, as_bf16x8(finite_bias_words(panel[panel_slot(prow, c0 + 1)])), x);
        x = mfma(as_bf16x8(lds_k[(t * 2 + 0) * 64 + lane]), q0, x);
        x = mfma(as_bf16x8(lds_k[(t * 2 + 1) * 64 + lane]), q1, x);
    };

    f32x16 xa, xb;
    logits(0, xa);
    int t = 0;
    // main loop: two key tiles per iteration while a further staged pair follows; straight-line body
    auto main_loop = [&](auto with_mask) {
        for (int pair = 0; pair + 1 < staged_pairs; ++pair) {
            const int t0 = 2 * pair;
            logits_staged(t0 + 1, xb, with_mask);
            softmax_pv(t0, xa);
            panel_store(panel, lane, pf); // pair+1; the reads of this pair were issued above
            // prefetch pair+2 (clamped to the last staged pair: a harmless re-read instead of a branch)
            const int nxt = pair + 2 < staged_pairs ? pair + 2 : staged_pairs - 1;
            pf = panel_load(nb_head, nb_sq, q0row, S - 1, nxt * 64, lane);
            logits_staged(t0 + 2, xa, with_mask);
            softmax_pv(t0 + 1, xb);
        }
    };
    if (HAS_NB && staged_pairs > 1) {
        if (flags != 0u) {
            main_loop(std::true_type{});
        } else {
            main_loop(std::false_type{});
        }
        t = 2 * (staged_pairs - 1);
    }
    // remaining tiles (last staged pair, unstaged or ragged tail, or everything when nothing is staged)
    for (; t < NB; t += 2) {
        step(t, xa, xb);
        if (t + 1 < NB) {
            step(t + 1, xb, xa);
        }
    }
    o_out = o;
    l_out = half_swap_sum(lsum);
}

// ---- attention of one 32-query block in log2 units (the mode the persistent kernel runs in whenever
// it can) ----
// All inputs of the logits are pre-scaled by log2(e): the Q fragments by the kernel, the pair bias by
// pair_bias_fragments_kernel, the mask bias when it is staged.  The accumulator of the logits MFMAs is
// then the exponent itself, and the softmax of a tile is 16 v_exp_f32 and 8 packed converts -- the
// vector ALU no longer bounds the loop.  What the VALU used to do is done by the matrix core:
//  * no running maximum: the probabilities are 2^logit, unshifted.  Softmax is shift invariant and
//    fp32 and bf16 both carry 8 exponent bits, so this is exact in the same sense as the shifted form
//    as long as nothing overflows or the whole row underflows; the caller checks the row sum for
//    that (1e-30 < l < 1e30) and repeats the block with SHIFT = true and the true row maximum
//    (row_max_l2) when the check fails.  SHIFT costs one subtract per logit.
//  * the row sums come from a 16x16x32 MFMA whose A operand adds up the keys of each query
//    (rowsum_selector), fed with the same bf16 probabilities as the P.V product.
// Every operand of a tile is fetched ahead into registers that the loop carries: K and V fragments
// from LDS one tile ahead, pair-bias fragments from global memory two tiles ahead (two contiguous 1 KB
// loads per tile and wave).  The 8 MFMAs of a tile sit, fenced, between the exp/convert pieces of the
// neighbouring tile's softmax.  The loop runs one extra (clamped) logits computation at the end
// instead of a peeled epilogue.  Requires an even number of key tiles.
// TILES: the pair bias comes as fp32 tiles in accumulator order (pair_bias_tiles_kernel), which seed the logits MFMAs: twice the
// bytes of the fragments, no selector MFMAs, and no second rounding of the bias.
//   nbf : this wave's fragment-major pair bias, already offset by the lane: tile t at nbf[(2t+m)*64] (TILES: nbf[(4t+a)*64])
//   returns the row sum of every lane's query in l_out

// Issue priority of a wave among the (up to three) waves of its workgroup on one SIMD, by time slices of the clock they
// all see: in slice s the wave with turn (s + d) mod 3 gets priority 2 - d, so over three slices every wave is first,
// second and third once, however far it has come.  Left to the arbiter's oldest-first rule the oldest wave runs its
// attention almost alone and the youngest is left to finish by itself while the others wait at the barrier.  The
// branches sit inside one asm statement: as branches of a loop body they split the body into blocks, and the register
// allocator spills across them.  Call once per tile pair; reset with s_setprio 0 after the loop.
__device__ __forceinline__ void timeslice_priority(uint32_t turn, int shift)
{
    const uint32_t tick = ((uint32_t)__builtin_amdgcn_s_memtime() >> shift) & 0x3fffu;
    const uint32_t slice = tick - 3u * ((tick * 0x5556u) >> 16); // tick mod 3
    const uint32_t d = turn >= slice ? turn - slice : turn + 3u - slice;
    asm volatile("s_cmp_eq_u32 %0, 0\n\t"
                 "s_cbranch_scc1 .Lfirst_%=\n\t"
                 "s_cmp_eq_u32 %0, 1\n\t"
                 "s_cbranch_scc1 .Lsecond_%=\n\t"
                 "s_setprio 0\n\t"
                 "s_branch .Ldone_%=\n"
                 ".Lfirst_%=:\n\t"
                 "s_setprio 2\n\t"
                 "s_branch .Ldone_%=\n"
                 ".Lsecond_%=:\n\t"
                 "s_setprio 1\n"
                 ".Ldone_%=:"
                 :
                 : "s"(d)
                 : "scc");
}

// fp32 tile t of the pair bias, from a pointer offset by the lane
__device__ __forceinline__ f32x16 pair_bias_tile(const uint4 *nbf, int t)
{
    f32x16 c;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        const f32x4 v = *reinterpret_cast<const f32x4 *>(nbf + (t * 4 + a) * 64);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            c[4 * a + e] = v[e];
        }
    }
    return c;
}

template <bool HAS_NB, bool WITH_MASK, bool SHIFT, bool TILES = false, bool ODD = false>
__device__ __forceinline__ void attend_block_l2(const uint4 *lds_k, const uint4 *lds_v, const f32x4 *mask4,
                                                const uint4 *nbf, bf16x8 q0, bf16x8 q1, f16x8 sel0, f16x8 sel1,
                                                bf16x8 sumsel, int NB, int lane, float shift, f32x16 &o_out, float &l_out,
                                                int prio_phase = -1, int fair_turn = -1)
{
    // ODD: the last tile is the one of zeros behind an odd number of them, and left out (us, triangle attention of 77 residues 18.9 -> 18.4, 150
    // 33.6 -> 32.4, 288 70.9 -> 67.9, 450 211.5 -> 206, 600 391 -> 382; MSA rows, two rows a step, 512 x 224 186.3 -> 184.1).  A loop of its own, and
    // in the kernels of single rows a kernel of its own: decided inside one loop, even numbers lost 0.5 to 1 %, and both loops in one kernel spill
    // registers (triangle attention of 185 padded residues 38.2 us so, 36.8 now, 300 83.0 and 75.7, 450 193 and 189).
    const int npairs = NB >> 1;
    const uint4 *kp = lds_k + lane;
    const uint4 *vp = lds_v + lane;

    auto init = [&](int t) {
        f32x16 x;
        if (WITH_MASK) {
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const f32x4 mv = mask4[t * 8 + a];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    x[4 * a + c] = mv[c];
                }
            }
        } else {
            x = zero16();
        }
        return x;
    };
    auto clampt = [&](int t) { return t < NB ? t : NB - 1; };
    auto load_tile = [&](int t) { return pair_bias_tile(nbf, t); };
    auto seed = [&](int t, const f32x16 &C) { // of the logits, where the mask has to be added to the tile
        f32x16 x = init(t);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            x[v] += C[v];
        }
        return x;
    };

    // pair-bias words: wa* belong to even tiles, wb* to odd tiles; tiles Ca and Cb likewise
    uint4 wa0 = {}, wa1 = {}, wb0 = {}, wb1 = {}, k0, k1, v0, v1;
    f32x16 Ca, Cb;
    if constexpr (TILES) {
        Ca = load_tile(0), Cb = load_tile(clampt(1));
    } else if (HAS_NB) {
        wa0 = nbf[0], wa1 = nbf[64];
        wb0 = nbf[2 * 64], wb1 = nbf[3 * 64];
        // Pinned in this order, ahead of the reload of wa below: the loop then finds the loads in flight in the order it
        // leaves them in itself (odd tile's words older than the even tile's), and its wait at the top lets the two
        // newest stay in flight instead of draining the queue.
        __builtin_amdgcn_sched_barrier(0);
    }
    k0 = kp[0], k1 = kp[64];
    f32x16 xa = init(0), xb;
    if constexpr (TILES) {
        xa = seed(0, Ca);
        Ca = load_tile(clampt(2));
    } else if (HAS_NB) {
        xa = mfma_f16(sel0, as_f16x8(wa0), xa);
        xa = mfma_f16(sel1, as_f16x8(wa1), xa);
        wa0 = nbf[clampt(2) * 128], wa1 = nbf[clampt(2) * 128 + 64];
    }
    xa = mfma(as_bf16x8(k0), q0, xa);
    xa = mfma(as_bf16x8(k1), q1, xa);
    k0 = kp[2 * 64], k1 = kp[3 * 64];
    v0 = vp[0], v1 = vp[64];

    f32x16 o = zero16();
    f32x4 lacc = {0.f, 0.f, 0.f, 0.f};

    auto exp4 = [&](f32x16 &x, int base) {
#pragma unroll
        for (int v = base; v < base + 4; ++v) {
            x[v] = __builtin_amdgcn_exp2f(SHIFT ? x[v] - shift : x[v]);
        }
    };
    auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
    // One half step: the softmax and P.V of the finished tile `xc`, with the logits MFMAs of the
    // following tile `xn` (pair-bias words w0, w1) spread between its pieces; t_w is the tile whose
    // pair-bias words replace w0, w1 once consumed, t_k the tile whose K fragments replace k0, k1.
    auto half_step = [&](f32x16 &xc, f32x16 &xn, int t_next, uint4 &w0, uint4 &w1, f32x16 &C, int t_w, int t_k) {
        bf16x8 p0, p1;
        if constexpr (TILES) {
            xn = WITH_MASK ? seed(t_next, C) : C;
            exp4(xc, 0);
            exp4(xc, 4);
            p0 = pack8(xc, 0);
            fence();
            xn = mfma(as_bf16x8(k0), q0, xn);
            asm volatile("" ::"v"(C)); // C stays live past its reader: the logits get registers of their own
            o = mfma(as_bf16x8(v0), p0, o);
            C = load_tile(t_w);
            exp4(xc, 8);
            fence();
            xn = mfma(as_bf16x8(k1), q1, xn);
            lacc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(sumsel, p0, lacc, 0, 0, 0);
            k0 = kp[(t_k * 2 + 0) * 64], k1 = kp[(t_k * 2 + 1) * 64];
            exp4(xc, 12);
            p1 = pack8(xc, 8);
            fence();
            o = mfma(as_bf16x8(v1), p1, o);
            lacc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(sumsel, p1, lacc, 0, 0, 0);
            return;
        }
        xn = init(t_next);
        if (HAS_NB) {
            xn = mfma_f16(sel0, as_f16x8(w0), xn);
            exp4(xc, 0);
            fence();
            xn = mfma_f16(sel1, as_f16x8(w1), xn);
            w0 = nbf[t_w * 128], w1 = nbf[t_w * 128 + 64];
            exp4(xc, 4);
            p0 = pack8(xc, 0);
            fence();
        } else {
            exp4(xc, 0);
            exp4(xc, 4);
            p0 = pack8(xc, 0);
            fence();
        }
        xn = mfma(as_bf16x8(k0), q0, xn);
        o = mfma(as_bf16x8(v0), p0, o);
        exp4(xc, 8);
        fence();
        xn = mfma(as_bf16x8(k1), q1, xn);
        lacc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(sumsel, p0, lacc, 0, 0, 0);
        k0 = kp[(t_k * 2 + 0) * 64], k1 = kp[(t_k * 2 + 1) * 64];
        exp4(xc, 12);
        p1 = pack8(xc, 8);
        fence();
        o = mfma(as_bf16x8(v1), p1, o);
        lacc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(sumsel, p1, lacc, 0, 0, 0);
    };

    for (int pair = 0; pair < (ODD ? npairs - 1 : npairs); ++pair) {
        if (fair_turn >= 0) {
            timeslice_priority((uint32_t)fair_turn, FAIR_SLICE_SHIFT);
        }
        if (prio_phase >= 0) {
            // two waves of one workgroup share a SIMD in lock step; the arbiter prefers the older one, which then runs
            // ahead and leaves the other to finish alone.  Alternating the issue priority per tile pair keeps them level.
            if ((pair + prio_phase) & 1) {
                __builtin_amdgcn_s_setprio(1);
            } else {
                __builtin_amdgcn_s_setprio(0);
            }
        }
        const int t1 = 2 * pair + 1;
        const int tn = pair + 1 < npairs ? 2 * pair + 2 : 2 * pair; // next pair's first tile, clamped
        // ---- odd tile's logits under the even tile's softmax ----
        half_step(xa, xb, t1, wb0, wb1, Cb, clampt(t1 + 2), tn);
        v0 = vp[(t1 * 2 + 0) * 64], v1 = vp[(t1 * 2 + 1) * 64];
        fence();
        // ---- next pair's even tile under the odd tile's softmax ----
        half_step(xb, xa, tn, wa0, wa1, Ca, clampt(tn + 2), tn + 1);
        v0 = vp[(tn * 2 + 0) * 64], v1 = vp[(tn * 2 + 1) * 64];
        fence();
    }
    if constexpr (ODD) { // the last tile by itself: its logits are there
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            exp4(xa, 8 * k);
            exp4(xa, 8 * k + 4);
            const bf16x8 pv = pack8(xa, 8 * k);
            o = mfma(as_bf16x8(k == 0 ? v0 : v1), pv, o);
            lacc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(sumsel, pv, lacc, 0, 0, 0);
        }
    }
    if (fair_turn >= 0) {
        __builtin_amdgcn_s_setprio(0);
    }
    o_out = o;
    l_out = rowsum_fetch(lacc, lane);
}

// Row maxima of the logits (log2 units) of one 32-query block over all key tiles: the shift for the
// repeat of attend_block_l2 after an overflow or underflow.  Not a hot path: operands are loaded at use.
template <bool HAS_NB, bool TILES = false>
__device__ __forceinline__ float row_max_l2(const uint4 *lds_k, const f32x4 *mask4, const uint4 *nbf, bf16x8 q0, bf16x8 q1,
                                            f16x8 sel0, f16x8 sel1, int NB, int lane)
{
    float mx = -INFINITY;
    for (int t = 0; t < NB; ++t) {
        f32x16 x;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const f32x4 mv = mask4[t * 8 + a];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                x[4 * a + c] = mv[c];
            }
        }
        if constexpr (TILES) {
            const f32x16 C = pair_bias_tile(nbf, t);
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                x[v] += C[v];
            }
        } else if (HAS_NB) {
            x = mfma_f16(sel0, as_f16x8(nbf[t * 128]), x);
            x = mfma_f16(sel1, as_f16x8(nbf[t * 128 + 64]), x);
        }
        x = mfma(as_bf16x8(lds_k[(t * 2 + 0) * 64 + lane]), q0, x);
        x = mfma(as_bf16x8(lds_k[(t * 2 + 1) * 64 + lane]), q1, x);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            mx = fmaxf(mx, x[v]);
        }
    }
    mx = half_swap_max(mx);
    return mx; // finite: a fully masked row has -1e9*log2(e) everywhere
}

// The same attention of one 32-query block for kernels without a staging panel (long sequences, where
// K and V fill the LDS): every lane reads the pair bias of its own query row directly, 16 consecutive
// keys per tile, prefetched one tile ahead into registers.
template <bool HAS_NB>
__device__ __forceinline__ void attend_block_direct(const uint4 *lds_k, const uint4 *lds_v, const f32x4 *mask4,
                                                    uint32_t flags, const bf16_t *nbrow, bool nb_vec, bf16x8 q0,
                                                    bf16x8 q1, bf16x8 sel0, bf16x8 sel1, int NB, int S, int lane,
                                                    f32x16 &o_out, float &l_out)
{
    const int g = lane >> 5;
    f32x16 o = zero16();
    float m_run = -1e30f; // finite, so the first rescale factor is exp2(-huge) = 0, never NaN
    float lsum = 0.f;     // this lane's share of the row sum; the two halves are added at the end
    uint32_t nbw[8];      // pair-bias words of the NEXT tile to be turned into logits (prefetched)
    bf16x2 one2;
    one2[0] = (bf16_t)1.0f, one2[1] = (bf16_t)1.0f;

    // raw pair-bias of key tile t for this lane: 16 consecutive keys, two bf16 per word
    auto fetch_nb = [&](int t) {
        if (!HAS_NB) {
            return;
        }
        const bf16_t *src = nbrow + t * 32;
        if (nb_vec && (t + 1) * 32 <= S) {
            const uint4 lo = *reinterpret_cast<const uint4 *>(src);
            const uint4 hi = *reinterpret_cast<const uint4 *>(src + 8);
            nbw[0] = lo.x, nbw[1] = lo.y, nbw[2] = lo.z, nbw[3] = lo.w;
            nbw[4] = hi.x, nbw[5] = hi.y, nbw[6] = hi.z, nbw[7] = hi.w;
        } else {
            const uint16_t *s16 = reinterpret_cast<const uint16_t *>(src);
            const int key0 = t * 32 + 16 * g;
#pragma unroll
            for (int v = 0; v < 8; ++v) {
                const uint32_t a0 = key0 + 2 * v < S ? s16[2 * v] : 0u;
                const uint32_t a1 = key0 + 2 * v + 1 < S ? s16[2 * v + 1] : 0u;
                nbw[v] = a0 | (a1 << 16);
            }
        }
    };
    // logits^T of key tile t (rows = keys, columns = this wave's 32 queries), natural-log units
    auto logits = [&](int t, f32x16 &x) {
        if ((flags >> t) & 1u) {
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const f32x4 mv = mask4[t * 8 + a];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    x[4 * a + c] = mv[c];
                }
            }
        } else {
            x = zero16();
        }
        if (HAS_NB) {
            uint4 w0, w1;
            w0.x = nbw[0], w0.y = nbw[1], w0.z = nbw[2], w0.w = nbw[3];
            w1.x = nbw[4], w1.y = nbw[5], w1.z = nbw[6], w1.w = nbw[7];
            x = mfma(sel0, as_bf16x8(finite_bias_words(w0)), x);
            x = mfma(sel1, as_bf16x8(finite_bias_words(w1)), x);
            if (t + 1 < NB) {
                fetch_nb(t + 1); // in flight while this tile's MFMAs and the previous tile's softmax run
            }
        }
        x = mfma(as_bf16x8(lds_k[(t * 2 + 0) * 64 + lane]), q0, x);
        x = mfma(as_bf16x8(lds_k[(t * 2 + 1) * 64 + lane]), q1, x);
    };
    // online softmax of tile t held in xc, then O^T += V^T . P; before that, start tile t+1 into xn
    auto step = [&](int t, f32x16 &xc, f32x16 &xn) {
        if (t + 1 < NB) {
            logits(t + 1, xn);
        }
        float mx = xc[0];
#pragma unroll
        for (int v = 1; v < 16; ++v) {
            mx = fmaxf(mx, xc[v]);
        }
        mx = half_swap_max(mx);
        if (__any(mx > m_run + RESCALE_GAP)) {
            const float m_new = fmaxf(m_run, mx);
            const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * LOG2E);
            lsum *= alpha;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                o[v] *= alpha;
            }
            m_run = m_new;
        }
        const float ml = -m_run * LOG2E;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            xc[v] = __builtin_amdgcn_exp2f(fmaf(xc[v], LOG2E, ml));
        }
        // the row sum is taken over the bf16-rounded probabilities, two per dot2 instruction
        const bf16x8 p0 = pack8(xc, 0), p1 = pack8(xc, 8);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            bf16x2 a, c;
            a[0] = p0[2 * v], a[1] = p0[2 * v + 1];
            c[0] = p1[2 * v], c[1] = p1[2 * v + 1];
            lsum = __builtin_amdgcn_fdot2_f32_bf16(a, one2, lsum, false);
            lsum = __builtin_amdgcn_fdot2_f32_bf16(c, one2, lsum, false);
        }
        o = mfma(as_bf16x8(lds_v[(t * 2 + 0) * 64 + lane]), p0, o);
        o = mfma(as_bf16x8(lds_v[(t * 2 + 1) * 64 + lane]), p1, o);
    };

    f32x16 xa, xb;
    fetch_nb(0);
    logits(0, xa);
    for (int t = 0; t < NB; t += 2) {
        step(t, xa, xb);
        if (t + 1 < NB) {
            step(t + 1, xb, xa);
        }
    }
    o_out = o;
    l_out = half_swap_sum(lsum);
}

// Again, for a block in which the two functions above ended with a sum out of range: a row's logits lie all below the -1e30 at which their
// maximum starts, or its product with log2 e, which is rounded, is off by more than an exponential holds (from 1e10 on: rows of a pair bias or a mask of
// -1e11 throughout were not numbers).  The true row maxima first, then the logits less these, a difference that is exact where it counts.  Not a hot
// path: one tile at a time, nothing ahead, the pair bias (nbrow: of this lane's query, offset by 16 (lane >> 5)) element by element.
template <bool HAS_NB>
__device__ __forceinline__ void attend_block_far(const uint4 *lds_k, const uint4 *lds_v, const f32x4 *mask4, const bf16_t *nbrow, bf16x8 q0, bf16x8 q1,
                                                 bf16x8 sel0, bf16x8 sel1, int NB, int S, int lane, f32x16 &o_out, float &l_out)
{
    const int g = lane >> 5;
    auto logits = [&](int t) {
        f32x16 x;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const f32x4 mv = mask4[t * 8 + a];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                x[4 * a + c] = mv[c];
            }
        }
        if (HAS_NB) {
            const uint16_t *src = reinterpret_cast<const uint16_t *>(nbrow + t * 32);
            const int key0 = t * 32 + 16 * g;
            uint32_t w[8];
#pragma unroll
            for (int v = 0; v < 8; ++v) {
                const uint32_t a0 = key0 + 2 * v < S ? src[2 * v] : 0u, a1 = key0 + 2 * v + 1 < S ? src[2 * v + 1] : 0u;
                w[v] = a0 | (a1 << 16);
            }
            x = mfma(sel0, as_bf16x8(finite_bias_words(make_uint4(w[0], w[1], w[2], w[3]))), x);
            x = mfma(sel1, as_bf16x8(finite_bias_words(make_uint4(w[4], w[5], w[6], w[7]))), x);
        }
        x = mfma(as_bf16x8(lds_k[(t * 2 + 0) * 64 + lane]), q0, x);
        return mfma(as_bf16x8(lds_k[(t * 2 + 1) * 64 + lane]), q1, x);
    };
    float mx = -INFINITY;
#pragma unroll 1
    for (int t = 0; t < NB; ++t) {
        const f32x16 x = logits(t);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            mx = fmaxf(mx, x[v]);
        }
    }
    mx = half_swap_max(mx);
    f32x16 o = zero16();
    float lsum = 0.f;
    bf16x2 one2;
    one2[0] = (bf16_t)1.0f, one2[1] = (bf16_t)1.0f;
#pragma unroll 1
    for (int t = 0; t < NB; ++t) {
        f32x16 x = logits(t);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            x[v] = __builtin_amdgcn_exp2f((x[v] - mx) * LOG2E);
        }
        const bf16x8 p0 = pack8(x, 0), p1 = pack8(x, 8);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            bf16x2 a, c;
            a[0] = p0[2 * v], a[1] = p0[2 * v + 1];
            c[0] = p1[2 * v], c[1] = p1[2 * v + 1];
            lsum = __builtin_amdgcn_fdot2_f32_bf16(a, one2, lsum, false);
            lsum = __builtin_amdgcn_fdot2_f32_bf16(c, one2, lsum, false);
        }
        o = mfma(as_bf16x8(lds_v[(t * 2 + 0) * 64 + lane]), p0, o);
        o = mfma(as_bf16x8(lds_v[(t * 2 + 1) * 64 + lane]), p1, o);
    }
    o_out = o;
    l_out = half_swap_sum(lsum);
}

// Copies head h's rows of the four weight matrices into LDS in MFMA fragment order.  A unit -- a matrix's 32 rows by 32 channels, two fragments
// -- is two wave-wide loads of half lines, put in order through 2 KB of the LDS that are the wave's own: in fragment order, 16 bytes of another
// row in every lane, a load takes the address path 42 cycles instead of 16.  The unit's index is wave-uniform and the matrix pointer
// is picked with scalar selects (indexing the pointer array per lane made every copy wait for a load of the pointer
// first).  Four units per wave are asked for at once: their round trips overlap instead of queueing (one at a time they were 9 % of
// the long-sequence kernel).  Half lines against fragment order, 256 channels: MSA rows 200 x 200 84.2 -> 83.7 us, columns 128 x 200 52.9 ->
// 52.2, attention of 128 x 256 48.7 -> 48.0; with 128 channels, half as many, no difference.
// ------------------------------------------------------------------------------------------------
template <int C>
__device__ inline void stage_weight_fragments(uint4 *lds_w, uint4 *own, const FusedParams &p, int h, int wave, int nwaves, int lane)
{
    constexpr int CK = C / 16, UNITS = 2 * CK, TOGETHER = 4;
    for (int u0 = wave; u0 < UNITS; u0 += TOGETHER * nwaves) {
        bf16x8 t[TOGETHER][2];
#pragma unroll
        for (int k = 0; k < TOGETHER; ++k) {
            const int u = min(u0 + k * nwaves, UNITS - 1), m = u / (CK / 2);
            const bf16_t *w = m == 0 ? p.w[0] : m == 1 ? p.w[1] : m == 2 ? p.w[2] : p.w[3];
            load_half_lines<2>(t[k], w + (int64_t)h * HEAD * C + u % (CK / 2) * 32, C, lane);
        }
#pragma unroll
        for (int k = 0; k < TOGETHER; ++k) {
            const int u = min(u0 + k * nwaves, UNITS - 1); // (a unit of another wave's once more, the same values)
            half_lines_to_fragments<2>(t[k], own, lane);
            lds_w[2 * u * 64 + lane] = as_uint4(t[k][0]);
            lds_w[(2 * u + 1) * 64 + lane] = as_uint4(t[k][1]);
        }
    }
}

// The same in whole lines, eight rows by 64 channels a copy (in fragment order, a 16-byte piece of another row in every
// lane, a load takes the address path 42 cycles instead of 16, and a workgroup of one unit waits for them all), straight into the LDS: no
// registers, all copies of a wave on their way at once.  Through registers, most copies one after the other, the weights of 77 residues took 1.6 us of
// that kernel's 7; with this and a wave's rows asked for before them the whole block takes 15.8 us, 16.8 before, 96 residues 17.3 and 17.7, 420 160 and
// 164.  A wave's copies follow each other by their scalar instructions: with the matrix chosen for each of them (45 and six branches, now 20 and one) 77 residues
// took 16.1, and rows of 290 and 350 keys with 256 channels (16 x 350 35.5 us, now 35.0) more than through registers (35.1).  A matrix lies as panels of 32 rows x 64 channels (panel_slot); complete when the wave's
// loads are and behind a barrier.
__device__ inline int weight_slot(int lane, int ks) { return (ks >> 2) * 256 + (panel_slot(lane & 31, lane >> 5) ^ (2 * (ks & 3))); }
template <int C>
__device__ inline void stage_weight_lines(uint4 *lds_w, const FusedParams &p, int first, int count, int h, int wave, int nwaves, int lane)
{
    constexpr int CK = C / 16;
    const uint32_t to = (uint32_t)(uintptr_t)(const lds_char *)reinterpret_cast<char *>(lds_w);
    const int rl = lane >> 3;
    uint32_t lane_bytes[2]; // rows 16 - 31 of a panel swizzle with bit 0 flipped
#pragma unroll
    for (int hi = 0; hi < 2; ++hi) {
        lane_bytes[hi] = 2u * (uint32_t)(rl * C + 8 * ((lane & 7) ^ rl ^ hi));
    }
    // the copies of all matrices are dealt to the waves in turn
    for (int i = 0, k = wave; i < count; ++i, k -= CK) {
        const bf16_t *const *at = &p.w[first + i];
        const bf16_t *w = *at + (int64_t)h * HEAD * C;
        for (; k < CK; k += nwaves) {
            load_to_lds(to + (uint32_t)(i * CK + k) * 1024u, w + 8 * (k & 3) * C + (k >> 2) * 64, k & 2 ? lane_bytes[1] : lane_bytes[0]);
        }
    }
    wait_for_loads<0>();
}

// ------------------------------------------------------------------------------------------------
// fused_head_kernel: one workgroup per (b, h) unit
// LDS carve-up, in 16-byte units unless noted:
//   [0, GW*CK*64)               staged weights           [matrix][panel of 64 channels][32 rows x 8 pieces, weight_slot]
//   [.., +NT*2*64)              K fragments              [tile][kstep][lane]
//   [.., +NT*2*64)              V fragments              [tile][kstep][lane]
// The mask of the batch row (floats, -inf past S) and the tile flags are needed only by the attention phase and take
// the place of the weight fragments once the projections are done; every thread fetches its mask values at the start
// and keeps them in registers until then.  At 1024 keys that leaves room for all four weight matrices of a
// 128-channel head (two of a 256-channel one) beside K and V, so the input rows are read once (twice).
// ------------------------------------------------------------------------------------------------
template <int C, int BPW, bool HAS_NB, bool TILES, bool ODD>
__global__ __launch_bounds__(64 * max_waves(C, BPW)) void fused_head_kernel(FusedParams p)
{
    constexpr int CK = C / 16;
    constexpr bool V_ALIAS = C == 256 && BPW == 4; // second LDS layout, below
    constexpr bool ONE_GROUP = V_ALIAS || C == 128; // all four weight matrices staged at once, always (see make_plan)
    constexpr bool ONE_PASS = C == 128 && BPW > 1;  // rows of one mask attended once: see below
    const bool l2mode = TILES || ODD || p.l2mode != 0;
    extern __shared__ uint4 lds[];

    // XCD-aware unit mapping: consecutive workgroup ids land on different XCDs (8 of them), so the H
    // heads of one batch row are placed 8 ids apart and share one XCD's L2 for their reads of x[b].
    const int u = blockIdx.x;
    const int xcd = u & 7;
    const int slot = u >> 3;
    const int h = slot % p.H;
    const int b = (slot / p.H) * 8 + xcd;
    if (b >= p.B) {
        return;
    }
    const int tid = threadIdx.x;
    const int nthreads = p.NW * 64;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6); // uniform, kept in a scalar register
    const int r = lane & 31, g = lane >> 5;
    const int S = p.S, NB = p.NB, NT = p.NT, NW = p.NW, GW = ONE_GROUP ? 4 : p.GW;

    // Second layout (256 channels at the longest sequences, NT == NB): all four weight matrices (64 KB) lie on the V array,
    // whose fragments wait in registers until the projections are done; K, then V / weights, then one 4 KB input panel
    // per wave (the mask's place afterwards).  The input rows are then staged once for all four projections.
    uint4 *lds_w = lds;
    uint4 *lds_k = lds_w + GW * CK * 64;
    uint4 *lds_v = lds_k + NT * 2 * 64;
    uint4 *own_panel = nullptr;
    float *mask = reinterpret_cast<float *>(lds_w);
    if constexpr (V_ALIAS) {
        lds_k = lds, lds_v = lds_k + NT * 2 * 64, lds_w = lds_v;
        uint4 *panels = lds_v + (NT * 2 * 64 > 4 * CK * 64 ? NT * 2 * 64 : 4 * CK * 64); // past the longer of V and weights
        own_panel = panels + wave * 256;
        mask = reinterpret_cast<float *>(panels);
    }
    uint32_t *part_flags = reinterpret_cast<uint32_t *>(mask + NT * 32); // two flag bits per 64 keys and one more unless all have one mask, one word each
    uint4 vpark[V_ALIAS ? BPW : 1][2];

    if (NT > NB) { // phantom key tile: zero K and V fragments (V after the projections when the weights lie there)
        const uint4 z4 = {0u, 0u, 0u, 0u};
        for (int idx = tid; idx < 128; idx += nthreads) {
            lds_k[NB * 2 * 64 + idx] = z4;
            if constexpr (!V_ALIAS) {
                lds_v[NB * 2 * 64 + idx] = z4;
            }
        }
    }
    // wave w holds the mask of keys [64(w + q NW), +64): NT <= 4 NW + 1 tiles are at most 2 NW such parts
    constexpr int MASK_PARTS = (BPW + 1) / 2;
    bf16_t mask_raw[MASK_PARTS];
#pragma unroll
    for (int q = 0; q < MASK_PARTS; ++q) {
        mask_raw[q] = mask_bias_fetch(p.bias + (int64_t)b * p.bias_sb, S, (wave + q * NW) * 64 + lane, p.bias_sk);
    }

    const float qmul = l2mode ? p.qscale * LOG2E : p.qscale;
    // ---- projections, in groups of GW weight matrices staged through LDS ----
    bf16x8 qf[BPW][2];   // Q^T fragments (B operand of the logits MFMA), scaled by 1/sqrt(d)
    bf16x8 gate[BPW][2]; // sigmoid(gate) in accumulator order, packed
    const int npass = ONE_GROUP ? 1 : 4 / GW;
    // With at least two matrices per group K and V (matrices 0 and 1) share a group; the groups are then walked from the
    // last to the first, so that K and V come last and the K/V fragment slots of a block stay free until that block's
    // own results land in them.  That lets the input rows take the coalesced route: a 4 KB staging panel aliased onto
    // the block's K slot (rows 0-15) and V slot (rows 16-31), private to the wave that owns the block.  With one matrix
    // per group there is no such free space (LDS is full at that sequence length) and the fragments are loaded from
    // global memory directly.
    const bool staged_input = ONE_GROUP || GW >= 2;
    const int prow = pi_row(r);
    for (int pi = 0; pi < npass; ++pi) {
        const int pass = staged_input ? npass - 1 - pi : pi;
        if (pi > 0) {
            __syncthreads(); // previous group's fragments are no longer being read
        }
        // One block a wave: its rows and its gate's bias are asked for in front of the weights, one round trip for all (with 256 channels, columns of
        // 500 sequences x 100 lose 1.8 % by it).
        constexpr bool EARLY = BPW == 1 && C == 128;
        PanelRegs early[EARLY ? CK / 4 : 1];
        f32x4 early_bg[EARLY ? 4 : 1];
        if constexpr (EARLY) {
#pragma unroll
            for (int c = 0; c < CK / 4; ++c) {
                early[c] = panel_load(p.x + (int64_t)b * p.x_sb, p.x_ld, min(wave, NB - 1) * 32, S - 1, c * 64, lane);
            }
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                early_bg[a] = *reinterpret_cast<const f32x4 *>(p.bg + h * HEAD + 4 * g + 8 * a);
            }
        }
        stage_weight_lines<C>(lds_w, p, pass * GW, GW, h, wave, NW, lane);
        __syncthreads();
        if constexpr (C == 128 && BPW >= 3) {
            // Two blocks of the wave per walk over the weight fragments: the input fragments of both stay in registers
            // (64 of them) and every fragment of the weights is read from LDS once for the pair (1 KB per MFMA when the
            // blocks are projected one after the other); all rows of a pair are asked for at once.  A pair whose second
            // block does not exist projects the first one twice and stores it once.
#pragma unroll
            for (int i0 = 0; i0 < BPW; i0 += 2) {
                constexpr int PAIR = 2;
                int j0 = wave + i0 * NW;
                if (j0 >= NB) {
                    continue;
                }
                asm volatile("" : "+s"(j0)); // opaque, as below: addresses are formed per pair, not kept across the loop
                const bool second = i0 + 1 < BPW && j0 + NW < NB;
                const bf16_t *xb = p.x + (int64_t)b * p.x_sb;
                bf16x8 xf[PAIR][CK];
                int jn[PAIR];
                jn[0] = j0, jn[1] = second ? j0 + NW : j0;
                PanelRegs t[PAIR][CK / 4];
#pragma unroll
                for (int n = 0; n < PAIR; ++n) {
#pragma unroll
                    for (int c = 0; c < CK / 4; ++c) {
                        t[n][c] = panel_load_near(xb + c * 64, (uint32_t)p.x_ld, jn[n] * 32, S - 1, 0, lane);
                    }
                }
#pragma unroll
                for (int n = 0; n < PAIR; ++n) {
                    const int j = jn[n];
                    uint4 *kslot = lds_k + j * 128, *vslot = lds_v + j * 128 - 128; // panel slots 0-127 and 128-255
                    const uint4 *fsrc = prow < 16 ? kslot : vslot;
                    const int srow8 = lane >> 3, chunk = lane & 7;
#pragma unroll
                    for (int c = 0; c < CK / 4; ++c) {
                        kslot[panel_slot(srow8, chunk)] = t[n][c].r0;
                        kslot[panel_slot(srow8 + 8, chunk)] = t[n][c].r1;
                        vslot[panel_slot(srow8 + 16, chunk)] = t[n][c].r2;
                        vslot[panel_slot(srow8 + 24, chunk)] = t[n][c].r3;
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            xf[n][4 * c + k] = as_bf16x8(fsrc[panel_slot(prow, 2 * k + g)]);
                        }
                    }
                }
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const uint4 *wsrc = lds_w + m * CK * 64;
                    f32x16 acc[PAIR];
                    acc[0] = zero16(), acc[1] = zero16();
#pragma unroll
                    for (int ks = 0; ks < CK; ++ks) {
                        const bf16x8 wf = as_bf16x8(wsrc[weight_slot(lane, ks)]);
#pragma unroll
                        for (int n = 0; n < PAIR; ++n) {
                            // V[s][d]: rows = sequence positions; the others W_h . x^T: rows = head-dim
                            acc[n] = m == PROJ_V ? mfma(xf[n][ks], wf, acc[n]) : mfma(wf, xf[n][ks], acc[n]);
                        }
                    }
#pragma unroll
                    for (int n = 0; n < PAIR; ++n) {
                        if (n == 1 && i0 + 1 >= BPW) {
                            continue;
                        }
                        const int i = i0 + n;
                        if (m == PROJ_V) {
                            if (n == 0 || second) {
                                lds_v[(jn[n] * 2 + 0) * 64 + lane] = as_uint4(pack8(acc[n], 0));
                                lds_v[(jn[n] * 2 + 1) * 64 + lane] = as_uint4(pack8(acc[n], 8));
                            }
                        } else if (m == PROJ_K) {
                            if (n == 0 || second) {
                                lds_k[(jn[n] * 2 + 0) * 64 + lane] = as_uint4(pack8(acc[n], 0));
                                lds_k[(jn[n] * 2 + 1) * 64 + lane] = as_uint4(pack8(acc[n], 8));
                            }
                        } else if (m == PROJ_Q) {
#pragma unroll
                            for (int v = 0; v < 16; ++v) {
                                acc[n][v] *= qmul;
                            }
                            qf[i][0] = pack8(acc[n], 0);
                            qf[i][1] = pack8(acc[n], 8);
                        } else {
                            const float *bgp = p.bg + h * HEAD + 4 * g;
#pragma unroll
                            for (int a = 0; a < 4; ++a) {
                                const f32x4 bv = *reinterpret_cast<const f32x4 *>(bgp + 8 * a);
#pragma unroll
                                for (int c = 0; c < 4; ++c) {
                                    acc[n][4 * a + c] = sigmoid_fast(acc[n][4 * a + c] + bv[c]);
                                }
                            }
                            gate[i][0] = pack8(acc[n], 0);
                            gate[i][1] = pack8(acc[n], 8);
                        }
                    }
                }
            }
        } else {
#pragma unroll
        for (int i = 0; i < BPW; ++i) {
            int j = wave + i * NW;
            if (j >= NB) {
                continue;
            }
            // Opaque to the optimiser: otherwise the row addresses of every block of the wave are computed once, ahead
            // of the loop over the groups, and with three or four blocks of 256-channel rows they no longer fit the
            // registers -- each spilled address then costs a scratch round trip in front of the load it feeds.
            asm volatile("" : "+s"(j));
            bf16x8 xf[CK];
            if (staged_input) {
                const bf16_t *xb = p.x + (int64_t)b * p.x_sb;
                uint4 *kslot = lds_k + j * 128, *vslot = lds_v + j * 128 - 128; // panel slots 0-127 and 128-255
                if constexpr (V_ALIAS) {
                    kslot = vslot = own_panel;
                }
                const uint4 *fsrc = prow < 16 ? kslot : vslot;
                const int srow8 = lane >> 3, chunk = lane & 7;
                PanelRegs t;
                if constexpr (!EARLY) {
                    t = panel_load(xb, p.x_ld, j * 32, S - 1, 0, lane);
                }
#pragma unroll
                for (int c = 0; c < CK / 4; ++c) {
                    if constexpr (EARLY) {
                        t = early[c];
                    }
                    kslot[panel_slot(srow8, chunk)] = t.r0;
                    kslot[panel_slot(srow8 + 8, chunk)] = t.r1;
                    vslot[panel_slot(srow8 + 16, chunk)] = t.r2;
                    vslot[panel_slot(srow8 + 24, chunk)] = t.r3;
                    if (!EARLY && c + 1 < CK / 4) {
                        t = panel_load(xb, p.x_ld, j * 32, S - 1, (c + 1) * 64, lane);
                    }
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        xf[4 * c + k] = as_bf16x8(fsrc[panel_slot(prow, 2 * k + g)]);
                    }
                }
            } else {
                int srow = j * 32 + prow;
                srow = srow < S ? srow : S - 1; // rows past the end repeat the last row; they are never stored
                const bf16_t *xrow = p.x + (int64_t)b * p.x_sb + (int64_t)srow * p.x_ld + g * 8;
#pragma unroll
                for (int ks = 0; ks < CK; ++ks) {
                    xf[ks] = as_bf16x8(*reinterpret_cast<const uint4 *>(xrow + ks * 16));
                }
            }
            for (int mm = 0; mm < GW; ++mm) {
                const int m = pass * GW + mm;
                const uint4 *wsrc = lds_w + mm * CK * 64;
                f32x16 acc = zero16();
                if (m == PROJ_V) {
                    // V[s][d]: rows = sequence positions, so a lane ends up with 16 keys of one head-dim
#pragma unroll
                    for (int ks = 0; ks < CK; ++ks) {
                        acc = mfma(xf[ks], as_bf16x8(wsrc[weight_slot(lane, ks)]), acc);
                    }
                    if constexpr (V_ALIAS) {
                        vpark[i][0] = as_uint4(pack8(acc, 0));
                        vpark[i][1] = as_uint4(pack8(acc, 8));
                    } else {
                        lds_v[(j * 2 + 0) * 64 + lane] = as_uint4(pack8(acc, 0));
                        lds_v[(j * 2 + 1) * 64 + lane] = as_uint4(pack8(acc, 8));
                    }
                } else {
                    // W_h . x^T: rows = head-dim, columns = sequence positions
#pragma unroll
                    for (int ks = 0; ks < CK; ++ks) {
                        acc = mfma(as_bf16x8(wsrc[weight_slot(lane, ks)]), xf[ks], acc);
                    }
                    if (m == PROJ_K) {
                        lds_k[(j * 2 + 0) * 64 + lane] = as_uint4(pack8(acc, 0));
                        lds_k[(j * 2 + 1) * 64 + lane] = as_uint4(pack8(acc, 8));
                    } else if (m == PROJ_Q) {
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            acc[v] *= qmul;
                        }
                        qf[i][0] = pack8(acc, 0);
                        qf[i][1] = pack8(acc, 8);
                    } else {
                        const float *bgp = p.bg + h * HEAD + 4 * g;
#pragma unroll
                        for (int a = 0; a < 4; ++a) {
                            const f32x4 bv = EARLY ? early_bg[EARLY ? a : 0] : *reinterpret_cast<const f32x4 *>(bgp + 8 * a);
#pragma unroll
                            for (int c = 0; c < 4; ++c) {
                                acc[4 * a + c] = sigmoid_fast(acc[4 * a + c] + bv[c]);
                            }
                        }
                        gate[i][0] = pack8(acc, 0);
                        gate[i][1] = pack8(acc, 8);
                    }
                }
            }
        }
        } // one block at a time
    }
    __syncthreads(); // K and V of the whole sequence are in LDS; the weight fragments are no longer read
    if constexpr (V_ALIAS) {
#pragma unroll
        for (int i = 0; i < BPW; ++i) {
            const int j = wave + i * NW;
            if (j < NB) {
                lds_v[(j * 2 + 0) * 64 + lane] = vpark[i][0];
                lds_v[(j * 2 + 1) * 64 + lane] = vpark[i][1];
            }
        }
        if (NT > NB && tid < 128) {
            lds_v[NB * 2 * 64 + tid] = uint4{0u, 0u, 0u, 0u};
        }
    }
#pragma unroll
    for (int q = 0; q < MASK_PARTS; ++q) {
        const int part = wave + q * NW;
        if (part * 64 < NT * 32) {
            const float mv = mask_bias_finish(mask_raw[q], part * 64 + lane < S, l2mode ? LOG2E : 1.0f, p.bias_is_mask != 0);
            mask[part * 64 + lane] = mv;
            // (in log2 units the copies of the pair bias take keys past the end out by themselves)
            const unsigned long long nz = __ballot(mv != 0.f && (part * 64 + lane < S || !HAS_NB || !l2mode));
            const bool differ = ONE_PASS && __any(part * 64 + lane < S && (mv == 0.f || mv != __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(mv)))));
            if (lane == 0) {
                part_flags[part] = ((uint32_t)nz != 0u ? 1u : 0u) | ((uint32_t)(nz >> 32) != 0u ? 2u : 0u) | (differ ? 4u : 0u);
            }
        }
    }
    __syncthreads();

    // ---- attention: each wave walks the key tiles for its own query blocks ----
    uint32_t flags = 0; // bit t: key tile t needs the mask added (a non-zero one; past the end only where no copy of the pair bias takes those keys out)
    uint32_t differ = 0;
    for (int part = 0; part * 64 < NT * 32; ++part) {
        flags |= (ONE_PASS ? part_flags[part] & 3u : part_flags[part]) << (2 * part);
        differ |= part_flags[part] & 4u;
    }
    // A row whose keys all have one mask (a padded residue's: -1e9 everywhere) would end with every exponential at zero: its logits are
    // taken against that mask, which absorbs in each sum what it absorbs in the reference; with 128 channels and several blocks a wave from the start.  Such
    // rows used to be attended three times (triangle attention of 450 residues, 5 % of them padding, whole block 218 -> 203 us, 203 without
    // padding).  With 256 channels (columns of 501 sequences x 91 95.6 -> 96.9), with one block a wave, and in persistent_head_kernel, the choice in front of the loops slows rows without such a mask
    // (77 residues 22.0 -> 22.15 us, 320 74.4 -> 77.9); there the first pass is made in vain (128 residues 22.9 -> 22.3, 320 85.0 -> 83.3).
    // persistent_pair_kernel, which has no register for a choice in front of its loop (three more spilled: the operator at 384 residues 88.1 -> 89.5), makes
    // that first pass in vain too, and repeats such a row with its one mask.
    constexpr uint32_t ONE_MASK = 2;
    if (ONE_PASS && l2mode && flags != 0u) { // whose loops know no mask, masks, and one mask
        flags = differ == 0u && one_mask_of(mask, S, lane) != 0.f ? ONE_MASK : 1u;
    }
    const f32x4 *mask4 = reinterpret_cast<const f32x4 *>(mask + 16 * g);
    // one pair of selector fragments, as bits: fp16 ones for the log2-unit loop (fp16 pair-bias fragments), bf16 ones otherwise
    uint4 selw0, selw1;
    if (l2mode) {
        f16x8 a, b;
        make_selectors_f16(lane, a, b);
        selw0 = as_uint4(a), selw1 = as_uint4(b);
    } else {
        bf16x8 a, b;
        make_selectors(lane, a, b);
        selw0 = as_uint4(a), selw1 = as_uint4(b);
    }
    const bf16x8 sumsel = rowsum_selector(lane);

#pragma unroll
    for (int i = 0; i < BPW; ++i) {
        const int j = wave + i * NW;
        if (j >= NB) {
            continue;
        }
        const int qpos = j * 32 + pi_row(r);
        const int qrow = qpos < S ? qpos : S - 1;
        f32x16 o;
        float l;
        if (l2mode) {
            const uint4 *nbf = HAS_NB ? p.nbf + ((int64_t)(h * NB + j) * NT * (TILES ? 4 : 2)) * 64 + lane : nullptr;
            bool again = true; // some probability overflowed or a whole row underflowed
            if (!ONE_PASS || flags != ONE_MASK) {
                if ((HAS_NB || !ODD) && flags == 0u) { // (without a pair bias the tile of zeros behind an odd number has a mask)
                    attend_block_l2<HAS_NB, false, false, TILES, ODD>(lds_k, lds_v, mask4, nbf, qf[i][0], qf[i][1], as_f16x8(selw0), as_f16x8(selw1), sumsel,
                                                          NT, lane, 0.f, o, l, (wave >> 2) & 1);
                } else {
                    attend_block_l2<HAS_NB, true, false, TILES, ODD>(lds_k, lds_v, mask4, nbf, qf[i][0], qf[i][1], as_f16x8(selw0), as_f16x8(selw1), sumsel,
                                                         NT, lane, 0.f, o, l, (wave >> 2) & 1);
                }
                __builtin_amdgcn_s_setprio(0);
                again = __any(!(l > 1e-30f && l < 1e30f));
            }
            float shift = again ? one_mask_of(mask, S, lane) : 0.f;
            while (again) { // shifted by the row's one mask, if it has one, or by the true row maxima
                const bool maxima = shift == 0.f;
                if (maxima) {
                    shift = row_max_l2<HAS_NB, TILES>(lds_k, mask4, nbf, qf[i][0], qf[i][1], as_f16x8(selw0), as_f16x8(selw1), NT, lane);
                }
                attend_block_l2<HAS_NB, true, true, TILES>(lds_k, lds_v, mask4, nbf, qf[i][0], qf[i][1], as_f16x8(selw0), as_f16x8(selw1), sumsel, NT,
                                                    lane, shift, o, l);
                again = !maxima && __any(!(l > 1e-30f && l < 1e30f));
                shift = 0.f;
            }
        } else {
            const bf16_t *nbrow = HAS_NB ? p.nb + (int64_t)h * p.nb_sh + (int64_t)qrow * p.nb_sq + 16 * g : nullptr;
            attend_block_direct<HAS_NB>(lds_k, lds_v, mask4, flags, nbrow, p.nb_vec != 0, qf[i][0], qf[i][1], as_bf16x8(selw0), as_bf16x8(selw1), NB,
                                        S, lane, o, l);
            if (__any(!(l > 1e-30f && l < 1e30f))) {
                attend_block_far<HAS_NB>(lds_k, lds_v, mask4, nbrow, qf[i][0], qf[i][1], as_bf16x8(selw0), as_bf16x8(selw1), NB, S, lane, o, l);
            }
        }
        if (qpos < S) {
            f32x16 gv;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                gv[v] = to_f32(gate[i][v >> 3][v & 7]);
            }
            store_gated(p.avg + (int64_t)b * p.avg_sb + (int64_t)qpos * p.avg_ss + (int64_t)h * p.avg_sh + 4 * g, o,
                        __builtin_amdgcn_rcpf(l), gv);
        }
    }
}

// ------------------------------------------------------------------------------------------------
// persistent_head_kernel: one workgroup per CU keeps one head for its lifetime and walks batch rows;
// wave j owns sequence block j (its K/V projection and its 32 queries).  Compared with one workgroup
// per (b, h) unit this stages the head's weights once, pays no workgroup launch per unit, and moves
// the two big streams -- input rows and pair bias -- through wave-private staging panels with fully
// coalesced loads.
// LDS, 16-byte units: W[4][CK][64]  K[NB][2][64]  V[NB][2][64]  panel[NB waves][256]  gate[NB waves][2][64];
// then floats mask[2][NB*32] and two uint32 of tile flags (both alternating by batch row).
// Per batch row: load and project (K, V, Q -> registers; gate -> LDS), barrier (previous row's attention
// is over everywhere), K and V -> LDS, barrier, attend.  A wave that finishes its attention early starts
// on the next row's loads and projections while the slower waves of its SIMD still attend, so the
// latency- and MFMA-bound projection phase overlaps the VALU-heavy attention phase.
// ------------------------------------------------------------------------------------------------
template <int C, bool HAS_NB, bool L2MODE, bool FUSED_LN, bool TILES, bool ODD>
__global__ __launch_bounds__(64 * max_waves(C, 1)) void persistent_head_kernel(FusedParams p)
{
    constexpr int CK = C / 16;
    constexpr int NP = CK / 4; // staging panels (64 channels each) per input row block
    extern __shared__ uint4 lds[];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6); // uniform: values derived from it stay in scalar registers
    const int r = lane & 31, g = lane >> 5;
    const int S = p.S, NB = p.NB, NT = p.NT;
    const int nthreads = NB * 64;
    const int prow = pi_row(r);

    // workgroup -> (XCD, head, batch-row group): the H workgroups that share a batch-row sequence sit
    // on the same XCD (ids 8 apart) and walk it in step, so x[b] is read from HBM once per XCD
    const int w = blockIdx.x;
    const int xcd = w & 7;
    const int slot = w >> 3;
    const int h = slot % p.H;
    const int grp = slot / p.H;
    const int b0 = xcd + 8 * grp;
    const int bstep = 8 * p.ngrp;
    const int nrows = b0 < p.B ? (p.B - b0 + bstep - 1) / bstep : 0;

    uint4 *lds_w = lds;
    uint4 *lds_k = lds_w + 4 * CK * 64;
    uint4 *lds_v = lds_k + NT * 2 * 64;
    uint4 *panel = lds_v + NT * 2 * 64 + wave * 256;
    uint4 *gate_park_base = lds_v + NT * 2 * 64 + NB * 256 + wave * 128; // sigmoid(gate) waits here during attention
    float *mask_base = reinterpret_cast<float *>(lds_v + NT * 2 * 64 + NB * 256 + NB * 128); // two buffers of NT*32
    uint32_t *flag_words = reinterpret_cast<uint32_t *>(mask_base + 2 * NT * 32);            // two, alternating by batch row

    // the head's rows of the four weight matrices, in fragment order, for the whole kernel
    stage_weight_fragments<C>(lds_w, panel, p, h, wave, nthreads >> 6, lane);
    if (tid == 0) {
        flag_words[0] = 0;
        flag_words[1] = 0;
    }
    if (NT > NB) { // phantom key tile: zero K and V fragments, never written again
        const uint4 z4 = {0u, 0u, 0u, 0u};
        for (int idx = tid; idx < 128; idx += nthreads) {
            lds_k[NB * 2 * 64 + idx] = z4;
            lds_v[NB * 2 * 64 + idx] = z4;
        }
    }
    std::conditional_t<L2MODE, f16x8, bf16x8> sel0, sel1; // fp16 ones for the log2-unit loop, whose pair-bias fragments are fp16
    if constexpr (L2MODE) {
        make_selectors_f16(lane, sel0, sel1);
    } else {
        make_selectors(lane, sel0, sel1);
    }
    __syncthreads();

    const int j = wave; // this wave's sequence block
    // With three waves per SIMD (128 channels) the waves take turns at the issue priorities during the attention; with two
    // (256 channels) the arbiter's own order measured 2 % faster.
    const int fair_turn = C == 128 ? wave >> 2 : -1;
    const float qmul = L2MODE ? p.qscale * LOG2E : p.qscale;
    const float mask_scale = L2MODE ? LOG2E : 1.0f;
    const bf16x8 sumsel = rowsum_selector(lane);
    for (int n = 0; n < nrows; ++n) {
        const int b = b0 + n * bstep;
        uint32_t *flag_word = flag_words + (n & 1);
        float *mask = mask_base + (n & 1) * NT * 32;
        // The lane index is opaque to the optimiser here: the row addresses and panel offsets derived from it are then
        // formed anew for every batch row (a few dozen vector instructions) instead of being kept across the attention
        // loop, where there is no register for them -- spilled, each costs a scratch round trip per batch row.
        int lane_x = lane;
        asm volatile("" : "+v"(lane_x));
        // (in log2 units the copies of the pair bias take keys past the end out by themselves)
        stage_mask_part<true>(p.bias + (int64_t)b * p.bias_sb, mask, flag_word, S, NT, HAS_NB && L2MODE ? S : NT * 32, wave, lane_x, mask_scale, p.bias_sk,
                              p.bias_is_mask != 0);

        // ---- input rows of the block -> fragments, 64 channels per staging panel ----
        const int prow_x = pi_row(lane_x & 31), g_x = lane_x >> 5;
        const bf16_t *xb = p.x + (int64_t)b * p.x_sb;
        const uint32_t x_pitch = (uint32_t)p.x_ld; // the host sends only near-addressable rows here
        bf16x8 xf[CK];
        if constexpr (FUSED_LN) {
            // The rows arrive un-normalised and are normalised between their load and their staging (arithmetic of
            // reference src/normalization/layernorm_kernel.h:21-53, result rounded to bf16 as the tensor it replaces
            // was).  A lane holds 8 channels per panel of four rows; a row's C channels sit in the 8 lanes that loaded
            // it, so its two sums cross three DPP steps.
            PanelRegs t[NP];
#pragma unroll
            for (int c = 0; c < NP; ++c) {
                t[c] = panel_load_near(xb + c * 64, x_pitch, j * 32, S - 1, 0, lane_x);
            }
            float gm[NP][8], bt[NP][8];
#pragma unroll
            for (int c = 0; c < NP; ++c) {
                const float *gsrc = p.ln_gamma + c * 64 + (lane_x & 7) * 8, *bsrc = p.ln_beta + c * 64 + (lane_x & 7) * 8;
#pragma unroll
                for (int e = 0; e < 8; e += 4) {
                    const f32x4 gv = *reinterpret_cast<const f32x4 *>(gsrc + e), bv = *reinterpret_cast<const f32x4 *>(bsrc + e);
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        gm[c][e + k] = gv[k], bt[c][e + k] = bv[k];
                    }
                }
            }
            auto normalise_row = [&](uint4 (&words)[NP]) {
                float v[NP][8];
#pragma unroll
                for (int c = 0; c < NP; ++c) {
                    const bf16x8 in = as_bf16x8(words[c]);
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        v[c][e] = to_f32(in[e]);
                    }
                }
                const float x0 = __shfl(v[0][0], lane_x & ~7, 64); // first element of the row
                float s1 = 0.f, s2 = 0.f;
#pragma unroll
                for (int c = 0; c < NP; ++c) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float d = v[c][e] - x0;
                        s1 += d;
                        s2 = fmaf(d, d, s2);
                    }
                }
                float rstd, shift;
                norm_from_sums<false>(group_sum<8>(s1), group_sum<8>(s2), x0, (float)C, p.ln_eps, rstd, shift); // as the row kernels form it
#pragma unroll
                for (int c = 0; c < NP; ++c) {
                    bf16x8 o;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        o[e] = (bf16_t)fmaf(fmaf(v[c][e], rstd, shift), gm[c][e], bt[c][e]);
                    }
                    words[c] = as_uint4(o);
                }
            };
            {
                uint4 w0[NP], w1[NP], w2[NP], w3[NP];
#pragma unroll
                for (int c = 0; c < NP; ++c) {
                    w0[c] = t[c].r0, w1[c] = t[c].r1, w2[c] = t[c].r2, w3[c] = t[c].r3;
                }
                normalise_row(w0), normalise_row(w1), normalise_row(w2), normalise_row(w3);
#pragma unroll
                for (int c = 0; c < NP; ++c) {
                    t[c].r0 = w0[c], t[c].r1 = w1[c], t[c].r2 = w2[c], t[c].r3 = w3[c];
                }
            }
#pragma unroll
            for (int c = 0; c < NP; ++c) {
                panel_store(panel, lane_x, t[c]);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    xf[4 * c + k] = as_bf16x8(panel[panel_slot(prow_x, 2 * k + g_x)]);
                }
            }
        } else {
            PanelRegs ta, tb;
            ta = panel_load_near(xb, x_pitch, j * 32, S - 1, 0, lane_x);
#pragma unroll
            for (int c = 0; c < NP; c += 2) {
                if (c + 1 < NP) {
                    tb = panel_load_near(xb + (c + 1) * 64, x_pitch, j * 32, S - 1, 0, lane_x);
                }
                panel_store(panel, lane_x, ta);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    xf[4 * c + k] = as_bf16x8(panel[panel_slot(prow_x, 2 * k + g_x)]);
                }
                if (c + 1 < NP) {
                    if (c + 2 < NP) {
                        ta = panel_load_near(xb + (c + 2) * 64, x_pitch, j * 32, S - 1, 0, lane_x);
                    }
                    panel_store(panel, lane_x, tb);
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        xf[4 * (c + 1) + k] = as_bf16x8(panel[panel_slot(prow_x, 2 * k + g_x)]);
                    }
                }
            }
        }
        // ---- four projections of the block ----
        bf16x8 q0, q1;
        uint4 kfrag0, kfrag1, vfrag0, vfrag1; // this block's K and V fragments, parked until the LDS arrays are free
        {
            uint4 *gate_park_x = gate_park_base + lane_x;
            const uint4 *wsrc = lds_w + lane_x;
            f32x16 acc = zero16();
#pragma unroll
            for (int ks = 0; ks < CK; ++ks) {
                acc = mfma(as_bf16x8(wsrc[(PROJ_K * CK + ks) * 64]), xf[ks], acc);
            }
            kfrag0 = as_uint4(pack8(acc, 0));
            kfrag1 = as_uint4(pack8(acc, 8));
            acc = zero16();
#pragma unroll
            for (int ks = 0; ks < CK; ++ks) {
                acc = mfma(xf[ks], as_bf16x8(wsrc[(PROJ_V * CK + ks) * 64]), acc);
            }
            vfrag0 = as_uint4(pack8(acc, 0));
            vfrag1 = as_uint4(pack8(acc, 8));
            acc = zero16();
#pragma unroll
            for (int ks = 0; ks < CK; ++ks) {
                acc = mfma(as_bf16x8(wsrc[(PROJ_Q * CK + ks) * 64]), xf[ks], acc);
            }
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                acc[v] *= qmul;
            }
            q0 = pack8(acc, 0);
            q1 = pack8(acc, 8);
            // the gate's accumulator starts at its bias (register v of a lane holds feature 8 (v / 4) + 4 g + v % 4)
            const float *bgp = p.bg + h * HEAD + 4 * g_x;
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const f32x4 bv = *reinterpret_cast<const f32x4 *>(bgp + 8 * a);
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    acc[4 * a + c] = bv[c];
                }
            }
#pragma unroll
            for (int ks = 0; ks < CK; ++ks) {
                acc = mfma(as_bf16x8(wsrc[(PROJ_G * CK + ks) * 64]), xf[ks], acc);
            }
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                acc[v] = sigmoid_fast(acc[v]);
            }
            gate_park_x[0] = as_uint4(pack8(acc, 0));
            gate_park_x[64] = as_uint4(pack8(acc, 8));
        }
        __syncthreads(); // every wave is done with the previous row's attention: the K and V arrays are free
        lds_k[(j * 2 + 0) * 64 + lane] = kfrag0;
        lds_k[(j * 2 + 1) * 64 + lane] = kfrag1;
        lds_v[(j * 2 + 0) * 64 + lane] = vfrag0;
        lds_v[(j * 2 + 1) * 64 + lane] = vfrag1;
        if (tid == 0) {
            flag_words[(n + 1) & 1] = 0; // its readers (previous row) are done, its writers (next row) start after the next barrier
        }
        __syncthreads(); // K, V and the mask of this batch row are complete

        const f32x4 *mask4 = reinterpret_cast<const f32x4 *>(mask + 16 * g);
        f32x16 o;
        float l;
        const uint32_t flags = *flag_word;
        const bf16_t *nb_head = HAS_NB ? p.nb + (int64_t)h * p.nb_sh : nullptr;
        if constexpr (L2MODE) {
            const uint4 *nbf = HAS_NB ? p.nbf + ((int64_t)(h * NB + j) * NT * (TILES ? 4 : 2)) * 64 + lane : nullptr;
            if ((HAS_NB || !ODD) && flags == 0u) { // (without a pair bias the tile of zeros behind an odd number has a mask)
                attend_block_l2<HAS_NB, false, false, TILES, ODD>(lds_k, lds_v, mask4, nbf, q0, q1, sel0, sel1, sumsel, NT, lane, 0.f, o,
                                                      l, -1, fair_turn);
            } else {
                attend_block_l2<HAS_NB, true, false, TILES, ODD>(lds_k, lds_v, mask4, nbf, q0, q1, sel0, sel1, sumsel, NT, lane, 0.f, o,
                                                     l, -1, fair_turn);
            }
            // some probability overflowed or a whole row underflowed: shift by the row's one mask, if it has one, or by the true row maxima
            float shift = __any(!(l > 1e-30f && l < 1e30f)) ? one_mask_of(mask, S, lane) : 0.f;
            while (__any(!(l > 1e-30f && l < 1e30f))) {
                const bool maxima = shift == 0.f;
                if (maxima) {
                    shift = row_max_l2<HAS_NB, TILES>(lds_k, mask4, nbf, q0, q1, sel0, sel1, NT, lane);
                }
                attend_block_l2<HAS_NB, true, true, TILES>(lds_k, lds_v, mask4, nbf, q0, q1, sel0, sel1, sumsel, NT, lane, shift, o, l);
                if (maxima) {
                    break;
                }
                shift = 0.f;
            }
        } else {
            attend_block<HAS_NB>(lds_k, lds_v, mask4, flags, nb_head, p.nb_sq, j * 32, p.nb_vec != 0, panel, q0, q1, sel0,
                                 sel1, NB, S, lane, o, l);
            if (__any(!(l > 1e-30f && l < 1e30f))) {
                const bf16_t *nbrow = HAS_NB ? nb_head + (int64_t)min(j * 32 + prow, S - 1) * p.nb_sq + 16 * g : nullptr;
                attend_block_far<HAS_NB>(lds_k, lds_v, mask4, nbrow, q0, q1, sel0, sel1, NB, S, lane, o, l);
            }
        }
        int lane_o = lane; // as above: the addresses of the epilogue are not worth a register during the attention loop
        asm volatile("" : "+v"(lane_o));
        const int qpos = j * 32 + pi_row(lane_o & 31);
        if (qpos < S) {
            const uint4 *gate_park_o = gate_park_base + lane_o;
            const bf16x8 gate0 = as_bf16x8(gate_park_o[0]), gate1 = as_bf16x8(gate_park_o[64]);
            f32x16 gv;
#pragma unroll
            for (int v = 0; v < 8; ++v) {
                gv[v] = to_f32(gate0[v]);
                gv[8 + v] = to_f32(gate1[v]);
            }
            store_gated(p.avg + (int64_t)b * p.avg_sb + (int64_t)qpos * p.avg_ss + (int64_t)h * p.avg_sh + 4 * (lane_o >> 5), o,
                        __builtin_amdgcn_rcpf(l), gv);
        }
    }
}

// ------------------------------------------------------------------------------------------------
// persistent_pair_kernel: persistent_head_kernel walking its batch rows two at a time (128 or 256 channels, log2 units).
// The pair bias of a (head, query block, key tile) is the same for every batch row, so a wave that attends the same query
// block of two rows at once fetches it once -- as fp32, in accumulator order, straight into the C operand of the logits
// MFMAs of both rows (pair_bias_tiles_kernel writes that copy).  Per row and key tile this moves the same bytes as the
// fp16 fragments of persistent_head_kernel and takes the two selector MFMAs out of the loop (matrix pipe 224 -> 160 clocks
// per tile); the two rows' instruction streams are independent, which gives the scheduler what a fourth wave per SIMD
// would; and every weight fragment read from LDS in the projection phase serves two rows.
// LDS, 16-byte units: W[4][CK][64]  K[2 rows][NT][2][64]  V[2 rows][NT][2][64]  panel[NB waves][128];
// then mask words mask[2 pairs in flight][2 rows][NT*32] (a key's mask bias as two bf16: the rows' masks enter the logits
// by one more MFMA per tile, see stage_mask_words) and four uint32 of tile flags.  At 128 channels and 384 positions that
// is 32 + 96 + 24 + 6 KB, at 256 channels and 256 positions 64 + 64 + 16 + 4 KB: the panels are half the size of
// persistent_head_kernel's (32 rows x 32 channels); during the attention a wave's panel holds the sigmoid of the first
// row's gate, the second row's waits in eight registers.
// ------------------------------------------------------------------------------------------------

// Wave-private 2 KB staging panel: 32 rows x 64 bytes in 16-byte slots, filled with two coalesced loads (lane l -> row
// l / 4 + 16 i, chunk l % 4) and read back in MFMA fragment order; the chunk index is XOR-swizzled by row so that both
// access patterns are free of LDS bank conflicts.
__device__ __forceinline__ int panel32_slot(int row, int chunk) { return row * 4 + (chunk ^ (((row >> 2) & 1) | (((row >> 4) & 1) << 1))); }

struct Panel32Regs {
    uint4 r0, r1;
};

// rows row0 .. row0 + 31 (clamped to last_row) of a row-major bf16 matrix, 32 columns from col0; 32-bit byte offsets from
// a wave-uniform base as in panel_load_near
__device__ __forceinline__ Panel32Regs panel32_load_near(const bf16_t *base, uint32_t ld, int row0, int last_row, int col0, int lane)
{
    const char *bytes = reinterpret_cast<const char *>(base);
    const uint32_t pitch = 2u * ld;
    const uint32_t col = 2u * (uint32_t)col0 + 16u * (uint32_t)(lane & 3);
    const uint32_t last = (uint32_t)last_row * pitch + col;
    const uint32_t first = __umul24((uint32_t)(row0 + (lane >> 2)), pitch) + col;
    Panel32Regs p;
    p.r0 = *reinterpret_cast<const uint4 *>(bytes + min(first, last));
    p.r1 = *reinterpret_cast<const uint4 *>(bytes + min(first + 16u * pitch, last));
    return p;
}

__device__ __forceinline__ void panel32_store(uint4 *panel, int lane, const Panel32Regs &p)
{
    const int row = lane >> 2, chunk = lane & 3;
    panel[panel32_slot(row, chunk)] = p.r0;
    panel[panel32_slot(row + 16, chunk)] = p.r1;
}

// Pair bias [H, S, S] -> fp32 tiles in accumulator order, in log2 units: for head h, query block j and key tile t,
// [h][j][t][4][64 lanes] x 16 bytes; lane (r, g) holds keys 32 t + 16 g .. + 15 of query 32 j + pi(r), four per 16-byte
// piece -- registers 4 a .. 4 a + 3 of the logits accumulator.  Queries past S repeat row S - 1, keys past S are at
// LOWEST_BIAS, and so are entries below it (-inf): a row of them still has a
// finite maximum.
__global__ __launch_bounds__(64) void pair_bias_tiles_kernel(const bf16_t *__restrict__ nb, int64_t nb_sh, int64_t nb_sq, int S,
                                                             int NB, int NT, int vec, f32x4 *__restrict__ out)
{
    const int lane = threadIdx.x;
    const int r = lane & 31, g = lane >> 5;
    const int t = blockIdx.x % NT, j = blockIdx.x / NT, h = blockIdx.y;
    int q = 32 * j + pi_row(r);
    q = q < S ? q : S - 1;
    const int key0 = 32 * t + 16 * g;
    const bf16_t *src = nb + (int64_t)h * nb_sh + (int64_t)q * nb_sq + key0;
    float v[16];
    if (vec && key0 + 16 <= S) {
        const bf16x8 s0 = as_bf16x8(*reinterpret_cast<const uint4 *>(src)), s1 = as_bf16x8(*reinterpret_cast<const uint4 *>(src + 8));
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            v[e] = to_f32(s0[e]), v[8 + e] = to_f32(s1[e]);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            v[e] = key0 + e < S ? to_f32(src[e]) : LOWEST_BIAS;
        }
    }
    f32x4 *dst = out + ((((int64_t)h * NB + j) * NT + t) * 4) * 64 + lane;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        f32x4 o;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float x = v[4 * a + c] * LOG2E;
            o[c] = x < LOWEST_BIAS ? LOWEST_BIAS : x; // a comparison, not a max: a NaN stays a NaN
        }
        dst[a * 64] = o;
    }
}

// Attention of one 32-query block of two batch rows A and B (same head) in log2 units; see attend_block_l2 for the
// formulation.  Tiles are walked A(0) B(0) A(1) B(1) ...: while the softmax and P.V of one (row, tile) run on the vector
// ALU, the logits MFMAs of the next one are in the matrix pipe.
//   lds_kA/vA/kB/vB : K and V fragments of the two rows, [tile][kstep][lane]
//   mwA / mwB       : mask bias of the rows (log2 units) as hi/lo bf16 words (stage_mask_words), offset by the key the
//                     lane's accumulator row stands for; one more MFMA per tile adds them (WITH_MASK only)
//   nbc             : fp32 pair-bias tiles of this head and query block, offset by the lane: tile t, piece a at
//                     nbc[(4 t + a) * 64]; nullptr without a pair bias
//   ODD             : the last tile is the one of zeros behind an odd number of them, and left out.  Not with 128 channels, where the
//                     branch costs nine registers more than there are (352 residues 104.6 us with it and without)
//   MFMA_SUMS       : the row sums on the matrix pipe (one 16x16x32 MFMA per 16 keys and row) instead of four dot products
//                     on the vector ALU; costs ten more registers, which the 256-channel kernel (two waves per SIMD) has
template <bool HAS_NB, bool WITH_MASK, bool MFMA_SUMS, bool ODD = false>
__device__ __forceinline__ void attend_pair_l2(const uint4 *lds_kA, const uint4 *lds_vA, const uint4 *lds_kB, const uint4 *lds_vB,
                                               const uint32_t *mwA, const uint32_t *mwB, const f32x4 *nbc, bf16x8 qA0, bf16x8 qA1,
                                               bf16x8 qB0, bf16x8 qB1, int NB, int lane, f32x16 &oA_out,
                                               float &lA_out, f32x16 &oB_out, float &lB_out, int turn)
{
    const int npairs = NB >> 1;
    // The mask of a row as a rank-one MFMA: A holds (hi, lo) of the key of accumulator row i in k-slots 0 and 1, B holds
    // ones there, everything else is zero -- in the lanes of the upper half (k-slots 8..15) both operands are all zero,
    // so that an infinite mask value never meets a zero.
    const uint32_t lower = lane < 32 ? 0xffffffffu : 0u;
    uint4 ones4 = {0x3f803f80u & lower, 0u, 0u, 0u};
    const bf16x8 onesf = as_bf16x8(ones4);
    auto mask_fragment = [&](const uint32_t *mw, int t) {
        uint4 u = {0u, 0u, 0u, 0u};
        if constexpr (WITH_MASK) {
            u.x = mw[32 * t] & lower;
        }
        return as_bf16x8(u);
    };
    const uint4 *kA = lds_kA + lane, *vA = lds_vA + lane, *kB = lds_kB + lane, *vB = lds_vB + lane;
    auto clampt = [&](int t) { return t < NB ? t : NB - 1; };
    auto loadC = [&](int t) {
        f32x16 c;
        if constexpr (HAS_NB) {
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const f32x4 v = nbc[(t * 4 + a) * 64];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    c[4 * a + e] = v[e];
                }
            }
        } else {
            c = zero16();
        }
        return c;
    };
    f32x16 C0 = loadC(0), C1 = loadC(1);
    uint4 k0 = kA[0], k1 = kA[64], v0, v1;
    f32x16 xa, xb;
    xa = mfma(as_bf16x8(k0), qA0, C0);
    xa = mfma(as_bf16x8(k1), qA1, xa);
    if constexpr (WITH_MASK) {
        xa = mfma(mask_fragment(mwA, 0), onesf, xa);
    }
    k0 = kB[0], k1 = kB[64];
    v0 = vA[0], v1 = vA[64];
    f32x16 oA = zero16(), oB = zero16();
    float lsumA = 0.f, lsumB = 0.f; // this lane's share of the row sums; the two halves of the wave are added at the end
    // MFMA_SUMS: as in attend_block_l2 -- rowsum_selector's A operand sums the keys of each query in a 16x16x32 product
    // fed with the probability fragment; the sums of queries n and n + 16 end up in lane n, registers 0 and 1
    f32x4 sumsA = {0.f, 0.f, 0.f, 0.f}, sumsB = {0.f, 0.f, 0.f, 0.f};
    const bf16x8 ones_rows = rowsum_selector(lane);
    bf16x2 one2;
    one2[0] = (bf16_t)1.0f, one2[1] = (bf16_t)1.0f;
    // Probabilities -> bf16 by truncation: one byte permute per pair of values where the rounding conversion is a slower
    // instruction.  The row sums are taken over the same truncated values, so the bias (2^-9 on average) cancels in the
    // normalisation and what is left is a rounding error of up to 2^-8 per probability instead of 2^-9.
    auto pack_trunc = [&](const f32x16 &x, int base) {
        uint4 u;
        u.x = __builtin_amdgcn_perm(__float_as_uint(x[base + 1]), __float_as_uint(x[base + 0]), 0x07060302u);
        u.y = __builtin_amdgcn_perm(__float_as_uint(x[base + 3]), __float_as_uint(x[base + 2]), 0x07060302u);
        u.z = __builtin_amdgcn_perm(__float_as_uint(x[base + 5]), __float_as_uint(x[base + 4]), 0x07060302u);
        u.w = __builtin_amdgcn_perm(__float_as_uint(x[base + 7]), __float_as_uint(x[base + 6]), 0x07060302u);
        return as_bf16x8(u);
    };
    // row sums on the vector ALU, two probabilities per dot2: with two rows in flight the row-sum MFMAs of
    // attend_block_l2 (a selector fragment and an accumulator per row) cost more registers than the loop has
    auto rowsum = [&](float &lsum, f32x4 &sums, bf16x8 pv) {
        if constexpr (MFMA_SUMS) {
            sums = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones_rows, pv, sums, 0, 0, 0);
            return;
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            bf16x2 a;
            a[0] = pv[2 * v], a[1] = pv[2 * v + 1];
            lsum = __builtin_amdgcn_fdot2_f32_bf16(a, one2, lsum, false);
        }
    };
    auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
    auto exp4 = [&](f32x16 &x, int base) {
#pragma unroll
        for (int v = base; v < base + 4; ++v) {
            x[v] = __builtin_amdgcn_exp2f(x[v]);
        }
    };
    // softmax and P.V of the finished tile xc (into o, lacc); logits of the next tile into xn from seed C with query
    // fragments q0, q1; then k0, k1 <- knext[0], knext[64].  No scheduling fences inside: with two independent rows in
    // flight the compiler's own interleaving measured faster than a fixed one.  The empty asm keeps C live past the MFMA
    // that reads it: the compiler then writes xn to registers of its own (D != C) instead of computing it in place in
    // C's registers, which rotated the roles of the register blocks from one iteration to the next and cost 40 copies
    // per iteration, behind a wait for every load in flight.
    auto half_step = [&](f32x16 &xc, f32x16 &xn, const f32x16 &C, bf16x8 q0, bf16x8 q1, f32x16 &o, float &lsum, f32x4 &sums,
                         const uint4 *knext, const uint32_t *mw_next, int t_next) {
        bf16x8 p0, p1;
        const bf16x8 mnext = mask_fragment(mw_next, t_next); // requested first, used by the last MFMA of the step
        exp4(xc, 0);
        exp4(xc, 4);
        p0 = pack_trunc(xc, 0);
        xn = mfma(as_bf16x8(k0), q0, C);
        asm volatile("" ::"v"(C));
        o = mfma(as_bf16x8(v0), p0, o);
        exp4(xc, 8);
        xn = mfma(as_bf16x8(k1), q1, xn);
        if constexpr (WITH_MASK) {
            xn = mfma(mnext, onesf, xn);
        }
        rowsum(lsum, sums, p0);
        k0 = knext[0], k1 = knext[64];
        exp4(xc, 12);
        p1 = pack_trunc(xc, 8);
        o = mfma(as_bf16x8(v1), p1, o);
        rowsum(lsum, sums, p1);
    };
    for (int pair = 0; pair < npairs; ++pair) {
        if (turn >= 0) {
            timeslice_priority((uint32_t)turn, FAIR_SLICE_SHIFT);
        }
        const int t0 = 2 * pair, t1 = t0 + 1;
        const int tn = pair + 1 < npairs ? t0 + 2 : t0; // next pair's first tile, clamped
        // (A, t0) finished; logits of (B, t0) from C0
        half_step(xa, xb, C0, qB0, qB1, oA, lsumA, sumsA, kA + t1 * 128, mwB, t0);
        v0 = vB[t0 * 128], v1 = vB[t0 * 128 + 64];
        fence(); // the loads stay behind the last reader of the registers they fill
        C0 = loadC(clampt(t0 + 2));
        fence();
        // (B, t0) finished; logits of (A, t1) from C1
        half_step(xb, xa, C1, qA0, qA1, oB, lsumB, sumsB, kB + t1 * 128, mwA, t1);
        v0 = vA[t1 * 128], v1 = vA[t1 * 128 + 64];
        if (ODD && pair == npairs - 1) {
            break;
        }
        // (A, t1) finished; logits of (B, t1) from C1
        half_step(xa, xb, C1, qB0, qB1, oA, lsumA, sumsA, kA + tn * 128, mwB, t1);
        v0 = vB[t1 * 128], v1 = vB[t1 * 128 + 64];
        fence();
        C1 = loadC(clampt(t1 + 2));
        fence();
        // (B, t1) finished; logits of (A, tn) from C0
        half_step(xb, xa, C0, qA0, qA1, oB, lsumB, sumsB, kB + tn * 128, mwA, tn);
        v0 = vA[tn * 128], v1 = vA[tn * 128 + 64];
    }
    __builtin_amdgcn_s_setprio(0);
    oA_out = oA, oB_out = oB;
    if constexpr (MFMA_SUMS) {
        lA_out = rowsum_fetch(sumsA, lane), lB_out = rowsum_fetch(sumsB, lane);
    } else {
        lA_out = half_swap_sum(lsumA), lB_out = half_swap_sum(lsumB);
    }
}

// The repeat of one row's block after an overflow or underflow of the unshifted exponentials, with the pair bias as fp32
// tiles: a first pass over the key tiles for the true row maxima, a second one with them subtracted, or (shift != 0) that one alone with the
// row's one mask subtracted (triangle attention of 384 residues, 4 % of them padding, whole block 117 -> 112 us, 199 54.2 -> 50.4).  Not a hot path: one
// row, nothing prefetched, few registers.
template <bool HAS_NB>
__device__ __forceinline__ void attend_row_shifted(const uint4 *lds_k, const uint4 *lds_v, const uint32_t *words, const f32x4 *nbc, bf16x8 q0,
                                                bf16x8 q1, int NB, int lane, float shift, f32x16 &o_out, float &l_out)
{
    // words: the row's mask words (stage_mask_words), offset by 16 (lane >> 5): register 4 a + c stands for key 4 a + c of them
    auto logits = [&](int t) {
        f32x16 x;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const uint4 w4 = *reinterpret_cast<const uint4 *>(words + 32 * t + 4 * a);
            f32x4 mv = {mask_word_value(w4.x), mask_word_value(w4.y), mask_word_value(w4.z), mask_word_value(w4.w)};
            if constexpr (HAS_NB) {
                const f32x4 cv = nbc[(t * 4 + a) * 64];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    mv[c] += cv[c];
                }
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                x[4 * a + c] = mv[c];
            }
        }
        x = mfma(as_bf16x8(lds_k[(t * 2 + 0) * 64 + lane]), q0, x);
        return mfma(as_bf16x8(lds_k[(t * 2 + 1) * 64 + lane]), q1, x);
    };
    float mx = shift;
    if (shift == 0.f) {
        mx = -INFINITY;
        for (int t = 0; t < NB; ++t) {
            const f32x16 x = logits(t);
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                mx = fmaxf(mx, x[v]);
            }
        }
        mx = half_swap_max(mx); // finite: a fully masked row has -1e9*log2(e) everywhere
    }
    f32x16 o = zero16();
    float lsum = 0.f;
    bf16x2 one2;
    one2[0] = (bf16_t)1.0f, one2[1] = (bf16_t)1.0f;
    for (int t = 0; t < NB; ++t) {
        f32x16 x = logits(t);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            x[v] = __builtin_amdgcn_exp2f(x[v] - mx);
        }
        const bf16x8 p0 = pack8(x, 0), p1 = pack8(x, 8);
        o = mfma(as_bf16x8(lds_v[(t * 2 + 0) * 64 + lane]), p0, o);
        o = mfma(as_bf16x8(lds_v[(t * 2 + 1) * 64 + lane]), p1, o);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            bf16x2 a, c;
            a[0] = p0[2 * v], a[1] = p0[2 * v + 1];
            c[0] = p1[2 * v], c[1] = p1[2 * v + 1];
            lsum = __builtin_amdgcn_fdot2_f32_bf16(a, one2, lsum, false);
            lsum = __builtin_amdgcn_fdot2_f32_bf16(c, one2, lsum, false);
        }
    }
    o_out = o;
    l_out = half_swap_sum(lsum);
}

template <int C, bool HAS_NB>
__global__ __launch_bounds__(64 * max_waves(C, 1)) void persistent_pair_kernel(FusedParams p)
{
    constexpr int CK = C / 16;
    // the row sums on the matrix pipe where the registers are there: with 256 channels (two waves per SIMD) always, with
    // 128 (three) in the loop without mask products only -- the masked loop spills with them
    constexpr bool PAIR_MFMA_SUMS = C == 256;
    extern __shared__ uint4 lds[];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int S = p.S, NB = p.NB, NT = p.NT;
    const int nthreads = NB * 64;

    // workgroup -> (XCD, head, batch-row group) as in persistent_head_kernel
    const int w = blockIdx.x;
    const int xcd = w & 7;
    const int slot = w >> 3;
    const int h = slot % p.H;
    const int grp = slot / p.H;
    const int b0 = xcd + 8 * grp;
    const int bstep = 8 * p.ngrp;
    const int nrows = b0 < p.B ? (p.B - b0 + bstep - 1) / bstep : 0;

    uint4 *lds_w = lds;
    uint4 *lds_k = lds_w + 4 * CK * 64;     // [row of the pair][NT][2][64]
    uint4 *lds_v = lds_k + 2 * NT * 2 * 64; // likewise
    uint4 *panel = lds_v + 2 * NT * 2 * 64 + wave * 128;
    uint32_t *mask_base = reinterpret_cast<uint32_t *>(lds_v + 2 * NT * 2 * 64 + NB * 128); // [pair parity][row of the pair][NT*32] mask words
    uint32_t *flag_words = mask_base + 4 * NT * 32;                                         // [pair parity][row of the pair]

    stage_weight_fragments<C>(lds_w, panel, p, h, wave, nthreads >> 6, lane);
    if (tid < 4) {
        flag_words[tid] = 0;
    }
    if (NT > NB) { // phantom key tile of both rows: zero K and V fragments, never written again
        const uint4 z4 = {0u, 0u, 0u, 0u};
        for (int idx = tid; idx < 256; idx += nthreads) {
            const int row = idx >> 7, i = idx & 127;
            lds_k[(row * NT + NB) * 128 + i] = z4;
            lds_v[(row * NT + NB) * 128 + i] = z4;
        }
    }
    __syncthreads();

    const int j = wave; // this wave's sequence block
    const int fair_turn = C == 128 ? wave >> 2 : -1; // time-sliced priorities pay with three waves per SIMD only
    const float qmul = p.qscale * LOG2E;
    const uint32_t x_pitch = (uint32_t)p.x_ld; // the host sends only near-addressable rows here
    for (int n = 0; n < nrows; n += 2) {
        const int par = (n >> 1) & 1;
        const bool have_b = n + 1 < nrows; // an odd row count: the last pair attends its one row twice and stores it once
        const int bA = b0 + n * bstep, bB = have_b ? bA + bstep : bA;
        uint32_t *flag_word = flag_words + 2 * par;
        uint32_t *mask = mask_base + par * 2 * NT * 32;
        // opaque lane index: addresses derived from it are formed anew per pair instead of living across the attention loop
        int lane_x = lane;
        asm volatile("" : "+v"(lane_x));
        stage_mask_words<true>(p.bias + (int64_t)bA * p.bias_sb, mask, flag_word, S, NT, HAS_NB ? S : NT * 32, wave, lane_x, LOG2E, p.bias_sk,
                               p.bias_is_mask != 0);
        stage_mask_words<true>(p.bias + (int64_t)bB * p.bias_sb, mask + NT * 32, flag_word + 1, S, NT, HAS_NB ? S : NT * 32, wave, lane_x, LOG2E, p.bias_sk,
                               p.bias_is_mask != 0);

        // ---- input rows of the block, both batch rows -> fragments, 32 channels per staging panel ----
        const int prow_x = pi_row(lane_x & 31), g_x = lane_x >> 5;
        const bf16_t *xA = p.x + (int64_t)bA * p.x_sb, *xB = p.x + (int64_t)bB * p.x_sb;
        bf16x8 xfA[CK], xfB[CK];
#pragma unroll
        for (int q = 0; q < C / 128; ++q) { // 128 channels of both rows at a time
            Panel32Regs ta[4], tb[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                ta[c] = panel32_load_near(xA, x_pitch, j * 32, S - 1, 128 * q + 32 * c, lane_x);
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                tb[c] = panel32_load_near(xB, x_pitch, j * 32, S - 1, 128 * q + 32 * c, lane_x);
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                panel32_store(panel, lane_x, ta[c]);
                xfA[8 * q + 2 * c] = as_bf16x8(panel[panel32_slot(prow_x, g_x)]);
                xfA[8 * q + 2 * c + 1] = as_bf16x8(panel[panel32_slot(prow_x, 2 + g_x)]);
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                panel32_store(panel, lane_x, tb[c]);
                xfB[8 * q + 2 * c] = as_bf16x8(panel[panel32_slot(prow_x, g_x)]);
                xfB[8 * q + 2 * c + 1] = as_bf16x8(panel[panel32_slot(prow_x, 2 + g_x)]);
            }
        }
        // ---- four projections of the block, both rows per weight fragment ----
        // Gate first, then Q, K, V, each packed to bf16 as soon as it is complete;
        // the scheduling barriers keep the compiler from running the four loops into one another, which needs four
        // pairs of accumulators at once and spilled the input fragments.
        bf16x8 qA0, qA1, qB0, qB1;
        bf16x8 gateB0, gateB1;                                  // sigmoid(gate) of the second row, until the epilogue
        bf16x8 kfA0, kfA1, vfA0, vfA1, kfB0, kfB1, vfB0, vfB1; // parked until the LDS arrays are free
        {
            const uint4 *wsrc = lds_w + lane_x;
            auto project = [&](int proj, f32x16 &accA, f32x16 &accB, bool weights_left) {
#pragma unroll
                for (int ks = 0; ks < CK; ++ks) {
                    const bf16x8 wf = as_bf16x8(wsrc[(proj * CK + ks) * 64]);
                    if (weights_left) {
                        accA = mfma(wf, xfA[ks], accA);
                        accB = mfma(wf, xfB[ks], accB);
                    } else {
                        accA = mfma(xfA[ks], wf, accA);
                        accB = mfma(xfB[ks], wf, accB);
                    }
                }
            };
            __builtin_amdgcn_sched_barrier(0);
            {
                // the gate's accumulator starts at its bias (register v of a lane holds feature 8 (v / 4) + 4 g + v % 4)
                f32x16 accA, accB;
                const float *bgp = p.bg + h * HEAD + 4 * g_x;
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    const f32x4 bv = *reinterpret_cast<const f32x4 *>(bgp + 8 * a);
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        accA[4 * a + c] = bv[c], accB[4 * a + c] = bv[c];
                    }
                }
                project(PROJ_G, accA, accB, true);
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    accA[v] = sigmoid_fast(accA[v]), accB[v] = sigmoid_fast(accB[v]);
                }
                // the first row's into the wave's panel (its input rows are all staged), the second row's stay in registers
                panel[lane_x] = as_uint4(pack8(accA, 0));
                panel[64 + lane_x] = as_uint4(pack8(accA, 8));
                gateB0 = pack8(accB, 0), gateB1 = pack8(accB, 8);
                asm volatile("" : "+v"(gateB0), "+v"(gateB1));
            }
            __builtin_amdgcn_sched_barrier(0);
            {
                f32x16 accA = zero16(), accB = zero16();
                project(PROJ_Q, accA, accB, true);
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    accA[v] *= qmul, accB[v] *= qmul;
                }
                qA0 = pack8(accA, 0), qA1 = pack8(accA, 8);
                qB0 = pack8(accB, 0), qB1 = pack8(accB, 8);
                asm volatile("" : "+v"(qA0), "+v"(qA1), "+v"(qB0), "+v"(qB1)); // packed here, not after the barrier
            }
            __builtin_amdgcn_sched_barrier(0);
            {
                f32x16 accA = zero16(), accB = zero16();
                project(PROJ_K, accA, accB, true);
                kfA0 = pack8(accA, 0), kfA1 = pack8(accA, 8);
                kfB0 = pack8(accB, 0), kfB1 = pack8(accB, 8);
                asm volatile("" : "+v"(kfA0), "+v"(kfA1), "+v"(kfB0), "+v"(kfB1));
            }
            __builtin_amdgcn_sched_barrier(0);
            {
                f32x16 accA = zero16(), accB = zero16();
                project(PROJ_V, accA, accB, false);
                vfA0 = pack8(accA, 0), vfA1 = pack8(accA, 8);
                vfB0 = pack8(accB, 0), vfB1 = pack8(accB, 8);
                asm volatile("" : "+v"(vfA0), "+v"(vfA1), "+v"(vfB0), "+v"(vfB1));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads(); // every wave is done with the previous pair's attention: the K and V arrays are free
        {
            uint4 *ka = lds_k + (j * 2) * 64 + lane, *va = lds_v + (j * 2) * 64 + lane;
            ka[0] = as_uint4(kfA0), ka[64] = as_uint4(kfA1), va[0] = as_uint4(vfA0), va[64] = as_uint4(vfA1);
            ka[NT * 128] = as_uint4(kfB0), ka[NT * 128 + 64] = as_uint4(kfB1);
            va[NT * 128] = as_uint4(vfB0), va[NT * 128 + 64] = as_uint4(vfB1);
        }
        if (tid < 2) {
            flag_words[2 * (par ^ 1) + tid] = 0; // its readers (previous pair) are done, its writers (next pair) start after the next barrier
        }
        __syncthreads(); // K, V and the masks of this pair are complete

        // opaque once more: the loops' LDS and pair-bias addresses are formed here, per pair,
        // rather than hoisted out of the pair loop and spilled
        int lane_a = lane;
        asm volatile("" : "+v"(lane_a));
        const int g = lane_a >> 5;
        const uint32_t *mwA = mask + pi_row(lane_a & 31), *mwB = mwA + NT * 32; // accumulator row i of a tile is its key pi(i)
        const uint32_t flagsA = flag_word[0], flagsB = flag_word[1];
        const f32x4 *nbc = HAS_NB ? reinterpret_cast<const f32x4 *>(p.nbf) + ((int64_t)(h * NB + j) * NT * 4) * 64 + lane_a : nullptr;
        const uint4 *kA = lds_k, *vA = lds_v, *kB = lds_k + NT * 128, *vB = lds_v + NT * 128;
        f32x16 oA, oB;
        float lA, lB;
        if (C == 256 && HAS_NB && (flagsA | flagsB) == 0u && NB < NT) {
            attend_pair_l2<HAS_NB, false, true, C == 256>(kA, vA, kB, vB, mwA, mwB, nbc, qA0, qA1, qB0, qB1, NT, lane_a, oA, lA, oB, lB, fair_turn);
        } else if ((flagsA | flagsB) == 0u) {
            attend_pair_l2<HAS_NB, false, true>(kA, vA, kB, vB, mwA, mwB, nbc, qA0, qA1, qB0, qB1, NT, lane_a, oA, lA, oB, lB, fair_turn);
        } else if (C == 256 && NB < NT) {
            attend_pair_l2<HAS_NB, true, PAIR_MFMA_SUMS, C == 256>(kA, vA, kB, vB, mwA, mwB, nbc, qA0, qA1, qB0, qB1, NT, lane_a, oA, lA, oB, lB, fair_turn);
        } else {
            attend_pair_l2<HAS_NB, true, PAIR_MFMA_SUMS>(kA, vA, kB, vB, mwA, mwB, nbc, qA0, qA1, qB0, qB1, NT, lane_a, oA, lA, oB, lB, fair_turn);
        }
        // some probability overflowed or a whole row underflowed: repeat that row, shifted by its one mask if it has one (a padded residue's row), or
        // by its true row maxima
        auto repeat = [&](const uint4 *k, const uint4 *v, const uint32_t *words, bf16x8 q0, bf16x8 q1, f32x16 &o, float &l) __attribute__((always_inline)) {
            bool differ = false;
            for (int key = lane_a; key < S; key += 64) {
                differ |= words[key] != words[0];
            }
            float shift = __any(differ) ? 0.f : mask_word_value(words[0]);
            bool again = true;
            while (again) {
                const bool maxima = shift == 0.f;
                attend_row_shifted<HAS_NB>(k, v, words + 16 * g, nbc, q0, q1, NT, lane_a, shift, o, l);
                again = !maxima && __any(!(l > 1e-30f && l < 1e30f));
                shift = 0.f;
            }
        };
        if (__any(!(lA > 1e-30f && lA < 1e30f))) {
            repeat(kA, vA, mask, qA0, qA1, oA, lA);
        }
        if (__any(!(lB > 1e-30f && lB < 1e30f))) {
            repeat(kB, vB, mask + NT * 32, qB0, qB1, oB, lB);
        }
        int lane_o = lane; // as above: the addresses of the epilogue are not worth a register during the attention loop
        asm volatile("" : "+v"(lane_o));
        const int qpos = j * 32 + pi_row(lane_o & 31);
        if (qpos < S) {
            const int64_t off = (int64_t)qpos * p.avg_ss + (int64_t)h * p.avg_sh + 4 * (lane_o >> 5);
            const bf16x8 gateA0 = as_bf16x8(panel[lane_o]), gateA1 = as_bf16x8(panel[64 + lane_o]);
            f32x16 gv;
#pragma unroll
            for (int v = 0; v < 8; ++v) {
                gv[v] = to_f32(gateA0[v]), gv[8 + v] = to_f32(gateA1[v]);
            }
            store_gated(p.avg + (int64_t)bA * p.avg_sb + off, oA, __builtin_amdgcn_rcpf(lA), gv);
            if (have_b) {
#pragma unroll
                for (int v = 0; v < 8; ++v) {
                    gv[v] = to_f32(gateB0[v]), gv[8 + v] = to_f32(gateB1[v]);
                }
                store_gated(p.avg + (int64_t)bB * p.avg_sb + off, oB, __builtin_amdgcn_rcpf(lB), gv);
            }
        }
    }
}

// out[t][o] = sum_c avg[t][c] * Wo[o][c] + bo[o]  (reference src/attention/gating_attention.cpp:152-157).
// HBM-bound: each row of avg is read once and each row of out written once, both as whole cache
// lines through the wave-private staging panel.  A workgroup stages the fragments of a 128-feature
// slab of Wo once and its four waves walk 32-row tiles.  The product is formed transposed
// (rows = output features, columns = tokens), which leaves every lane with 4 consecutive features
// of its own token per accumulator group -- an 8-byte panel write.
// EPILOGUE 1 (gated residual): the rounded result is not stored but folded into `out`, out += result * sigmoid(gate),
// with gate and out read in the order they are written, 16 bytes per lane -- the last two steps of the triangle
// multiplication (reference src/attention/triangle_multiplication.cpp:129-150) and the residual update fused into
// its output projection.  EPILOGUE 2 (residual; output_projection_tile_kernel only): out += result, where row (i, j) of the result goes to
// row (j, i) of `out` when swap_n != 0 (rows are pairs (i, j) of an [M / swap_n, swap_n] grid): the residual update of a
// triangle-attention block, transposed back for the ending node.
constexpr int EPILOGUE_STORE = 0, EPILOGUE_GATED_RESIDUAL = 1, EPILOGUE_RESIDUAL = 2;

// With 256 input features a workgroup has eight waves and keeps two 128-feature slabs of Wo (128 KB, the whole matrix of
// the attention's output projection), so a row is read once for all 256 output features; with 128 it has four waves,
// one slab, and two workgroups share a CU.
template <int C, int EPILOGUE>
__global__ __launch_bounds__(C == 128 ? 256 : 512, C == 128 ? 2 : 1) void output_projection_kernel(
    const bf16_t *__restrict__ avg, int64_t avg_ld, const bf16_t *__restrict__ wo, const float *__restrict__ bo,
    bf16_t *__restrict__ out, int64_t out_ld, int64_t M, int N, int rows_per_wave, const bf16_t *__restrict__ gate,
    int64_t gate_ld)
{
    constexpr int CK = C / 16;
    constexpr int NP = CK / 4;
    constexpr int SLABS = C / 128, WAVES = 4 * SLABS, THREADS = 64 * WAVES;
    extern __shared__ uint4 lds[]; // W slabs [SLABS][4 feature blocks][CK][64 lanes], then one panel of 256 per wave
    constexpr bool NEAR = C == 128; // 32-bit row offsets from a wave-uniform base; measured slower with 256 features
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = NEAR ? __builtin_amdgcn_readfirstlane(tid >> 6) : tid >> 6;
    const int r = lane & 31, g = lane >> 5;
    const int nbase = blockIdx.y * (128 * SLABS);               // first output feature of this workgroup
    // slabs it has: with two per workgroup the last workgroup of a row of them may have one
    const int nslab = (SLABS == 1 || N - nbase >= 128 * SLABS) ? SLABS : (N - nbase) / 128;
    uint4 *panel = lds + SLABS * 4 * CK * 64 + wave * 256;
    // Every wave owns a contiguous range of rows_per_wave rows (a multiple of 8), walked 32 rows at a
    // time; the last step of a range may be partial.  Equal ranges rather than whole 32-row tiles dealt
    // round robin: the kernel is short, and a wave with one tile more than its neighbours would set its
    // duration.  The first two panels of a step are fetched while the previous step is multiplied and
    // stored; those of the first step while the weight slab is staged.
    const int64_t start = ((int64_t)blockIdx.x * WAVES + wave) * rows_per_wave;
    const int64_t stop = start + rows_per_wave < M ? start + rows_per_wave : M;
    // With 128 features rows are addressed relative to the wave's first one: 32-bit byte offsets from a wave-uniform
    // base (the host keeps a wave's range below 2^31 bytes), no 64-bit multiply per row.
    const int last_rel = (int)(stop - 1 - start);
    const bf16_t *avg_w = avg + start * avg_ld;
    auto load_panel = [&](int rel_row, int c, int ln) { // 32 rows from rel_row (relative to start), channels 64 c .. 64 c + 63
        if constexpr (NEAR) {
            return panel_load_near(avg_w + c * 64, (uint32_t)avg_ld, rel_row, last_rel, 0, ln);
        } else {
            return panel_load(avg, avg_ld, (int)start + rel_row, (int)(stop - 1), c * 64, ln);
        }
    };
    PanelRegs ta, tb;
    if (start < stop) {
        ta = load_panel(0, 0, lane);
        tb = load_panel(0, 1, lane);
    }
    {
        constexpr int PER = SLABS * 4 * CK * 64 / THREADS; // weight fragments per thread, all loads issued before the first store
        uint4 wreg[PER];
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int idx = tid + i * THREADS;
            int nb_ = idx / (CK * 64);
            nb_ = nb_ < 4 * nslab ? nb_ : 0; // a slab this workgroup does not have: any valid rows, never used
            const int ks = (idx >> 6) % CK;
            const int ln = idx & 63;
            wreg[i] = *reinterpret_cast<const uint4 *>(wo + (int64_t)(nbase + nb_ * 32 + (ln & 31)) * C + ks * 16 + (ln >> 5) * 8);
        }
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            lds[tid + i * THREADS] = wreg[i];
        }
    }
    __syncthreads();
    for (int64_t rbase = start; rbase < stop; rbase += 32) {
        const int row0 = (int)rbase, rel0 = (int)(rbase - start);
        // With 256 input features the lane index is opaque to the optimiser, so that addresses and panel offsets are
        // formed per step instead of being kept (and partly spilled) across the loop.  With 128 the kernel fits either
        // way, and the smaller footprint would let a third workgroup onto some CUs of a grid sized for two.
        int lv = lane;
        if constexpr (C > 128) {
            asm volatile("" : "+v"(lv));
        }
        const int rv = lv & 31, gv = lv >> 5;
        bf16x8 af[CK];
        panel_store(panel, lv, ta);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            af[k] = as_bf16x8(panel[panel_slot(rv, 2 * k + gv)]);
        }
        panel_store(panel, lv, tb);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            af[4 + k] = as_bf16x8(panel[panel_slot(rv, 2 * k + gv)]);
        }
#pragma unroll
        for (int c = 2; c < NP; ++c) {
            ta = load_panel(rel0, c, lv);
            panel_store(panel, lv, ta);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                af[4 * c + k] = as_bf16x8(panel[panel_slot(rv, 2 * k + gv)]);
            }
        }
        {
            // clamped to the last step instead of a branch: one harmless re-read at the end
            const int rnext = rbase + 32 < stop ? rel0 + 32 : rel0;
            ta = load_panel(rnext, 0, lv);
            tb = load_panel(rnext, 1, lv);
        }
#pragma unroll 1
        for (int slab = 0; slab < nslab; ++slab) {
        const int n0 = nbase + slab * 128;
        const uint4 *wslab = lds + slab * 4 * CK * 64;
        const float *bias = bo + n0 + 4 * gv; // read per use: 16 cached loads per tile instead of 64 live registers
#pragma unroll
        for (int half = 0; half < 2; ++half) { // 64 output features per panel
            uint4 gq[4], zq[4];
            if constexpr (EPILOGUE == EPILOGUE_GATED_RESIDUAL) { // requested before the MFMAs, used after them
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    int64_t row = (int64_t)row0 + 8 * i + (lv >> 3);
                    row = row < stop ? row : stop - 1;
                    const int64_t col = n0 + half * 64 + (lv & 7) * 8;
                    gq[i] = *reinterpret_cast<const uint4 *>(gate + row * gate_ld + col);
                    zq[i] = *reinterpret_cast<const uint4 *>(out + row * out_ld + col);
                }
            }
            f32x16 acc[2];
            acc[0] = zero16(), acc[1] = zero16();
#pragma unroll
            for (int ks = 0; ks < CK; ++ks) {
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    acc[n] = mfma(as_bf16x8(wslab[((2 * half + n) * CK + ks) * 64 + lv]), af[ks], acc[n]);
                }
            }
            // accumulators -> panel as bf16 [row][64 features], then whole-line stores
#pragma unroll
            for (int n = 0; n < 2; ++n) {
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    const f32x4 bv = *reinterpret_cast<const f32x4 *>(bias + (2 * half + n) * 32 + 8 * a);
                    bf16x4 ov;
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        ov[c] = (bf16_t)(acc[n][4 * a + c] + bv[c]);
                    }
                    bf16x4 *dst = reinterpret_cast<bf16x4 *>(panel + panel_slot(rv, n * 4 + a)) + gv;
                    *dst = ov;
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int prow_ = 8 * i + (lv >> 3);
                uint4 v = panel[panel_slot(prow_, lv & 7)];
                const int64_t row = (int64_t)row0 + prow_;
                if constexpr (EPILOGUE == EPILOGUE_GATED_RESIDUAL) {
                    const bf16x8 o = as_bf16x8(v), gt = as_bf16x8(gq[i]), z = as_bf16x8(zq[i]);
                    bf16x8 res;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        // bf16(out * sigmoid(gate)) as the reference stores it, then the residual sum in fp32
                        const float upd = to_f32((bf16_t)(to_f32(o[e]) * sigmoid_fast(to_f32(gt[e]))));
                        res[e] = (bf16_t)(to_f32(z[e]) + upd);
                    }
                    v = as_uint4(res);
                }
                if (row < stop) {
                    if constexpr (!NEAR) {
                        *reinterpret_cast<uint4 *>(out + row * out_ld + n0 + half * 64 + (lv & 7) * 8) = v;
                    } else {
                        char *out_w = reinterpret_cast<char *>(out + start * out_ld + n0 + half * 64);
                        *reinterpret_cast<uint4 *>(out_w + (__umul24((uint32_t)(rel0 + prow_), 2u * (uint32_t)out_ld) + 16u * (lv & 7))) = v;
                    }
                }
            }
        }
        } // slabs
    }
}

// The same product by tiles of 32 rows x 128 features, a wave 32 of those; same products in the same order: the same bits.  A workgroup asks
// for rows, weights, bias and the rows of `out` at once, where output_projection_kernel waits for its weights, then for the later channels of
// its rows and for `out` in turn, with a few dozen workgroups where rows are few.  With 128 channels it keeps its weights in registers and walks
// the tiles, three workgroups a CU, the next tile's rows and `out` under way: faster than output_projection_kernel at every size.
// With 256 four waves have no registers for that (128 sequences x 128 residues 39.5 -> 42); there eight waves walk for all 256 features, one
// workgroup a CU, where that gives each more than one tile and no half of its features is missing.  Fewer tiles, or an odd number
// of 128 features, have a workgroup of four waves each, which fetches the weights again: no gain is left past some twelve a CU (300000 rows
// to 128 features 43 in either kernel).
// Whole calls, us, output_projection_kernel's -> now: triangle attention of 50, 77, 128 and 200 residues 19.3 -> 15.3, 22.0 -> 18.0,
// 24.7 -> 21.9, 48.4 -> 44.3, of 256, 400, 450 and 691 52 -> 50, 174 -> 166, 218 -> 208, 504 -> 500; attention of 384 x 384, 4 heads
// 98.5 -> 93.2, of 256 x 384, 8 heads 190 -> 179; MSA rows, 64 x 100 38.2 -> 27.0, 128 x 128 48.4 -> 39.5, 150 x 150 63.5 -> 56,
// 200 x 200 89.8 -> 85.5; MSA columns, 600 x 160 222 -> 207.
constexpr int TILE_WORKGROUPS_PER_CU = 12;
template <int C, int EPILOGUE, int F, bool WALK>
__global__ __launch_bounds__(2 * F, WALK && F == 128 ? 3 : 2) void output_projection_tile_kernel(const bf16_t *__restrict__ avg, int64_t avg_ld, const bf16_t *__restrict__ wo,
                                                                     const float *__restrict__ bo, bf16_t *__restrict__ out, int64_t out_ld, int M, int swap_n)
{
    constexpr int CK = C / 16, SLOTS = C / 8, THREADS = 2 * F, LOADS = 32 * SLOTS / THREADS, PIECES = F / 8;
    __shared__ uint4 rows[32 * SLOTS], result[32 * PIECES]; // slots XOR-ed with row % 16
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, g = lane >> 5;
    const int n0 = (int)blockIdx.y * F, f0 = n0 + 32 * wave;
    const int tiles = (M + 31) / 32;
    bf16x8 in[LOADS];
    bf16_t *to[2], *next_to[2]; // the thread's two pieces of 8 features of `out`
    bf16x8 z[2], next_z[2];
    const auto fetch = [&](int tile) {
        const int row0 = tile * 32, last = min(M - 1 - row0, 31); // its last row that is one
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int idx = tid + THREADS * i;
            in[i] = *reinterpret_cast<const bf16x8 *>(avg + (int64_t)(row0 + min(idx / SLOTS, last)) * avg_ld + idx % SLOTS * 8);
        }
    };
    const auto fetch_out = [&](int tile) {
        const int row0 = tile * 32, last = min(M - 1 - row0, 31);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int at = tid / PIECES + 16 * i;
            const int row = row0 + min(at, last);
            const int target = EPILOGUE == EPILOGUE_RESIDUAL && swap_n ? (int)((uint32_t)row % (uint32_t)swap_n) * (M / swap_n) + (int)((uint32_t)row / (uint32_t)swap_n) : row;
            next_to[i] = out + (int64_t)target * out_ld + n0 + tid % PIECES * 8;
            if constexpr (EPILOGUE == EPILOGUE_RESIDUAL) {
                next_z[i] = *reinterpret_cast<const bf16x8 *>(next_to[i]);
            }
        }
    };
    fetch(blockIdx.x);
    bf16x8 w[CK];
    load_half_lines<CK>(w, wo + (int64_t)f0 * C, C, lane);
    fetch_out(blockIdx.x);
    f32x4 bv[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        bv[a] = *reinterpret_cast<const f32x4 *>(bo + f0 + 8 * a + 4 * g);
    }
    half_lines_to_fragments<CK>(w, result + 128 * wave, lane);
    for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int idx = tid + THREADS * i, row = idx / SLOTS;
            rows[row * SLOTS + (idx % SLOTS ^ (row & 15))] = as_uint4(in[i]);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            to[i] = next_to[i];
            z[i] = next_z[i];
        }
        __syncthreads(); // (the previous result has been read, too)
        if (WALK && tile + (int)gridDim.x < tiles) {
            fetch(tile + gridDim.x);
            fetch_out(tile + gridDim.x);
        }
        f32x16 acc = zero16();
#pragma unroll
        for (int ks = 0; ks < CK; ++ks) {
            acc = mfma(w[ks], as_bf16x8(rows[r * SLOTS + ((2 * ks + g) ^ (r & 15))]), acc);
        }
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            bf16x4 ov;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                ov[c] = (bf16_t)(acc[4 * a + c] + bv[a][c]);
            }
            *(reinterpret_cast<bf16x4 *>(result + r * PIECES + ((4 * wave + a) ^ (r & 15))) + g) = ov;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int at = tid / PIECES + 16 * i;
            uint4 v = result[at * PIECES + (tid % PIECES ^ (at & 15))];
            if constexpr (EPILOGUE == EPILOGUE_RESIDUAL) {
                const bf16x8 o = as_bf16x8(v), zz = z[i];
                bf16x8 sum;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    sum[e] = (bf16_t)(to_f32(zz[e]) + to_f32(o[e]));
                }
                v = as_uint4(sum);
            }
            if (tile * 32 + at < M) {
                *reinterpret_cast<uint4 *>(to[i]) = v;
            }
        }
        if (!WALK) {
            return;
        }
    }
}

// Pair bias [H, S, S] -> fragment-major order: for head h, query block j and key tile t the two B
// operands of the selector MFMAs, [h][j][t][2][64 lanes] x 16 bytes, so that a wave of the attention
// kernels fetches the pair bias of a tile with two contiguous 1 KB loads straight into registers.
// Lane (r, g) holds 16 consecutive keys 32t+16g.. of query row 32j+pi(r); queries past S repeat row
// S-1, keys past S and the phantom tile are PAST_THE_END_F16: the loops without a mask know those keys by that alone, so that
// every pass that writes such a copy (here, pair_bias_bf16_kernel; LOWEST_BIAS in tiles) must.  The pair bias is shared by every batch
// row, so this pass moves 2*H*S*S bytes once per call, against B times that in the attention kernel.
__global__ __launch_bounds__(64) void pair_bias_fragments_kernel(const bf16_t *__restrict__ nb, int64_t nb_sh,
                                                                 int64_t nb_sq, int S, int NB, int NT, int vec,
                                                                 uint4 *__restrict__ out)
{
    const int lane = threadIdx.x;
    const int r = lane & 31, g = lane >> 5;
    const int t = blockIdx.x % NT, j = blockIdx.x / NT, h = blockIdx.y;
    int q = 32 * j + pi_row(r);
    q = q < S ? q : S - 1;
    const int key0 = 32 * t + 16 * g;
    const bf16_t *src = nb + (int64_t)h * nb_sh + (int64_t)q * nb_sq + key0;
    uint4 w0, w1;
    if (vec && key0 + 16 <= S) {
        w0 = *reinterpret_cast<const uint4 *>(src);
        w1 = *reinterpret_cast<const uint4 *>(src + 8);
    } else {
        const uint16_t *s16 = reinterpret_cast<const uint16_t *>(src);
        uint32_t wds[8];
#pragma unroll
        for (int v = 0; v < 8; ++v) {
            const uint32_t a0 = key0 + 2 * v < S ? s16[2 * v] : 0u;
            const uint32_t a1 = key0 + 2 * v + 1 < S ? s16[2 * v + 1] : 0u;
            wds[v] = a0 | (a1 << 16);
        }
        w0.x = wds[0], w0.y = wds[1], w0.z = wds[2], w0.w = wds[3];
        w1.x = wds[4], w1.y = wds[5], w1.z = wds[6], w1.w = wds[7];
    }
    // into log2 units (the logits MFMAs of attend_block_l2 accumulate exponents of 2), as fp16: the product of a bf16 value
    // with log2(e) keeps eleven significant bits instead of eight, so the second rounding costs 2^-12 of the bias, not 2^-9
    const bf16x8 s0 = as_bf16x8(w0), s1 = as_bf16x8(w1);
    uint32_t d[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        d[e] = (uint32_t)pair_bias_log2_f16(to_f32(s0[2 * e])) | ((uint32_t)pair_bias_log2_f16(to_f32(s0[2 * e + 1])) << 16);
        d[4 + e] = (uint32_t)pair_bias_log2_f16(to_f32(s1[2 * e])) | ((uint32_t)pair_bias_log2_f16(to_f32(s1[2 * e + 1])) << 16);
    }
    if (key0 + 16 > S) { // keys past the end: 2^-65504 is zero
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t a0 = key0 + 2 * e < S ? d[e] & 0xffffu : PAST_THE_END_F16, a1 = key0 + 2 * e + 1 < S ? d[e] & 0xffff0000u : PAST_THE_END_F16 << 16;
            d[e] = a0 | a1;
        }
    }
    uint4 *dst = out + ((((int64_t)h * NB + j) * NT + t) * 2) * 64 + lane;
    dst[0] = make_uint4(d[0], d[1], d[2], d[3]);
    dst[64] = make_uint4(d[4], d[5], d[6], d[7]);
}

// Tuning hooks (kutacc_hip_set_tuning): a forced plan of the long-sequence kernel, the fragment-major pair bias switched
// off, one line per call on stderr.  Plain atomics: set from a test or an experiment, read on every launch.
std::atomic<int> g_forced_bpw{0}, g_forced_gw{0}, g_no_fragments{0}, g_debug{0};
std::atomic<int> g_pair_mode{0}; // persistent_pair_kernel: 0 = where row_pairs_pay says so, 1 = wherever it can run, 2 = never

bool fragments_disabled() { return g_no_fragments.load(std::memory_order_relaxed) != 0; }

struct Plan {
    bool persistent;
    int NB, NW, BPW, GW;
    size_t lds_bytes;
    bool tiles; // of a call: the pair bias as fp32 tiles instead of fp16 fragments
};

int max_lds_bytes()
{
    static int table[KUTACC_DEVICE_SLOTS] = {};
    return kutacc_device_attribute(hipDeviceAttributeMaxSharedMemoryPerBlock, 64 * 1024, table);
}

// batch-row groups per XCD of the persistent kernels: one workgroup per CU at most; groups of 8*H workgroups share
// batch-row sequences across the XCDs
int persistent_groups(int B, int H)
{
    const int per_ring = 8 * H;
    int ngrp = kutacc_cu_count() / per_ring;
    const int need = (B + 7) / 8;
    ngrp = ngrp < 1 ? 1 : ngrp;
    return ngrp > need ? need : ngrp;
}

size_t head_kernel_lds(int C, int NB, int GW, int NW, int BPW)
{
    const int NT = (NB + 1) & ~1; // key tiles, padded to a pair
    if (C == 256 && BPW == 4) {
        // second layout of fused_head_kernel: K, then V with all four weight matrices lying on it, then a 4 KB input
        // panel per wave (the mask's place later: 128 NT + 64 bytes always fit under 4 NW + 1 >= NT)
        const size_t kv = (size_t)NT * 2 * 64 * 16, wbytes = (size_t)4 * (C / 16) * 64 * 16;
        return kv + (kv > wbytes ? kv : wbytes) + (size_t)NW * 4096;
    }
    // weights (the mask, 4 bytes per key, and 16 flag words take their place later), K and V
    return (size_t)GW * (C / 16) * 64 * 16 + (size_t)NT * 2 * 64 * 16 * 2;
}

size_t persistent_kernel_lds(int C, int NB)
{
    // all four weight matrices of the head, K and V of one batch row, per wave one 4 KB panel and 2 KB of
    // parked gate fragments, two mask buffers, flags
    const int NT = (NB + 1) & ~1; // key tiles, padded to a pair
    return (size_t)4 * (C / 16) * 64 * 16 + (size_t)NT * 2 * 64 * 16 * 2 + (size_t)NB * (4096 + 2048) +
           (size_t)2 * NT * 32 * 4 + 16;
}

size_t pair_kernel_lds(int C, int NB)
{
    // persistent_pair_kernel: the head's four weight matrices, K and V of two batch rows, per wave one 2 KB panel, two
    // pairs' masks of two rows each, flags
    const int NT = (NB + 1) & ~1;
    return (size_t)4 * (C / 16) * 64 * 16 + (size_t)2 * NT * 2 * 64 * 16 * 2 + (size_t)NB * 2048 + (size_t)4 * NT * 32 * 4 + 16;
}

bool make_plan(int64_t S, int C, Plan &pl)
{
    const int64_t NB = (S + 31) / 32;
    if (NB > 32) {
        return false;
    }
    pl.NB = (int)NB;
    pl.persistent = pl.tiles = false;
    const size_t cap = (size_t)max_lds_bytes();
    const int forced_bpw = g_forced_bpw.load(std::memory_order_relaxed), forced_gw = g_forced_gw.load(std::memory_order_relaxed);
    // persistent kernel: one wave per sequence block, everything of one head resident in LDS
    const bool fits_persistent = NB <= max_waves(C, 1) && persistent_kernel_lds(C, (int)NB) <= cap;
    if (fits_persistent && forced_bpw == 0) {
        pl.persistent = true;
        pl.NW = (int)NB, pl.BPW = 1, pl.GW = 4, pl.lds_bytes = persistent_kernel_lds(C, (int)NB);
        return true;
    }
    if (forced_bpw != 0) {
        const int bpw = forced_bpw;
        const int gw = (C == 128 || bpw == 4) ? 4 : forced_gw; // those kernels are compiled for one group of four
        const int nw = (int)((NB + bpw - 1) / bpw);
        if (nw <= max_waves(C, bpw) && head_kernel_lds(C, pl.NB, gw, nw, bpw) <= cap) {
            pl.BPW = bpw, pl.NW = nw, pl.GW = gw, pl.lds_bytes = head_kernel_lds(C, pl.NB, gw, nw, bpw);
            return true;
        }
    }
    // Most waves resident on a CU first -- a second workgroup where registers and LDS allow one, if need be with the weights
    // staged in smaller groups --, then fewest idle block slots, then most matrices per group, then fewest blocks per wave.
    // With the idle slots first, lengths with many divisors of their block count got few waves: 256 channels and 259
    // positions (nine blocks) three a CU, 321 us at 400 rows against 244 with 2 x 3; 128 channels and 470 positions (15
    // blocks) five, 239 us against 192 with eight.
    int best_waves = 0, best_idle = 0, best_gw = 0;
    for (int bpw = 1; bpw <= 4; ++bpw) {
        const int nw = (int)((NB + bpw - 1) / bpw);
        if (nw > max_waves(C, bpw)) {
            continue;
        }
        // The 128-channel kernels and the 256-channel one with four blocks per wave are compiled for one group of four.
        const int gw_min = (C == 128 || bpw == 4) ? 4 : 1;
        for (int gw = 4; gw >= gw_min; gw >>= 1) {
            const size_t need = head_kernel_lds(C, (int)NB, gw, nw, bpw);
            if (need > cap) {
                continue;
            }
            const int by_lds = (int)(cap / need), by_waves = max_waves(C, bpw) / nw;
            const int waves = nw * (by_lds < by_waves ? by_lds : by_waves), idle = nw * bpw - (int)NB;
            if (waves > best_waves || (waves == best_waves && (idle < best_idle || (idle == best_idle && gw > best_gw)))) {
                best_waves = waves, best_idle = idle, best_gw = gw;
                pl.BPW = bpw, pl.NW = nw, pl.GW = gw, pl.lds_bytes = need;
            }
        }
    }
    return best_waves > 0;
}

inline bool aligned(const void *p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }

// Bytes of the fragment-major copy of the pair bias: [nheads][NB query blocks][NB rounded up to even key tiles][2][64] x 16
int64_t fragment_bytes(int64_t nheads, int NB) { return nheads * NB * ((NB + 1) & ~1) * 2048; }

// Where the fast attention loop keeps its fragment-major copy of the pair bias, or nullptr when the call gets none: the
// workspace the options bring, else the caller's q scratch tensor when that is dense, aligned and large enough.
// `scale`: 1 for the fp16 fragments, 2 for the fp32 tiles of persistent_pair_kernel
void *fragment_home(const kutacc_hip_attention_args_t &a, int NB, const kutacc_launch::FusedAttentionOptions &opt, int scale = 1)
{
    if (a.nonbatched_bias == nullptr || fragments_disabled()) {
        return nullptr;
    }
    const int64_t nbf_bytes = fragment_bytes(a.nheads, NB) * scale;
    if (opt.fragment_workspace != nullptr) {
        return (aligned(opt.fragment_workspace, 16) && (uint64_t)nbf_bytes <= opt.fragment_workspace_bytes)
                   ? opt.fragment_workspace
                   : nullptr;
    }
    const int64_t C = a.nheads * a.head_size;
    const bool q_dense = a.q != nullptr && aligned(a.q, 16) && a.q_stride_h == a.head_size && a.q_stride_s == C &&
                         a.q_stride_b == a.seq_len * C;
    return (q_dense && nbf_bytes <= a.batch * a.seq_len * C * 2) ? a.q : nullptr;
}

// Whether the rows of a workgroup are better walked in pairs.  With an odd number the last pair costs as much as a whole
// one, which a pair's gain over two single rows (2 % with 128 channels, 5 to 10 % with 256) makes up for from some number on.
// Operator, us, pairs against single rows on the same fp32 tiles.  128 channels: 187 x 200 (three rows) 38.6 34.4, 187 x 384 59.4
// 54.9, 315 x 290 (five) 75.5 69.0, 443 x 200 (seven) 65.0 63.1, 443 x 384 104.2 105.4, 571 x 200 (nine) 79.5 79.1, 699 x 200
// (eleven) 91.8 92.1, 699 x 384 159 163.  256 channels: 93 x 250 (three) 55.2 50.9, 157 x 250 (five) 70.8 69.3, 221 x 250
// (seven) 88.4 88.5, 285 x 250 (nine) 109.6 112.7, 349 x 128 (eleven) 69.8 70.5.
bool row_pairs_pay(const kutacc_hip_attention_args_t &a)
{
    const int64_t sequences = 8 * (int64_t)persistent_groups((int)a.batch, (int)a.nheads), rows = (a.batch + sequences - 1) / sequences;
    return a.batch >= 2 * sequences && (rows % 2 == 0 || rows >= (a.nheads * a.head_size == 128 ? 11 : 7));
}

// Two batch rows per step (persistent_pair_kernel): 128 or 256 channels, log2 units, a home for the fp32 tiles of the pair bias
// (twice the fragments' bytes), no LayerNorm inside the kernel and no ready-made fp16 fragments; by default only where
// that pays.
bool pair_kernel_applies(const kutacc_hip_attention_args_t &a, const Plan &pl, const kutacc_launch::FusedAttentionOptions &opt)
{
    const int pair_mode = g_pair_mode.load(std::memory_order_relaxed);
    const int64_t C = a.nheads * a.head_size;
    return pl.persistent && (C == 128 || C == 256) && pair_mode != 2 && !fragments_disabled() && opt.ln_gamma == nullptr &&
           !opt.nb_fragments_ready && pair_kernel_lds((int)C, pl.NB) <= (size_t)max_lds_bytes() &&
           (a.nonbatched_bias == nullptr || fragment_home(a, pl.NB, opt, 2) != nullptr) &&
           (pair_mode == 1 || row_pairs_pay(a));
}

// The plan of a call.  Short rows of 128 channels (two to four blocks) give the persistent kernel four waves a CU where a
// workgroup per unit, with a third of the LDS, has twelve.  Staging the weights for every unit costs less than that as soon as
// a workgroup of the persistent kernel would walk a second row.  Operator, us, persistent against one workgroup per unit: 66 x 96
// 18.7 17.0, 96 x 60 17.9 17.2; in pairs, both on fp32 tiles, 128 x 128 17.8 17.2, 190 x 80 24.4 20.0, 256 x 80 25.5 24.7, 500 x
// 128 41.4 39.8; one row a workgroup, 60 x 128: 15.5 15.6; five blocks, 128 x 150: 24.1 26.9.  With 256 channels the weights are four times as many, and it
// pays where some workgroups would walk two rows and none more: 40 x 77 30.3 29.0, 60 x 64 28.5 27.1, 60 x 110 31.4 30.6; two
// two rows each, in pairs, 64 x 128: 29.7 30.0; three, 90 x 80: 35.9 37.5.
//
// The pair bias: from two rows a workgroup on, where the persistent kernel fits, as fp32 tiles wherever those have a home, for pairs
// and for single rows alike (the 11 bits of the fragments were off by 1.1 % in the average at a bias of 50, the tiles by 0.3 %;
// single rows 2 to 4 % slower: 135 x 135 27.8 28.6, 290 x 290 64.2 66.8, 96 x 250 with 256 channels 49.7 51.3).
bool make_call_plan(const kutacc_hip_attention_args_t &a, const kutacc_launch::FusedAttentionOptions &opt, Plan &pl)
{
    const int C = (int)(a.nheads * a.head_size);
    if (!make_plan(a.seq_len, C, pl)) {
        return false;
    }
    const int64_t sequences = 8 * (int64_t)persistent_groups((int)a.batch, (int)a.nheads); // of rows, one per workgroup and head
    pl.tiles = pl.persistent && a.batch >= 2 * sequences && opt.ln_gamma == nullptr && !opt.nb_fragments_ready && fragment_home(a, pl.NB, opt, 2) != nullptr;
    if (pl.persistent && pl.NB >= 2 && pl.NB <= 4 && a.batch > sequences && (C == 128 || a.batch < 2 * sequences) &&
        opt.ln_gamma == nullptr && g_pair_mode.load(std::memory_order_relaxed) != 1 && !fragments_disabled() &&
        (a.nonbatched_bias == nullptr || fragment_home(a, pl.NB, opt) != nullptr)) {
        pl.persistent = false;
        pl.lds_bytes = head_kernel_lds(C, pl.NB, pl.GW, pl.NW, pl.BPW);
    }
    return true;
}

template <typename K>
int opt_in_lds(K kern, size_t bytes, size_t *table)
{
    return (int)kutacc_opt_in_lds(reinterpret_cast<const void *>(kern), bytes, table);
}

template <typename K>
int launch_rows_kernel(K kern, size_t *configured, int64_t workgroups, const FusedParams &p, const Plan &pl, hipStream_t stream)
{
    if (const int rc = opt_in_lds(kern, pl.lds_bytes, configured)) {
        return rc;
    }
    kern<<<dim3((unsigned)workgroups), dim3((unsigned)(pl.NW * 64)), pl.lds_bytes, stream>>>(p);
    return kutacc_hip_status(hipGetLastError());
}

// The kernels of an odd number of key tiles have the loop that leaves out the tile of zeros, and no other without a shift: beside the
// loops of even numbers it spilled registers that each pair of tiles then fetched back (eleven in the persistent kernel of 128 channels with fp32 tiles).
template <int C, int BPW, bool HAS_NB, bool TILES = false>
int launch_head_kernel(const FusedParams &p, const Plan &pl, hipStream_t stream)
{
    static size_t configured[2][KUTACC_DEVICE_SLOTS] = {}; // per instantiation and device: dynamic LDS opted into so far
    const int64_t units = ((int64_t)(p.B + 7) / 8) * 8 * p.H;
    return p.NB < p.NT && (TILES || p.l2mode) ? launch_rows_kernel(fused_head_kernel<C, BPW, HAS_NB, TILES, true>, configured[1], units, p, pl, stream)
                                              : launch_rows_kernel(fused_head_kernel<C, BPW, HAS_NB, TILES, false>, configured[0], units, p, pl, stream);
}

template <int C, bool HAS_NB, bool L2MODE, bool FUSED_LN = false, bool TILES = false>
int launch_persistent_kernel(FusedParams p, const Plan &pl, hipStream_t stream)
{
    static size_t configured[2][KUTACC_DEVICE_SLOTS] = {};
    p.ngrp = persistent_groups(p.B, p.H);
    const int64_t workgroups = 8 * (int64_t)p.H * p.ngrp;
    return p.NB < p.NT && L2MODE ? launch_rows_kernel(persistent_head_kernel<C, HAS_NB, L2MODE, FUSED_LN, TILES, L2MODE>, configured[1], workgroups, p, pl, stream)
                                 : launch_rows_kernel(persistent_head_kernel<C, HAS_NB, L2MODE, FUSED_LN, TILES, false>, configured[0], workgroups, p, pl, stream);
}

template <int C, bool HAS_NB>
int launch_pair_kernel(FusedParams p, const Plan &pl, hipStream_t stream)
{
    auto kern = persistent_pair_kernel<C, HAS_NB>;
    static size_t configured[KUTACC_DEVICE_SLOTS] = {};
    const size_t lds_bytes = pair_kernel_lds(C, pl.NB);
    if (const int rc = opt_in_lds(kern, lds_bytes, configured)) {
        return rc;
    }
    p.ngrp = persistent_groups(p.B, p.H);
    kern<<<dim3((unsigned)(8 * p.H * p.ngrp)), dim3((unsigned)(pl.NW * 64)), lds_bytes, stream>>>(p);
    return kutacc_hip_status(hipGetLastError());
}

template <int C>
int dispatch_head_kernel(const FusedParams &p, const Plan &pl, hipStream_t stream)
{
    const bool nb = p.nb != nullptr;
    if (pl.persistent) {
        if (p.ln_gamma != nullptr) { // only asked for where fused_layernorm_supported says so: log2 units
            return nb ? launch_persistent_kernel<C, true, true, true>(p, pl, stream)
                      : launch_persistent_kernel<C, false, true, true>(p, pl, stream);
        }
        if (pl.tiles) {
            return launch_persistent_kernel<C, true, true, false, true>(p, pl, stream);
        }
        if (p.l2mode) {
            return nb ? launch_persistent_kernel<C, true, true>(p, pl, stream) : launch_persistent_kernel<C, false, true>(p, pl, stream);
        }
        return nb ? launch_persistent_kernel<C, true, false>(p, pl, stream) : launch_persistent_kernel<C, false, false>(p, pl, stream);
    }
    if constexpr (C == 128) {
        if (pl.tiles) { // the short rows that make_call_plan takes from the persistent kernel: one block per wave
            return launch_head_kernel<C, 1, true, true>(p, pl, stream);
        }
    }
    switch (pl.BPW) {
        case 1: return nb ? launch_head_kernel<C, 1, true>(p, pl, stream) : launch_head_kernel<C, 1, false>(p, pl, stream);
        case 2: return nb ? launch_head_kernel<C, 2, true>(p, pl, stream) : launch_head_kernel<C, 2, false>(p, pl, stream);
        case 3: return nb ? launch_head_kernel<C, 3, true>(p, pl, stream) : launch_head_kernel<C, 3, false>(p, pl, stream);
        case 4: return nb ? launch_head_kernel<C, 4, true>(p, pl, stream) : launch_head_kernel<C, 4, false>(p, pl, stream);
        default: return KUTACC_HIP_EUNSUPPORTED;
    }
}

// How output_projection_kernel<C, .> splits M rows: workgroups along the rows and rows per wave (a multiple of 8).  Two
// workgroups of four waves per CU, or one of eight: each wave with an equal share of the rows (a third resident
// workgroup, where the registers allow one, measured slower: the weight slab is staged per workgroup).
inline void output_projection_split(int C, int64_t M, int64_t &gx, int64_t &rpw)
{
    const int waves = 4 * (C / 128);
    const int64_t tiles = (M + 31) / 32;
    gx = (tiles + waves - 1) / waves;
    const int64_t cap = (int64_t)kutacc_cu_count() * (C == 128 ? 2 : 1);
    gx = gx > cap ? cap : gx;
    rpw = ((M + gx * waves - 1) / (gx * waves) + 7) / 8 * 8;
}

// The kernel addresses a wave's rows with 32-bit byte offsets from the wave's first row: true when that range fits for
// these row pitches under the split the launcher will choose.
inline bool output_projection_rows_fit(int C, int64_t M, int64_t a_ld, int64_t out_ld)
{
    if (a_ld <= 0 || out_ld <= 0 || M <= 0) {
        return false;
    }
    int64_t gx, rpw;
    output_projection_split(C, M, gx, rpw);
    const int64_t pitch = a_ld > out_ld ? a_ld : out_ld;
    return pitch < (1 << 23) && (rpw + 32) * pitch * 2 < ((int64_t)1 << 31);
}

// out[M, N] = a[M, K] . w[N, K]^T + bias with K = C and N a multiple of 128 (one grid row per 128-feature slab)
template <int C, int EPILOGUE = EPILOGUE_STORE>
int launch_output_projection(const void *a, int64_t a_ld, const void *w, const float *bias, void *out, int64_t out_ld,
                             int64_t M, int64_t N, hipStream_t stream, const void *gate = nullptr, int64_t gate_ld = 0,
                             int64_t swap_n = 0)
{
    if (!output_projection_rows_fit(C, M, a_ld, out_ld)) {
        return KUTACC_HIP_EUNSUPPORTED; // the callers' support checks ask the same question first
    }
    const double flops = 2.0 * (double)M * (double)N * C;
    if constexpr (EPILOGUE != EPILOGUE_GATED_RESIDUAL) {
        const int64_t tiles = (M + 31) / 32, slabs = N / 128;
        // not where the result lies over the rows: one workgroup's features would be written while another still reads them (a residual is
        // added to an activation, of which the rows are never part)
        const uintptr_t from = reinterpret_cast<uintptr_t>(a), to = reinterpret_cast<uintptr_t>(out);
        const bool apart = EPILOGUE == EPILOGUE_RESIDUAL || from + (uintptr_t)(2 * ((M - 1) * a_ld + C)) <= to || to + (uintptr_t)(2 * ((M - 1) * out_ld + N)) <= from;
        const int64_t cus = kutacc_cu_count();
        const auto launch = [&](auto kern, bool walks, int features, int64_t per_cu) {
            kutacc_prof::KernelTimer t(EPILOGUE == EPILOGUE_RESIDUAL ? (walks ? "output_projection_tile_kernel<residual, walking>" : "output_projection_tile_kernel<residual>")
                                       : walks                       ? "output_projection_tile_kernel<walking>"
                                                                     : "output_projection_tile_kernel",
                                       flops, stream);
            const int64_t gx = std::min(tiles, std::max<int64_t>(per_cu * cus / (N / features), 1));
            kern<<<dim3((unsigned)gx, (unsigned)(N / features)), 2 * features, 0, stream>>>(
                (const bf16_t *)a, a_ld, (const bf16_t *)w, bias, (bf16_t *)out, out_ld, (int)M, (int)swap_n);
            return kutacc_hip_status(hipGetLastError());
        };
        if (apart && M < (1 << 30)) {
            if (C == 128) {
                return launch(output_projection_tile_kernel<C, EPILOGUE, 128, C == 128>, true, 128, 3);
            }
            if (N % 256 == 0 && tiles * (N / 256) > cus) {
                return launch(output_projection_tile_kernel<C, EPILOGUE, C, true>, true, 256, 1);
            }
            if (tiles * slabs <= TILE_WORKGROUPS_PER_CU * cus) {
                return launch(output_projection_tile_kernel<C, EPILOGUE, 128, C == 128>, false, 128, INT_MAX);
            }
        }
    }
    if constexpr (EPILOGUE != EPILOGUE_RESIDUAL) {
        auto kern = output_projection_kernel<C, EPILOGUE>;
        constexpr int SLABS = C / 128, WAVES = 4 * SLABS;
        const size_t lds_bytes = (size_t)SLABS * 4 * (C / 16) * 64 * 16 + WAVES * 4096;
        static size_t configured[KUTACC_DEVICE_SLOTS] = {};
        if (const int rc = opt_in_lds(kern, lds_bytes, configured)) {
            return rc;
        }
        int64_t gx, rpw;
        output_projection_split(C, M, gx, rpw);
        const int64_t gy = (N / 128 + SLABS - 1) / SLABS;
        kutacc_prof::KernelTimer t(EPILOGUE == EPILOGUE_GATED_RESIDUAL ? "output_projection_kernel<gated residual>" : "output_projection_kernel", flops, stream);
        kern<<<dim3((unsigned)gx, (unsigned)gy), 64 * WAVES, lds_bytes, stream>>>(
            (const bf16_t *)a, a_ld, (const bf16_t *)w, bias, (bf16_t *)out, out_ld, M, (int)N, (int)rpw, (const bf16_t *)gate, gate_ld);
        return kutacc_hip_status(hipGetLastError());
    }
    return KUTACC_HIP_EUNSUPPORTED; // (more rows than a device holds)
}

} // namespace

namespace kutacc_launch {

bool fused_attention_fragment_layout(const kutacc_hip_attention_args_t &a, int *nb, int *nt)
{
    Plan pl;
    if (!fused_attention_supports(a) || !make_plan(a.seq_len, (int)(a.nheads * a.head_size), pl) ||
        fragment_home(a, pl.NB, FusedAttentionOptions()) == nullptr) {
        return false;
    }
    *nb = pl.NB, *nt = (pl.NB + 1) & ~1;
    return true;
}

bool fused_attention_tile_layout(const kutacc_hip_attention_args_t &a, const FusedAttentionOptions &opt, int *nb, int *nt)
{
    Plan pl;
    if (a.nonbatched_bias == nullptr || opt.nb_fragments_ready || !fused_attention_supports(a) ||
        !make_call_plan(a, opt, pl) || !(pl.tiles || pair_kernel_applies(a, pl, opt))) {
        return false;
    }
    *nb = pl.NB, *nt = (pl.NB + 1) & ~1;
    return true;
}

bool fused_layernorm_supported(const kutacc_hip_attention_args_t &a, const FusedAttentionOptions &opt)
{
    Plan pl;
    if (!fused_attention_supports(a) || !make_plan(a.seq_len, (int)(a.nheads * a.head_size), pl) || !pl.persistent ||
        fragments_disabled()) {
        return false;
    }
    // log2 units need the fragment-major pair bias (none without a pair bias)
    return a.nonbatched_bias == nullptr || fragment_home(a, pl.NB, opt) != nullptr;
}

bool fused_attention_supports(const kutacc_hip_attention_args_t &a)
{
    if (a.dtype != KUTACC_DTYPE_BF16 || a.head_size != HEAD) {
        return false;
    }
    const int64_t C = a.nheads * a.head_size;
    if (C != 128 && C != 256) {
        return false;
    }
    if (a.batch > (1 << 24) || a.seq_len > 1024) {
        return false;
    }
    // the kernels address the rows of one batch row (the output projection: of a wave's range) with 32-bit byte offsets
    if (a.input_ld <= 0 || a.input_ld > (1 << 19) || a.out_ld <= 0 || a.out_ld > (1 << 19) || a.avg_stride_s <= 0 ||
        a.avg_stride_s > (1 << 19)) {
        return false;
    }
    // 16-byte row loads of input and weights, 8-byte stores of avg/out rows
    if (a.input_ld % 8 != 0 || !aligned(a.input, 16) || !aligned(a.query_w, 16) || !aligned(a.key_w, 16) ||
        !aligned(a.value_w, 16) || !aligned(a.gating_w, 16) || !aligned(a.output_w, 16) || !aligned(a.gating_b, 16) ||
        !aligned(a.output_b, 16)) {
        return false;
    }
    if (a.avg_stride_h != HEAD || a.avg_stride_s % 8 != 0 || a.avg_stride_b != a.seq_len * a.avg_stride_s ||
        !aligned(a.avg, 16) || a.out_ld % 8 != 0 || !aligned(a.out, 16)) {
        return false;
    }
    // ... and the output projection a wave's range of the batch * seq_len rows of avg and out
    if (!output_projection_rows_fit((int)C, a.batch * a.seq_len, a.avg_stride_s, a.out_ld)) {
        return false;
    }
    Plan pl;
    return make_plan(a.seq_len, (int)C, pl);
}

int pair_bias_tiles(const kutacc_hip_attention_args_t &a, void *tiles, hipStream_t stream)
{
    const int NB = (int)((a.seq_len + 31) / 32), NT = (NB + 1) & ~1;
    const int vec = aligned(a.nonbatched_bias, 16) && a.nb_stride_h % 8 == 0 && a.nb_stride_q % 8 == 0;
    kutacc_prof::KernelTimer t("pair_bias_tiles_kernel", 0.0, stream);
    pair_bias_tiles_kernel<<<dim3((unsigned)NB * NT, (unsigned)a.nheads), 64, 0, stream>>>(
        (const bf16_t *)a.nonbatched_bias, a.nb_stride_h, a.nb_stride_q, (int)a.seq_len, NB, NT, vec, (f32x4 *)tiles);
    return kutacc_hip_status(hipGetLastError());
}

int gating_attention_fused(const kutacc_hip_attention_args_t &a, hipStream_t stream, const FusedAttentionOptions &opt)
{
    const int residual = opt.out_mode;
    const int C = (int)(a.nheads * a.head_size);
    Plan pl;
    if (!make_call_plan(a, opt, pl)) {
        return KUTACC_HIP_EUNSUPPORTED;
    }
    if (opt.bias_stride_k < 0 || opt.bias_stride_k > (1 << 20) || a.input_ld <= 0 || a.input_ld > (1 << 19)) {
        return KUTACC_HIP_EUNSUPPORTED; // 32-bit offsets within a batch row (fused_attention_supports checks input_ld too)
    }
    FusedParams p;
    p.x = (const bf16_t *)a.input;
    p.w[PROJ_K] = (const bf16_t *)a.key_w, p.w[PROJ_V] = (const bf16_t *)a.value_w;
    p.w[PROJ_Q] = (const bf16_t *)a.query_w, p.w[PROJ_G] = (const bf16_t *)a.gating_w;
    p.bg = a.gating_b;
    p.bias = (const bf16_t *)a.bias;
    p.nb = (const bf16_t *)a.nonbatched_bias;
    p.avg = (bf16_t *)a.avg;
    p.x_ld = a.input_ld, p.bias_sb = a.bias_stride_b, p.nb_sh = a.nb_stride_h, p.nb_sq = a.nb_stride_q;
    p.x_sb = opt.input_stride_b != 0 ? opt.input_stride_b : a.seq_len * a.input_ld;
    p.ln_gamma = nullptr, p.ln_beta = nullptr, p.ln_eps = 0.f;
    p.bias_sk = opt.bias_stride_k, p.bias_is_mask = opt.bias_is_mask ? 1 : 0;
    p.avg_sb = a.avg_stride_b, p.avg_ss = a.avg_stride_s, p.avg_sh = a.avg_stride_h;
    p.B = (int)a.batch, p.S = (int)a.seq_len, p.H = (int)a.nheads, p.NB = pl.NB, p.NW = pl.NW, p.GW = pl.GW;
    p.NT = (pl.NB + 1) & ~1;
    p.nb_vec = (p.nb != nullptr && aligned(p.nb, 16) && a.nb_stride_h % 8 == 0 && a.nb_stride_q % 8 == 0) ? 1 : 0;
    // (float)(1/sqrt(head_size)) as the reference forms it (gating_attention.cpp:68)
    p.qscale = (float)(1.0 / sqrt((double)a.head_size));
    p.ngrp = 1;
    p.nbf = nullptr;
    p.l2mode = 0;
    // Fragment-major copy of the pair bias for the fast attention loop.  It lives in the workspace the options bring or in
    // the caller's q scratch tensor (which this path does not otherwise use; its contents are unspecified after any
    // call) when that is dense, aligned and large enough; otherwise the kernels read the pair bias in place through the
    // staging panels.
    void *const fragments = fragment_home(a, pl.NB, opt);
    if (opt.fragment_workspace != nullptr && p.nb != nullptr && fragments == nullptr && !fragments_disabled()) {
        return KUTACC_HIP_EINVAL; // the caller's workspace cannot hold the copy
    }
    void *const tiles = fragment_home(a, pl.NB, opt, 2);
    const bool pair_kernel = pair_kernel_applies(a, pl, opt);
    if (opt.nb_tiles_ready && (!(pl.tiles || pair_kernel) || p.nb == nullptr)) {
        return KUTACC_HIP_EINVAL; // the caller asks fused_attention_tile_layout under the same options and tuning first
    }

    const double BS = (double)a.batch * (double)a.seq_len;
    int rc;
    if (pair_kernel || pl.tiles) {
        if (p.nb != nullptr && opt.nb_tiles_ready) {
            p.nbf = (const uint4 *)tiles; // the producer of the pair bias wrote the tiles
        } else if (p.nb != nullptr) {
            rc = kutacc_launch::pair_bias_tiles(a, tiles, stream);
            if (rc != 0) {
                return rc;
            }
            p.nbf = (const uint4 *)tiles;
        }
    } else if (fragments != nullptr && opt.nb_fragments_ready) {
        p.nbf = (const uint4 *)fragments; // the producer of the pair bias wrote the copy
    } else if (fragments != nullptr) {
        kutacc_prof::KernelTimer t("pair_bias_fragments_kernel", 0.0, stream);
        pair_bias_fragments_kernel<<<dim3((unsigned)(pl.NB * p.NT), (unsigned)a.nheads), 64, 0, stream>>>(
            p.nb, p.nb_sh, p.nb_sq, p.S, pl.NB, p.NT, p.nb_vec, (uint4 *)fragments);
        rc = kutacc_hip_status(hipGetLastError());
        if (rc != 0) {
            return rc;
        }
        p.nbf = (const uint4 *)fragments;
    }
    p.l2mode = ((p.nb == nullptr || p.nbf != nullptr) && !fragments_disabled()) ? 1 : 0;
    if (opt.ln_gamma != nullptr) {
        if (!pl.persistent || !p.l2mode || opt.ln_beta == nullptr || !aligned(opt.ln_gamma, 16) || !aligned(opt.ln_beta, 16)) {
            return KUTACC_HIP_EUNSUPPORTED; // the caller asks fused_layernorm_supported first
        }
        p.ln_gamma = opt.ln_gamma, p.ln_beta = opt.ln_beta, p.ln_eps = opt.ln_eps;
    }
    if (g_debug.load(std::memory_order_relaxed)) {
        fprintf(stderr,
                "[kutacc] fused plan: persistent=%d C=%d NB=%d NT=%d NW=%d BPW=%d GW=%d lds=%zu max_lds=%d cus=%d log2_units=%d "
                "fragments=%d row_pairs=%d\n",
                (int)pl.persistent, C, pl.NB, p.NT, pl.NW, pl.BPW, pl.GW, pl.lds_bytes, max_lds_bytes(), kutacc_cu_count(), p.l2mode,
                p.nbf != nullptr ? 1 : 0, (int)pair_kernel);
    }
    {
        kutacc_prof::KernelTimer t(pair_kernel ? "persistent_pair_kernel" : pl.persistent ? "persistent_head_kernel" : "fused_head_kernel",
                                   8.0 * BS * C * C + 4.0 * BS * (double)a.seq_len * C, stream);
        rc = pair_kernel ? (C == 128 ? (p.nb != nullptr ? launch_pair_kernel<128, true>(p, pl, stream) : launch_pair_kernel<128, false>(p, pl, stream))
                                     : (p.nb != nullptr ? launch_pair_kernel<256, true>(p, pl, stream) : launch_pair_kernel<256, false>(p, pl, stream)))
             : (C == 128) ? dispatch_head_kernel<128>(p, pl, stream)
                          : dispatch_head_kernel<256>(p, pl, stream);
        if (rc != 0) {
            return rc;
        }
    }
    const int64_t M = a.batch * a.seq_len;
    if (residual != FUSED_OUT_STORE) {
        // out += result, row (b, s) of the result going to row (s, b) of out ([seq_len, batch, C]) in the transposed form
        const int64_t swap_n = residual == FUSED_OUT_ADD_TRANSPOSED ? a.seq_len : 0;
        return (C == 128) ? launch_output_projection<128, EPILOGUE_RESIDUAL>(a.avg, a.avg_stride_s, a.output_w, a.output_b, a.out,
                                                                             a.out_ld, M, C, stream, nullptr, 0, swap_n)
                          : launch_output_projection<256, EPILOGUE_RESIDUAL>(a.avg, a.avg_stride_s, a.output_w, a.output_b, a.out,
                                                                             a.out_ld, M, C, stream, nullptr, 0, swap_n);
    }
    return (C == 128) ? launch_output_projection<128>(a.avg, a.avg_stride_s, a.output_w, a.output_b, a.out, a.out_ld, M, C, stream)
                      : launch_output_projection<256>(a.avg, a.avg_stride_s, a.output_w, a.output_b, a.out, a.out_ld, M, C, stream);
}

// The attention's output-projection kernel on its own: out[m, n] = sum_k a[m, k] * w[n, k] + bias[n] for rows of
// 128 or 256 input features (w dense [n, k]) and n a multiple of 128.  HBM-bound; every row is read and written
// once per 128-feature slab of the output.
bool row_projection_supports(const void *a, int64_t a_ld, const void *w, const float *bias, const void *out, int64_t out_ld,
                             int64_t m, int64_t n, int64_t k)
{
    // row pitches the kernel's 32-bit offsets within a wave's range of rows can take under the launcher's split of m rows
    if (k != 128 && k != 256) {
        return false;
    }
    const bool pitches = a_ld > 0 && out_ld > 0 && a_ld <= (1 << 19) && out_ld <= (1 << 19) && m > 0 &&
                         output_projection_rows_fit((int)k, m, a_ld, out_ld);
    return n > 0 && n % 128 == 0 && n / 128 <= 65535 && m > 0 && m <= INT32_MAX - 64 && bias && pitches &&
           a_ld % 8 == 0 && out_ld % 8 == 0 && aligned(a, 16) && aligned(w, 16) && aligned(bias, 16) && aligned(out, 16);
}

int row_projection(const void *a, int64_t a_ld, const void *w, const float *bias, void *out, int64_t out_ld, int64_t m,
                   int64_t n, int64_t k, hipStream_t stream)
{
    if (!row_projection_supports(a, a_ld, w, bias, out, out_ld, m, n, k)) {
        return KUTACC_HIP_EUNSUPPORTED;
    }
    return k == 128 ? launch_output_projection<128>(a, a_ld, w, bias, out, out_ld, m, n, stream)
                    : launch_output_projection<256>(a, a_ld, w, bias, out, out_ld, m, n, stream);
}

// acc[m, n] += bf16(sum_k a[m, k] * w[n, k] + bias[n]) * sigmoid(gate[m, n]): same shapes as row_projection
int row_projection_gated_residual(const void *a, int64_t a_ld, const void *w, const float *bias, const void *gate,
                                  int64_t gate_ld, void *acc, int64_t acc_ld, int64_t m, int64_t n, int64_t k,
                                  hipStream_t stream)
{
    if (!row_projection_supports(a, a_ld, w, bias, acc, acc_ld, m, n, k) || !gate || gate_ld % 8 != 0 || !aligned(gate, 16)) {
        return KUTACC_HIP_EUNSUPPORTED;
    }
    return k == 128 ? launch_output_projection<128, EPILOGUE_GATED_RESIDUAL>(a, a_ld, w, bias, acc, acc_ld, m, n, stream, gate, gate_ld)
                    : launch_output_projection<256, EPILOGUE_GATED_RESIDUAL>(a, a_ld, w, bias, acc, acc_ld, m, n, stream, gate, gate_ld);
}

} // namespace kutacc_launch

// ------------------------------------------------------------------------------------------------
// Entry point that allocates nothing: the fragment-major copy of the pair bias -- the one scratch buffer of the fused
// path, which kutacc_hip_gating_attention keeps in the caller's q tensor -- lives in a device array that is part of the
// library image.  Every GPU the library runs on holds its own copy of the array, at its own address, until the process
// ends; the address is asked for once per device and kept.
// ------------------------------------------------------------------------------------------------
namespace {
constexpr size_t STATIC_SCRATCH_BYTES = (size_t)KUTACC_HIP_STATIC_SCRATCH_BYTES;
}
static __device__ __align__(256) unsigned char scratch[STATIC_SCRATCH_BYTES];

namespace {
std::atomic<void *> g_scratch_ptr[KUTACC_DEVICE_SLOTS];

// device address of `scratch` on the current device (the array's name is a host-side stand-in, never a device address)
int static_scratch_address(void **out)
{
    const int slot = kutacc_device_slot();
    if (slot < 0) {
        return KUTACC_HIP_EUNSUPPORTED;
    }
    void *ptr = g_scratch_ptr[slot].load(std::memory_order_acquire);
    if (ptr == nullptr) {
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || ptr == nullptr) {
            return e != hipSuccess ? (int)e : KUTACC_HIP_EUNSUPPORTED;
        }
        g_scratch_ptr[slot].store(ptr, std::memory_order_release); // every thread gets the same answer for a device
    }
    *out = ptr;
    return 0;
}
} // namespace

extern "C" kutacc_export int kutacc_hip_gating_attention_static(const kutacc_hip_attention_args_t *a, void *stream)
{
    if (!a || !a->input || !a->query_w || !a->key_w || !a->value_w || !a->gating_w || !a->output_w || !a->gating_b ||
        !a->output_b || !a->bias || !a->out || !a->avg) {
        return KUTACC_HIP_EINVAL;
    }
    if (a->batch <= 0 || a->seq_len <= 0 || a->nheads <= 0 || a->head_size <= 0 || a->batch > INT32_MAX / a->seq_len ||
        a->nheads > INT32_MAX / a->head_size) {
        return KUTACC_HIP_EINVAL;
    }
    const int64_t C = a->nheads * a->head_size;
    if (a->input_ld < C || a->out_ld < C) {
        return KUTACC_HIP_EINVAL;
    }
    if (!kutacc_launch::fused_attention_supports(*a)) {
        return KUTACC_HIP_EUNSUPPORTED; // the shape-agnostic kernels need the caller's q, k, v and gate tensors
    }
    kutacc_launch::FusedAttentionOptions opt;
    if (a->nonbatched_bias != nullptr) {
        const int64_t need = fragment_bytes(a->nheads, (int)((a->seq_len + 31) / 32));
        if ((uint64_t)need > STATIC_SCRATCH_BYTES) {
            fprintf(stderr,
                    "kutacc_hip_gating_attention_static: the pair bias of %lld heads x %lld positions needs %lld bytes of "
                    "scratch, the library's static array holds %zu\n",
                    (long long)a->nheads, (long long)a->seq_len, (long long)need, STATIC_SCRATCH_BYTES);
            return KUTACC_HIP_EINVAL;
        }
        void *ptr = nullptr;
        if (const int rc = static_scratch_address(&ptr)) {
            return rc;
        }
        opt.fragment_workspace = ptr;
        opt.fragment_workspace_bytes = STATIC_SCRATCH_BYTES;
    }
    kutacc_prof::Suppress no_events;
    return kutacc_launch::gating_attention_fused(*a, stream ? (hipStream_t)stream : kutacc_api::default_stream(), opt);
}

// Tuning hooks for tests and experiments: "plan" = "bpw,gw" forces the long-sequence kernel with that many query blocks
// per wave and weight matrices per group where it fits (anything else: the planner decides), "fragments" = "0" keeps the
// kernels off the fragment-major pair bias (general attention blocks), "debug" = "1" prints the plan of every call.
int kutacc_launch::fused_attention_tuning(const char *name, const char *value)
{
    const bool on = value && value[0] != '\0' && value[0] != '0';
    if (!strcmp(name, "plan")) {
        int bpw = 0, gw = 0;
        if (value && sscanf(value, "%d,%d", &bpw, &gw) == 2 && bpw >= 1 && bpw <= 4 && (gw == 1 || gw == 2 || gw == 4)) {
            g_forced_gw.store(gw), g_forced_bpw.store(bpw);
        } else {
            g_forced_bpw.store(0), g_forced_gw.store(0);
        }
        return 0;
    }
    if (!strcmp(name, "row_pairs")) { // "1": wherever the two-row kernel can run, "0": never, anything else: the default rule
        g_pair_mode.store(value && value[0] == '1' ? 1 : (value && value[0] == '0' ? 2 : 0));
        return 0;
    }
    if (!strcmp(name, "fragments")) {
        g_no_fragments.store((value && value[0] == '0') ? 1 : 0);
        return 0;
    }
    if (!strcmp(name, "debug")) {
        g_debug.store(on ? 1 : 0);
        return 0;
    }
    return KUTACC_HIP_EINVAL;
}
