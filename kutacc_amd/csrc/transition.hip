// The transition of the pair and MSA stacks (reference src/attention/transition.cpp:21-39) for gfx950, alone and as the
// whole block of an Evoformer layer: out += relu(LayerNorm(out) . W1^T + b1) . W2^T + b2 in place.
//
// The hidden layer (four fifths of the traffic if it went through memory, with c_i = 4 c_o) stays on chip.  A wave owns 32
// rows of x, as operand fragments in registers.  Both products are formed transposed (MFMA rows = hidden units, then output
// channels; columns = rows of x): the accumulators of the first, after ReLU and rounding to bf16, are the B operand of the
// second without leaving the registers.  For that, row i of a W1 block in the LDS is hidden unit sigma(i) (bits 2 and 3 of i
// swapped), which makes the eight values a lane holds per k-step consecutive hidden units.
//
// What bounds it: the clock and the rows' way in and out.  At 195072 rows, 256 -> 1024, the matrix pipes work for 58 % of the kernel's clocks (vector
// issue 32 %, both at once 10 %), at the 1.67 GHz that the chip holds under it; between a wave's loops over the weights lie its rows' load,
// LayerNorm, residual and store, which the other workgroup of the CU covers in part.  Weights come straight into the LDS
// (global_load_lds_dwordx4, no registers, no LDS write instructions) into a ring with one barrier per slice.
// The two products of a slice are a step apart: while W1 of slice j runs, W2 of slice j - 1 runs between its products, whose sums
// depend on each other; the hidden units of slice j are rounded beside the last products of W2, and every weight fragment leaves the LDS
// AHEAD products before its own.  With both products of one slice in a step a wave waited for the end of the first product, for its
// rounding and for most of its fragments.  A wave alone on its SIMD gains most: 20000 rows, 256 -> 1024 40.4 -> 35.0 us; 195072 rows 201
// -> 189 (1082 TFLOP/s), 400000 rows, 256 -> 512 263 -> 246, 147456 rows, 128 -> 256 33.6 -> 32.2, 64 -> 256 20.3 -> 18.9 (whole block, two sets of rows
// in turn).  Two workgroups or three per CU rather than one of twice the waves: one computes while the other fetches its rows or
// stores its result (400000 rows, 256 -> 512 232 against 245 us, 147456 rows, 128 -> 512 48 and 51).  Two sets of rows a wave, for half the fragments,
// leave no registers: 128 -> 512 70 us with 38 of them spilled.
//   195072 rows, 256 -> 1024, block: 328 us with weights through registers and one wave per SIMD; 500000 rows, 64 -> 256: 200 us in three
//   passes, 52 in this one.
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "launch_internal.h"
#include "mfma_tiles.h"
#include "profiler.h"


namespace {
using namespace kutacc_dev;

struct TransitionParams {
    const bf16_t *x, *w1, *w2;
    const float *b1, *b2, *ln_gamma, *ln_beta;
    bf16_t *out;
    int64_t rows;
    int c_i;
    float ln_eps;
    int full_groups, tail_waves; // workgroups whose waves all have rows, and how many waves of the others have
};

// 32 rows of x as they come from memory: lane (lane >> 3, lane & 7) holds chunk lane & 7 of every 64-channel panel of rows
// 8 i + (lane >> 3), and as operands of the first product
template <int CO>
struct Rows {
    PanelRegs panel[CO / 64];
};
template <int CO>
struct XFragments {
    bf16x8 f[CO / 16];
};

template <int CO>
__device__ __forceinline__ Rows<CO> load_rows(const bf16_t *x, int last_local, int lane)
{
    Rows<CO> t;
#pragma unroll
    for (int cp = 0; cp < CO / 64; ++cp) {
        t.panel[cp] = panel_load(x, CO, 0, last_local, cp * 64, lane);
    }
    return t;
}

// LayerNorm (arithmetic of reference src/normalization/layernorm_kernel.h:21-53; a row's chunks sit in 8 lanes: sums by DPP
// adds) if it is part of the block, then into fragment order through a private panel
template <int CO, bool BLOCK>
__device__ __forceinline__ XFragments<CO> fragments(Rows<CO> t, const TransitionParams &p, uint4 *panel, int lane)
{
    constexpr int CP = CO / 64;
    if constexpr (BLOCK) {
        float gm[CP][8], bt[CP][8];
#pragma unroll
        for (int cp = 0; cp < CP; ++cp) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                gm[cp][e] = p.ln_gamma[cp * 64 + (lane & 7) * 8 + e];
                bt[cp][e] = p.ln_beta[cp * 64 + (lane & 7) * 8 + e];
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint4 *regs[CP];
#pragma unroll
            for (int cp = 0; cp < CP; ++cp) {
                regs[cp] = i == 0 ? &t.panel[cp].r0 : i == 1 ? &t.panel[cp].r1 : i == 2 ? &t.panel[cp].r2 : &t.panel[cp].r3;
            }
            const float x0 = __shfl(to_f32(as_bf16x8(*regs[0])[0]), lane & ~7, 64); // first element of the row
            float s1 = 0.f, s2 = 0.f;
#pragma unroll
            for (int cp = 0; cp < CP; ++cp) {
                const bf16x8 b = as_bf16x8(*regs[cp]);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float d = to_f32(b[e]) - x0;
                    s1 += d;
                    s2 = fmaf(d, d, s2);
                }
            }
            float rstd, shift;
            norm_from_sums<true>(group_sum<8>(s1), group_sum<8>(s2), x0, (float)CO, p.ln_eps, rstd, shift);
#pragma unroll
            for (int cp = 0; cp < CP; ++cp) {
                const bf16x8 b = as_bf16x8(*regs[cp]);
                bf16x8 o;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    o[e] = (bf16_t)fmaf(fmaf(to_f32(b[e]), rstd, shift), gm[cp][e], bt[cp][e]);
                }
                *regs[cp] = as_uint4(o);
            }
        }
    }
    XFragments<CO> x;
#pragma unroll
    for (int cp = 0; cp < CP; ++cp) {
        panel_store(panel, lane, t.panel[cp]);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            x.f[cp * 4 + k] = as_bf16x8(panel[panel_slot(lane & 31, 2 * k + (lane >> 5))]);
        }
    }
    return x;
}

// One 32-hidden block's accumulator before its product, the bias: row 8 s + e stands for hidden unit 16 s + 8 g + e
__device__ __forceinline__ f32x16 hidden_bias(const float *b1, int g)
{
    f32x16 h;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const f32x4 b = *reinterpret_cast<const f32x4 *>(b1 + 16 * (q >> 1) + 4 * (q & 1) + 8 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            h[4 * q + e] = b[e];
        }
    }
    return h;
}

// ... and after it: ReLU, rounded to bf16 (the reference's rounding point: its intermediate is a bf16 tensor)
__device__ __forceinline__ bf16x8 hidden_operand(const f32x16 &h, int s)
{
    bf16x8 f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        f[e] = (bf16_t)__builtin_amdgcn_fmed3f(h[8 * s + e], 0.f, INFINITY); // fmaxf without an instruction that quiets the value; a NaN gives 0 as well
    }
    return f;
}

// 64 channels of 32 rows as store_channels adds to them and writes them: lane (lane >> 3, lane & 7) chunk lane & 7 of rows 8 i + (lane >> 3)
struct Residual {
    uint4 z[4];
};
template <int CO>
__device__ __forceinline__ Residual load_residual(const bf16_t *rows, int last_local, int channel, int lane)
{
    const PanelRegs t = panel_load(rows, CO, 0, last_local, channel, lane);
    return Residual{{t.r0, t.r1, t.r2, t.r3}};
}

// 64 channels of 32 rows: accumulators (+ b2) -> bf16 through the panel, out as whole 128-byte runs.  EARLY: the residual is there, else
// it is read where it is added
template <int CO, bool BLOCK, bool EARLY>
__device__ __forceinline__ void store_channels(const f32x16 &low, const f32x16 &high, const float *b2, const Residual &residual, bf16_t *rows, int last_local,
                                               int channel, uint4 *panel, int lane)
{
    const int r = lane & 31, g = lane >> 5;
#pragma unroll
    for (int n = 0; n < 2; ++n) {
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const f32x4 bv = *reinterpret_cast<const f32x4 *>(b2 + channel + n * 32 + 8 * a + 4 * g);
            bf16x4 ov;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                ov[c] = (bf16_t)((n ? high : low)[4 * a + c] + bv[c]);
            }
            *(reinterpret_cast<bf16x4 *>(panel + panel_slot(r, n * 4 + a)) + g) = ov;
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int prow = 8 * i + (lane >> 3);
        uint4 v = panel[panel_slot(prow, lane & 7)];
        if (prow <= last_local) {
            uint4 *dst = reinterpret_cast<uint4 *>(rows + (int64_t)prow * CO + channel + (lane & 7) * 8);
            if constexpr (BLOCK) { // residual: the row as it was before the LayerNorm
                const bf16x8 o = as_bf16x8(v), z = as_bf16x8(EARLY ? residual.z[i] : *dst);
                bf16x8 res;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    res[e] = (bf16_t)(to_f32(z[e]) + to_f32(o[e]));
                }
                v = as_uint4(res);
            }
            *dst = v;
        }
    }
}

// until at most N of a wave's own loads are on their way and none of its LDS reads
template <int N>
__device__ __forceinline__ void wait_and_barrier()
{
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"i"(N) : "memory");
}

// b2 lies behind b1 where a CU has one workgroup; where several share its LDS, in the place of b1's slices before the last one, once these have been read
// and if there are enough of them.  Always behind b1 it cost a CU its third workgroup at 128 -> 1088 and 1152 (300000 rows of the
// latter 181 us, 174 so) and its fourth at 64 -> 2048 (156, 153).
__host__ __device__ constexpr int b2_place(int c_o, int slice, int groups, int c_i) { return groups > 1 && c_i - slice >= c_o ? 0 : c_i; }

// SLICE: hidden units per stage of the ring of STAGES; GROUPS: workgroups a CU is meant to hold.
template <int CO, bool BLOCK, int SLICE, int STAGES, int WAVES, int GROUPS>
__global__ __launch_bounds__(64 * WAVES, GROUPS * WAVES / 4) void transition_rows_kernel(const TransitionParams p)
{
    constexpr int KS = CO / 16;                    // k-steps of the first product
    constexpr int CP = CO / 64;                    // 64-column panels across a row of x or W1
    constexpr int CB = CO / 32;                    // 32-channel blocks of the output
    constexpr int HB = SLICE / 32;
    constexpr int W1_SLOTS = SLICE * CO / 8, STAGE_SLOTS = 2 * W1_SLOTS;
    constexpr int UPW = STAGE_SLOTS / 64 / WAVES;  // loads of 1 KB a wave asks for per stage
    static_assert(SLICE == 32 || SLICE == 64, "layout of W2 slices");
    static_assert(WAVES * 256 <= STAGE_SLOTS && UPW >= 4, "the waves' panels lie in a stage; a wave's loads fill whole panels");
    extern __shared__ uint4 lds[]; // [STAGES][W1 slice, W2 slice], b1, and b2 (b2_place)
    static_assert(CP <= WAVES, "a thread brings one value of b2");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, g = lane >> 5, NJ = p.c_i / SLICE;
    float *b1s = reinterpret_cast<float *>(lds + STAGES * STAGE_SLOTS);
    float *b2s = b1s + b2_place(CO, SLICE, GROUPS, p.c_i);
    for (int i = tid; i < p.c_i; i += 64 * WAVES) {
        b1s[i] = p.b1[i]; // visible after the first barrier of the slice loop
    }
    float b2_value = 0.f;
    if (wave < CP) {
        b2_value = p.b2[wave * 64 + lane];
        if constexpr (GROUPS == 1) {
            b2s[wave * 64 + lane] = b2_value;
        }
    }

    const int past = (int)blockIdx.x - p.full_groups;
    const bool has_rows = past < 0 || wave < p.tail_waves; // the other waves only bring weights
    int64_t row0 = (past < 0 ? (int64_t)blockIdx.x * WAVES + wave : (int64_t)p.full_groups * WAVES + (int64_t)past * p.tail_waves + wave) * 32;
    const bool active = has_rows && row0 < p.rows;
    if (!active) {
        row0 = p.rows - 1; // keeps every address valid; nothing is stored
    }
    const int last_local = (int)(p.rows - row0 < 32 ? p.rows - row0 : 32) - 1;
    const Rows<CO> t = load_rows<CO>(p.x + row0 * CO, last_local, lane);

    // The first half of the waves brings the W1 slices, the second the W2 slices.
    const uint32_t lds0 = (uint32_t)(uintptr_t)(const lds_char *)lds;
    const bool first_matrix = wave < WAVES / 2;
    const int unit0 = wave % (WAVES / 2) * UPW; // within its matrix
    uint32_t lane_bytes[2];
#pragma unroll
    for (int hi = 0; hi < 2; ++hi) { // rows 16-31 of a panel swizzle with bit 0 flipped
        const int rl = lane >> 3;
        if (first_matrix) { // row i of the panel is hidden unit sigma(i): lane part of sigma
            lane_bytes[hi] = 2u * (uint32_t)(((rl & 3) | ((rl & 4) << 1)) * CO + 8 * ((lane & 7) ^ rl ^ hi));
        } else if constexpr (SLICE == 64) {
            lane_bytes[hi] = 2u * (uint32_t)(rl * p.c_i + 8 * ((lane & 7) ^ rl ^ hi));
        } else {
            lane_bytes[hi] = 2u * (uint32_t)((lane >> 2) * p.c_i + 8 * ((lane & 3) ^ ((lane >> 4) & 3)));
        }
    }
    const char *unit_src[UPW];
#pragma unroll
    for (int i = 0; i < UPW; ++i) {
        const int u = unit0 + i;
        int64_t e;
        if (first_matrix) {
            const int panel = u >> 2;
            e = (int64_t)((panel / CP) * 32 + 4 * (u & 1) + 16 * ((u >> 1) & 1)) * CO + (panel % CP) * 64;
        } else {
            e = (int64_t)u * (SLICE == 64 ? 8 : 16) * p.c_i;
        }
        unit_src[i] = reinterpret_cast<const char *>((first_matrix ? p.w1 : p.w2) + e);
    }
    const int64_t slice_bytes = first_matrix ? (int64_t)SLICE * CO * 2 : SLICE * 2;
    const uint32_t unit_lds = lds0 + (first_matrix ? 0u : W1_SLOTS * 16u) + (uint32_t)unit0 * 1024u;
    auto ask = [&](int slot) { // the next slice, into a stage
#pragma unroll
        for (int i = 0; i < UPW; ++i) {
            load_to_lds(unit_lds + (uint32_t)slot * (STAGE_SLOTS * 16u) + i * 1024u, unit_src[i], lane_bytes[(i >> 1) & 1]);
            unit_src[i] += slice_bytes;
        }
    };
    // Batch b of the loads: W1 of slice b and W2 of slice b - 1, which meet in step b of the loop.  A wave brings one matrix, so W1's
    // batches are 0 .. NJ - 1 and W2's 1 .. NJ.
    const int first_batch = first_matrix ? 0 : 1, last_batch = first_matrix ? NJ - 1 : NJ;
    auto ask_batch = [&](int batch) {
        if (batch >= first_batch && batch <= last_batch) {
            ask((first_matrix ? batch : batch - 1) % STAGES);
        }
    };
    for (int b = 0; b < STAGES - 1; ++b) {
        ask_batch(b);
    }

    const XFragments<CO> x = fragments<CO, BLOCK>(t, p, lds + (STAGES - 1) * STAGE_SLOTS + wave * 256, lane);

    f32x16 oacc[CB];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
        oacc[cb] = zero16();
    }
    const int w1_lane = panel_slot(r, g), w2_lane = SLICE == 64 ? w1_lane : r * 4 + (g ^ ((r >> 2) & 3));
    f32x16 h[HB];
    bf16x8 hf[HB][2];
    constexpr bool EARLY = CO != 64; // with 64 channels there are no registers for it
    Residual residual[CP];
    // Step j: W1 of slice j (if FIRST) and W2 of slice j - 1 (if SECOND), PRODUCTS of each.  Their operands come from the LDS AHEAD of their
    // use; the hidden units of slice j become operands while the last products of W2 run.
    constexpr int PRODUCTS = HB * KS, AHEAD = CO == 64 ? 2 : 3;
    auto step = [&](int j, auto has_first, auto has_second) __attribute__((always_inline)) {
        constexpr bool FIRST = decltype(has_first)::value, SECOND = decltype(has_second)::value;
        // batch j has landed (the later ones may be under way), and every wave is done with the stages of batch j - 1
        const int behind = max(0, min(STAGES - 2, last_batch - j));
        if (behind == 2) {
            wait_and_barrier<2 * UPW>();
        } else if (behind == 1) {
            wait_and_barrier<UPW>();
        } else {
            wait_and_barrier<0>();
        }
        ask_batch(j + STAGES - 1);
        if (!active) {
            return;
        }
        if constexpr (!FIRST && BLOCK && EARLY) { // the rows' place in the registers is free
            int lane = tid & 63; // opaque: its part of the addresses is formed here, not kept over the loop
            asm volatile("" : "+v"(lane));
#pragma unroll
            for (int cp = 0; cp < CP; ++cp) {
                residual[cp] = load_residual<CO>(p.out + row0 * CO, last_local, cp * 64, lane);
            }
        }
        const uint4 *w1 = lds + j % STAGES * STAGE_SLOTS, *w2 = lds + (j + STAGES - 1) % STAGES * STAGE_SLOTS + W1_SLOTS;
        if constexpr (FIRST) {
#pragma unroll
            for (int hb = 0; hb < HB; ++hb) {
                h[hb] = hidden_bias(b1s + j * SLICE + hb * 32, g);
            }
        }
        // product i of either matrix: of W1 k-step i / HB of hidden block i % HB, of W2 channels 32 (i % CB) by hidden units
        // 16 (i / CB) .. + 15 of the slice
        auto w1_fragment = [&](int i) {
            const int hb = i % HB, ks = i / HB;
            return as_bf16x8(w1[(hb * CP + ks / 4) * 256 + (w1_lane ^ (2 * (ks % 4)))]);
        };
        auto w2_fragment = [&](int i) {
            const int cb = i % CB, s = i / CB;
            return as_bf16x8(w2[SLICE == 64 ? cb * 256 + (w2_lane ^ (2 * s)) : cb * 128 + (w2_lane ^ (2 * s))]);
        };
        // the order: two of W1, one of W2, and so on, then the other half of W2's
        constexpr int TOTAL = (FIRST ? PRODUCTS : 0) + (SECOND ? PRODUCTS : 0);
        auto is_w1 = [](int m) { return FIRST && (!SECOND || (m < 3 * PRODUCTS / 2 && m % 3 != 2)); };
        auto index_of = [&](int m) {
            return !FIRST || !SECOND ? m : m >= 3 * PRODUCTS / 2 ? m - PRODUCTS : m % 3 == 2 ? m / 3 : m / 3 * 2 + m % 3;
        };
        auto fragment = [&](int m) { return is_w1(m) ? w1_fragment(index_of(m)) : w2_fragment(index_of(m)); };
        bf16x8 w[TOTAL];
#pragma unroll
        for (int m = 0; m < AHEAD; ++m) {
            w[m] = fragment(m);
        }
        bf16x8 next[HB][2];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < TOTAL; ++m) {
            const int i = index_of(m);
            if (is_w1(m)) {
                h[i % HB] = mfma(w[m], x.f[i / HB], h[i % HB]);
            } else {
                oacc[i % CB] = mfma(w[m], hf[i / CB / 2][i / CB % 2], oacc[i % CB]);
            }
            if (m + AHEAD < TOTAL) {
                w[m + AHEAD] = fragment(m + AHEAD);
            }
            if (FIRST && SECOND && m >= TOTAL - 2 * HB) { // one operand beside each of the last products
                const int q = m - (TOTAL - 2 * HB);
                next[q / 2][q % 2] = hidden_operand(h[q / 2], q % 2);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (FIRST) {
#pragma unroll
            for (int hb = 0; hb < HB; ++hb) {
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    hf[hb][s] = SECOND ? next[hb][s] : hidden_operand(h[hb], s);
                }
            }
        }
    };
    step(0, std::true_type{}, std::false_type{});
    for (int j = 1; j < NJ; ++j) {
        step(j, std::true_type{}, std::true_type{});
    }
    if (GROUPS > 1 && wave < CP) { // of b1, only the last slice may still be read
        b2s[wave * 64 + lane] = b2_value;
    }
    step(NJ, std::false_type{}, std::true_type{});

    if (!active) {
        return;
    }
    uint4 *panel = lds + NJ % STAGES * STAGE_SLOTS + wave * 256; // a stage that no wave reads any more
    int lane_o = lane;
    if constexpr (CO == 256) { // opaque, as above: no register to spare
        asm volatile("" : "+v"(lane_o));
    }
#pragma unroll
    for (int cp = 0; cp < CP; ++cp) {
        store_channels<CO, BLOCK, EARLY>(oacc[2 * cp], oacc[2 * cp + 1], b2s, residual[cp], p.out + row0 * CO, last_local, cp * 64, panel, lane_o);
    }
}

// Few rows: the time is that of one wave's chain through all hidden units (37 us for 256 -> 1024).  Here the four waves of a
// workgroup share 32 rows: each takes every fourth block of 32 hidden units, whose weights it brings into its own part of the
// LDS (no barrier; W1 of the next block while W2 of this one is used), and the four partial results are added in the LDS.
// 2048 rows: 256 -> 1024 20 us against 37 on the kernel above, 128 -> 512 9.3 against 13.4.  All weights pass through every
// CU's L1, 1 MB in about 8 us.
template <int CO, bool BLOCK, int WAVES>
__global__ __launch_bounds__(64 * WAVES, WAVES / 4) void transition_split_kernel(const TransitionParams p)
{
    constexpr int KS = CO / 16, CP = CO / 64, CB = CO / 32, UNITS = CO / 16; // UNITS: loads of 1 KB for 32 hidden units of either matrix
    constexpr int W1_SLOTS = 4 * CO, WAVE_SLOTS = 2 * W1_SLOTS;
    extern __shared__ uint4 lds[]; // [waves][W1 block, W2 block], [waves][panel], b1
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, g = lane >> 5, NB = p.c_i / 32;
    uint4 *mine = lds + wave * WAVE_SLOTS, *panel = lds + WAVES * WAVE_SLOTS + wave * 256;
    float *b1s = reinterpret_cast<float *>(lds + WAVES * (WAVE_SLOTS + 256));
    const int64_t row0 = (int64_t)blockIdx.x * 32;
    const int last_local = (int)(p.rows - row0 < 32 ? p.rows - row0 : 32) - 1;
    const Rows<CO> t = load_rows<CO>(p.x + row0 * CO, last_local, lane);

    const uint32_t to = (uint32_t)(uintptr_t)(const lds_char *)mine;
    const int rl = lane >> 3;
    uint32_t w1_bytes[2]; // row i of a panel is hidden unit sigma(i); rows 16-31 swizzle with bit 0 flipped
#pragma unroll
    for (int hi = 0; hi < 2; ++hi) {
        w1_bytes[hi] = 2u * (uint32_t)(((rl & 3) | ((rl & 4) << 1)) * CO + 8 * ((lane & 7) ^ rl ^ hi));
    }
    const uint32_t w2_bytes = 2u * (uint32_t)((lane >> 2) * p.c_i + 8 * ((lane & 3) ^ ((lane >> 4) & 3)));
    auto ask_w1 = [&](int block) {
        const bf16_t *from = p.w1 + (int64_t)block * 32 * CO;
#pragma unroll
        for (int u = 0; u < UNITS; ++u) {
            load_to_lds(to + u * 1024u, from + (4 * (u & 1) + 16 * ((u >> 1) & 1)) * CO + (u >> 2) * 64, w1_bytes[(u >> 1) & 1]);
        }
    };
    auto ask_w2 = [&](int block) {
        const bf16_t *from = p.w2 + block * 32;
#pragma unroll
        for (int u = 0; u < UNITS; ++u) {
            load_to_lds(to + W1_SLOTS * 16u + u * 1024u, from + (int64_t)u * 16 * p.c_i, w2_bytes);
        }
    };
    if (wave < NB) {
        ask_w1(wave);
        ask_w2(wave);
    }
    for (int i = tid; i < p.c_i; i += 64 * WAVES) {
        b1s[i] = p.b1[i];
    }
    const XFragments<CO> x = fragments<CO, BLOCK>(t, p, panel, lane);
    __syncthreads(); // b1

    f32x16 oacc[CB];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
        oacc[cb] = zero16();
    }
    const int w1_lane = panel_slot(r, g), w2_lane = r * 4 + (g ^ ((r >> 2) & 3));
    for (int block = wave; block < NB; block += WAVES) {
        const bool more = block + WAVES < NB;
        wait_for_loads<UNITS>(); // all but W2's
        f32x16 h = hidden_bias(b1s + block * 32, g);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            h = mfma(as_bf16x8(mine[(ks / 4) * 256 + (w1_lane ^ (2 * (ks % 4)))]), x.f[ks], h);
        }
        if (more) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // this block's fragments are out of the LDS
            ask_w1(block + WAVES);
            wait_for_loads<UNITS>(); // all but the next W1's
        } else {
            wait_for_loads<0>();
        }
        const bf16x8 hf[2] = {hidden_operand(h, 0), hidden_operand(h, 1)};
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                oacc[cb] = mfma(as_bf16x8(mine[W1_SLOTS + cb * 128 + (w2_lane ^ (2 * s))]), hf[s], oacc[cb]);
            }
        }
        if (more) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            ask_w2(block + WAVES);
        }
    }

    Residual residual;
    if (BLOCK && wave < CB / 2) {
        residual = load_residual<CO>(p.out + row0 * CO, last_local, wave * 64, lane);
    }
    // the waves' sums, each in its own region, then 64 channels a wave
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            *reinterpret_cast<f32x4 *>(mine + (cb * 4 + q) * 64 + lane) = f32x4{oacc[cb][4 * q], oacc[cb][4 * q + 1], oacc[cb][4 * q + 2], oacc[cb][4 * q + 3]};
        }
    }
    __syncthreads();
    if (wave < CB / 2) {
        f32x16 sum[2] = {zero16(), zero16()};
        for (int w = 0; w < WAVES; ++w) {
#pragma unroll
            for (int n = 0; n < 2; ++n) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const f32x4 part = *reinterpret_cast<const f32x4 *>(lds + w * WAVE_SLOTS + ((2 * wave + n) * 4 + q) * 64 + lane);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        sum[n][4 * q + e] += part[e];
                    }
                }
            }
        }
        store_channels<CO, BLOCK, true>(sum[0], sum[1], p.b2, residual, p.out + row0 * CO, last_local, wave * 64, panel, lane);
    }
}

constexpr int MAX_HIDDEN = 2048; // hidden units whose bias fits next to the weight stages in LDS

template <int CO, bool BLOCK, int SLICE, int STAGES, int WAVES, int GROUPS>
hipError_t launch_rows(TransitionParams p, hipStream_t stream)
{
    static size_t configured[KUTACC_DEVICE_SLOTS] = {};
    const size_t stages = (size_t)STAGES * SLICE * CO * 4;
    const auto kernel = &transition_rows_kernel<CO, BLOCK, SLICE, STAGES, WAVES, GROUPS>;
    if (const hipError_t e = kutacc_opt_in_lds(reinterpret_cast<const void *>(kernel), stages + (MAX_HIDDEN + CO) * sizeof(float), configured)) {
        return e;
    }
    // Full rounds of workgroups, then the rest dealt evenly over the CUs, as few waves with rows per workgroup as that takes
    // (147456 rows of 256 channels fill 2.25 rounds: 186 us with a third round of full workgroups on a quarter of the chip,
    // 172 so).
    const int64_t row_blocks = (p.rows + 31) / 32, cus = kutacc_cu_count();
    p.full_groups = (int)(row_blocks / (cus * GROUPS * WAVES) * cus * GROUPS);
    const int64_t rest = row_blocks - (int64_t)p.full_groups * WAVES, per_cu = std::max<int64_t>(1, (rest + cus - 1) / cus);
    const int64_t groups = (per_cu + WAVES - 1) / WAVES;
    p.tail_waves = (int)((per_cu + groups - 1) / groups);
    const int64_t blocks = p.full_groups + (rest + p.tail_waves - 1) / p.tail_waves;
    kernel<<<dim3((unsigned)blocks), 64 * WAVES, stages + (size_t)std::max(p.c_i, b2_place(CO, SLICE, GROUPS, p.c_i) + CO) * sizeof(float), stream>>>(p);
    return hipGetLastError();
}

template <int CO, bool BLOCK, int WAVES>
hipError_t launch_split(const TransitionParams &p, hipStream_t stream)
{
    static size_t configured[KUTACC_DEVICE_SLOTS] = {};
    const size_t fixed = (size_t)WAVES * (CO * 128 + 4096);
    const auto kernel = &transition_split_kernel<CO, BLOCK, WAVES>;
    if (const hipError_t e = kutacc_opt_in_lds(reinterpret_cast<const void *>(kernel), fixed + MAX_HIDDEN * sizeof(float), configured)) {
        return e;
    }
    kernel<<<dim3((unsigned)((p.rows + 31) / 32)), 64 * WAVES, fixed + (size_t)p.c_i * sizeof(float), stream>>>(p);
    return hipGetLastError();
}
template <bool BLOCK>
hipError_t launch(const TransitionParams &p, int64_t c_o, hipStream_t stream)
{
    const double flops = 4.0 * (double)p.rows * (double)c_o * (double)p.c_i;
    // The split kernel while its workgroups of 32 rows fit one round on the chip: in a second round it takes as long as the
    // other kernel (12000 rows, 256 -> 1024: 39 and 38 us; 128 -> 512: 18 and 14).  With 64 channels all is within 7 us.
    const int64_t blocks = (p.rows + 31) / 32, cus = kutacc_cu_count();
    const bool few = c_o != 64 && blocks <= cus;
    // While eight waves a CU take all rows, they are one workgroup, which brings the weights once, in four stages or in slices of twice the size.  Against
    // two or three workgroups (us): 256 -> 1024 40000 rows 53.7 51.7, 50000 58.7 55.4, 65000 66.9 63.7, 128 -> 512 9000 rows 12.9 12.15, 30000 14.6 13.7,
    // 65000 22.3 20.2, 128 -> 256 20000 10.1 9.9, 50000 15.2 13.4.  Beyond, a second round of it costs: 80000 89.5 94.2, 27.6 30.9.  With 256 channels and up
    // to four waves a CU no gain: 256 -> 1024 20000 34.1 34.0, 256 -> 512 22.0 22.5.  Few hidden units are one or two slices of twice the size, whose two
    // products cannot run side by side, which up to four waves a CU do not make up for: 128 -> 64 9000 rows 6.6 7.2, 32768 7.5 8.0, 40000 9.3 9.1, 65536 10.4 9.5,
    // 128 -> 128 9000 7.6 8.0, 24577 8.3 8.5, 33000 10.7 10.0; 256 -> 64 50000 17.6 17.9, 65536 19.3 19.4.
    const bool one_round = blocks <= 8 * cus && (c_o == 128 ? p.c_i > 128 || blocks > 4 * cus : p.c_i > 64 && blocks > 4 * cus);
    kutacc_prof::KernelTimer t(few ? (BLOCK ? "transition_split_kernel<block>" : "transition_split_kernel")
                                   : (BLOCK ? "transition_rows_kernel<block>" : "transition_rows_kernel"),
                               flops, stream);
    if (c_o == 256) {
        return few ? launch_split<256, BLOCK, 4>(p, stream) : one_round ? launch_rows<256, BLOCK, 32, 4, 8, 1>(p, stream) : launch_rows<256, BLOCK, 32, 2, 4, 2>(p, stream);
    }
    if (c_o == 128) {
        return few ? launch_split<128, BLOCK, 4>(p, stream) : one_round ? launch_rows<128, BLOCK, 64, 2, 8, 1>(p, stream) : launch_rows<128, BLOCK, 32, 3, 4, 3>(p, stream);
    }
    if constexpr (BLOCK) {
        return launch_rows<64, true, 64, 2, 4, 4>(p, stream);
    }
    return hipErrorInvalidValue;
}
} // namespace

namespace kutacc_launch {

static bool operands_fit(int64_t rows, int64_t c_i, const void *x, const void *w1, const float *b1, const void *w2, const float *b2, const void *out)
{
    return c_i >= 64 && c_i % 64 == 0 && c_i <= MAX_HIDDEN && rows > 0 && rows <= ((int64_t)1 << 31) * 32 && kutacc_hip_aligned16(x) &&
           kutacc_hip_aligned16(w1) && kutacc_hip_aligned16(b1) && kutacc_hip_aligned16(w2) && kutacc_hip_aligned16(b2) && kutacc_hip_aligned16(out);
}

bool transition_fused_supports(int64_t rows, int64_t c_o, int64_t c_i, const void *x, const void *w1, const float *b1,
                               const void *w2, const float *b2, const void *out)
{
    return (c_o == 128 || c_o == 256) && operands_fit(rows, c_i, x, w1, b1, w2, b2, out);
}

int transition_fused(const void *x, const void *w1, const float *b1, const void *w2, const float *b2, void *out,
                     int64_t rows, int64_t c_o, int64_t c_i, hipStream_t stream)
{
    if (!transition_fused_supports(rows, c_o, c_i, x, w1, b1, w2, b2, out)) {
        return KUTACC_HIP_EUNSUPPORTED;
    }
    const TransitionParams p = {(const bf16_t *)x, (const bf16_t *)w1, (const bf16_t *)w2, b1, b2, nullptr, nullptr, (bf16_t *)out, rows, (int)c_i, 0.f};
    return kutacc_hip_status(launch<false>(p, c_o, stream));
}

// act += transition(LayerNorm(act)) in place, one kernel (64 channels too: the operator alone keeps its two products there,
// which leave the hidden layer where the caller asked for it)
int transition_block_fused(void *act, const float *ln_gamma, const float *ln_beta, float ln_eps, const void *w1, const float *b1,
                           const void *w2, const float *b2, int64_t rows, int64_t c_o, int64_t c_i, hipStream_t stream)
{
    if (!ln_gamma || !ln_beta || (c_o != 64 && c_o != 128 && c_o != 256) || !operands_fit(rows, c_i, act, w1, b1, w2, b2, act)) {
        return KUTACC_HIP_EUNSUPPORTED;
    }
    const TransitionParams p = {(const bf16_t *)act, (const bf16_t *)w1, (const bf16_t *)w2, b1, b2, ln_gamma, ln_beta, (bf16_t *)act, rows, (int)c_i, ln_eps};
    return kutacc_hip_status(launch<true>(p, c_o, stream));
}

} // namespace kutacc_launch
