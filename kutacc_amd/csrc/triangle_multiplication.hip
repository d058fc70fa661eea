// The two ends of the triangle-multiplication block at 128 channels (reference
// src/attention/triangle_multiplication.cpp:25-150 with the LayerNorms and the residual a caller adds around it).  Between
// them lies the equation, one n x n product per channel (pair_stack.hip).
//
// Layout of the intermediates.  The projections and the centre are channel-first, one plane per channel, and a plane's
// rows are n positions padded to a pitch of np, n rounded up to 8 (to 32, and for incoming edges the rows too, where the
// product takes whole steps of that): every row then starts on 16 bytes, whatever n is, and the products run on the matrix
// cores with vector loads at every length.  The projections write zeros into the padding
// (their mask is zero there), so a contraction over np positions is one over n.  With dense rows an n that is no multiple
// of 8 left the product to scalar loads: 217 ms for the block at 691 residues, 0.39 ms so.
//
// Both kernels take the padded positions p = i np + j in steps of 64.  Eight consecutive positions share the row i, because
// np is a multiple of 8: a wave follows (i, j) of its eights with scalar additions.
//
// Both are bound by vector issue as much as by HBM, and by power: at 384 residues each moves its 113 MB
// (front: 256 bytes in, 512 out per position; back: 512 in, 256 out) in 37 to 38 us, 60 % of the rate of a copy,
// with the vector issue ports taken for some 60 % of the clocks and the matrix cores for 29 and 15.  Neither reads a normalised copy of the pair activation: the front kernel normalises the rows on their way into the LDS, the back kernel does it again for
// its gate, from the same rows that its residual needs.  At 384 residues that saves a pass of 76 MB and a read of 38 MB.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "launch_internal.h"
#include "mfma_tiles.h"
#include "profiler.h"

namespace {
using namespace kutacc_dev;

constexpr int C = 128, CK = C / 16;
constexpr int STEP = 64;              // positions per step
constexpr int ROW_SLOTS = C * 2 / 16; // 16-byte slots of a position's row

// (i, j) of the first of eight consecutive padded positions
struct Place {
    int i, j;
};

__device__ __forceinline__ Place place_of(uint32_t p, uint32_t np) { return Place{(int)(p / np), (int)(p % np)}; }

__device__ __forceinline__ void advance(Place &q, int np)
{
    q.j += STEP;
    while (q.j >= np) {
        q.j -= np, ++q.i;
    }
}

// Rows of the pair activation in the LDS: [64 positions][16 slots], the slot index XOR-ed with position % 16: a fragment read, lane -> its
// own position, is served sixteen lanes at a time (0-3, 12-15, 20-23, 24-27 and so on: sixteen different positions modulo 16), which then
// fall on all sixteen bank groups.  With position % 8 two of them shared each: 2/3 of the conflicts of either kernel, 1 % of the
// block (384 residues 101.8 -> 101.1 us, 1024 725.8 -> 721.0).
__device__ __forceinline__ int row_slot(int pos, int chunk) { return pos * ROW_SLOTS + (chunk ^ (pos & 15)); }

// LayerNorm of a row of 128 channels held by 16 consecutive lanes, 8 each: the arithmetic of layernorm_rows_bf16_kernel
// (reference src/normalization/layernorm_kernel.h:21-53)
__device__ __forceinline__ uint4 normalise_row(uint4 raw, int lane, const float (&gm)[8], const float (&bt)[8], float eps)
{
    const bf16x8 b = as_bf16x8(raw);
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        v[e] = to_f32(b[e]);
    }
    float rstd, shift;
    group_stats<16>(v, __shfl(v[0], lane & ~15, 64), (float)C, eps, rstd, shift);
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        o[e] = (bf16_t)fmaf(fmaf(v[e], rstd, shift), gm[e], bt[e]);
    }
    return as_uint4(o);
}

struct Side {
    const bf16_t *wp, *wg;
    const float *bp, *bg;
    bf16_t *out;
};

// LayerNorm and both gated projections: out[c][p] = bf16(bf16(y . wp[c] + bp[c]) * mask * sigmoid(y . wg[c] + bg[c])), y the
// normalised row of position p.  Sixteen waves, one workgroup per CU; a wave owns 16 channels of one side and keeps its two
// 16 x 128 weight blocks in 32 registers.  Per step it normalises four of the 64 rows, loaded two steps ahead, into the
// shared stage, multiplies the whole stage and writes 16 channels x 128 bytes.  Same arithmetic in the same order as
// LayerNorm followed by gated_projection_kernel: the results are bit-identical (a 16x16x32 product sums as two 32x32x16 ones do).
//
// Four waves a SIMD of 16 channels instead of two of 32: the older of two waves was through a step in 5500 clocks and waited 2000 at the
// barrier for the younger, which it had kept from issuing; products whose rows are channels leave a lane one mask a product and 18 % fewer
// vector instructions.  This kernel, us: 691 residues 101.4 -> 97.5, 1024 213.5 -> 205.7, 384 38.4 -> 38.2.  No barrier at all, with the weights of
// both sides in the LDS and 32 positions x 256 outputs a wave: 116, 213 and 41.6; one of two waves half a step behind the other: no difference.
constexpr int FRONT_WAVES = 16;
constexpr int FRONT_STAGE = STEP * ROW_SLOTS;
constexpr int FRONT_PANEL = STEP * 32; // bytes of a wave's panel: 64 positions x 16 channels
constexpr size_t FRONT_LDS = (size_t)2 * FRONT_STAGE * 16 + FRONT_WAVES * FRONT_PANEL + 2 * C * sizeof(float) + 2 * STEP * 2;

__global__ __launch_bounds__(64 * FRONT_WAVES, 1) void triangle_front_kernel(const bf16_t *__restrict__ x, const float *__restrict__ gamma,
                                                                             const float *__restrict__ beta, float eps, Side s0, Side s1,
                                                                             const bf16_t *__restrict__ mask, int64_t plane, int n, int rows,
                                                                             int np, int steps_per_group)
{
    extern __shared__ uint4 lds[]; // two stages, a panel per wave, gamma and beta, two mask rows
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, chunk = lane >> 4; // operands: row or column, eight k; results: column, rows 4 chunk .. + 3
    const Side &sd = wave >= 8 ? s1 : s0;
    const int cb = wave & 7; // this wave's 16 channels
    char *const panel = reinterpret_cast<char *>(lds + 2 * FRONT_STAGE) + wave * FRONT_PANEL;
    float *norm = reinterpret_cast<float *>(reinterpret_cast<char *>(lds + 2 * FRONT_STAGE) + FRONT_WAVES * FRONT_PANEL);
    uint16_t *mask_rows = reinterpret_cast<uint16_t *>(norm + 2 * C);

    const int positions = rows * np, total_steps = (positions + STEP - 1) / STEP;
    const int first = (int)blockIdx.x * steps_per_group;
    const int stop = first + steps_per_group < total_steps ? first + steps_per_group : total_steps;
    if (first >= stop) {
        return;
    }

    // This wave's four rows of a step, half of an eight: lane (l / 16, l % 16) holds chunk l % 16 of row l / 16.  Padding
    // repeats the row's last position, steps past the end repeat the last row: valid addresses, results masked or dropped.
    struct Rows {
        uint4 r;
        uint16_t m; // mask of the lane's position, if there is such a position
        bool there;
    };
    Place at = place_of((uint32_t)(first * STEP + 8 * (wave >> 1)), (uint32_t)np);
    auto load = [&](Rows &t) __attribute__((always_inline)) {
        const int i = min(at.i, n - 1), j = at.j + 4 * (wave & 1) + chunk;
        t.there = at.i < n && j < n;
        const uint32_t here = (uint32_t)min(j, n - 1);
        const char *row = reinterpret_cast<const char *>(x + (int64_t)i * n * C);
        t.r = *reinterpret_cast<const uint4 *>(row + (here * (2u * C) + 16u * col));
        t.m = reinterpret_cast<const uint16_t *>(mask + (int64_t)i * n)[here];
        advance(at, np);
    };
    auto stage_rows = [&](const Rows &t, int s) __attribute__((always_inline)) {
        float gm[8], bt[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            gm[e] = norm[8 * col + e], bt[e] = norm[C + 8 * col + e];
        }
        lds[s * FRONT_STAGE + row_slot(4 * wave + chunk, col)] = normalise_row(t.r, lane, gm, bt, eps);
        if (col == 0) {
            mask_rows[s * STEP + 4 * wave + chunk] = t.there ? t.m : (uint16_t)0;
        }
    };

    Rows even, odd;
    load(even);
    load(odd);
    if (tid < C) {
        norm[tid] = gamma[tid], norm[C + tid] = beta[tid];
    }
    bf16x8 wp[4], wg[4];
    f32x4 pbias, gneg;
    // in half lines, 16 rows by 32 channels a load, and into operand order through the panel (one load in operand order takes the address
    // path some 42 cycles instead of 16, and there are 128)
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        const int at = (cb * 16 + (lane >> 2)) * C + ks * 32 + (lane & 3) * 8;
        wp[ks] = *reinterpret_cast<const bf16x8 *>(sd.wp + at);
        wg[ks] = *reinterpret_cast<const bf16x8 *>(sd.wg + at);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        pbias[v] = sd.bp[cb * 16 + 4 * chunk + v], gneg[v] = -LOG2E * sd.bg[cb * 16 + 4 * chunk + v];
    }
    char *out = reinterpret_cast<char *>(sd.out + (int64_t)cb * 16 * plane);
    __syncthreads();
    stage_rows(even, 0);
    uint4 *own = reinterpret_cast<uint4 *>(panel);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        own[half_line_slot(lane >> 2, lane & 3)] = as_uint4(wp[ks]);
        own[64 + half_line_slot(lane >> 2, lane & 3)] = as_uint4(wg[ks]);
        wp[ks] = as_bf16x8(own[half_line_slot(col, chunk)]);
        wg[ks] = as_bf16x8(own[64 + half_line_slot(col, chunk)]);
    }
    __syncthreads();
    // The weights are waited for here: the waits that the compiler leaves to their first uses stand in the loop, where they are waits for
    // all rows and stores on their way.
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        asm volatile("" ::"v"(wp[ks]), "v"(wg[ks]));
    }
    asm volatile("" ::"v"(pbias), "v"(gneg));
    auto product = [](bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); };

    auto do_step = [&](int step, int s, Rows &next, Rows &after) __attribute__((always_inline)) {
        load(after); // (behind the last step as well: every step has the same loads and stores, and the wait for `next` lets them fly)
        if (step + 1 < stop) {
            stage_rows(next, s ^ 1);
        }
        const uint4 *stage = lds + s * FRONT_STAGE;
        const uint16_t *mask_row = mask_rows + s * STEP;
        // The panel: [64 positions][4 chunks of 4 channels], the chunk XOR-ed with 2 (position / 4 % 2), under which these writes and the
        // transposing reads below are free of bank conflicts.
        const uint32_t write_at = 32u * col + 8u * (uint32_t)(chunk ^ (2 * ((col >> 2) & 1)));
        auto multiply = [&](auto kept) __attribute__((always_inline)) {
#pragma unroll
            for (int pb = 0; pb < 4; ++pb) { // 16 positions
                f32x4 pa = {0.f, 0.f, 0.f, 0.f}, ga = pa;
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) {
                    const bf16x8 y = as_bf16x8(stage[row_slot(16 * pb + col, 4 * ks + chunk)]);
                    pa = product(wp[ks], y, pa);
                    ga = product(wg[ks], y, ga);
                }
                const float mk = decltype(kept)::value ? 1.0f : __uint_as_float((uint32_t)mask_row[16 * pb + col] << 16);
                bf16x4 pp, ov;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    pp[v] = (bf16_t)(pa[v] + pbias[v]);
                }
                asm volatile("" : "+v"(pp)); // else each value is rounded by itself
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    // sigmoid(gate + bias) = 1 / (1 + 2^-(gate*log2e + bias*log2e)); the gate stays in fp32
                    const float e = __builtin_amdgcn_exp2f(fmaf(ga[v], -LOG2E, gneg[v]));
                    ov[v] = (bf16_t)((decltype(kept)::value ? to_f32(pp[v]) : to_f32(pp[v]) * mk) * __builtin_amdgcn_rcpf(1.0f + e));
                }
                *reinterpret_cast<bf16x4 *>(panel + write_at + 512 * pb) = ov;
            }
        };
        // Positions that are all there are not multiplied by their masks: the same bits, 20 vector instructions of 370 a step and wave (whole block, two
        // activations in turn, us: 256 residues 46.9 -> 46.3, 384 92.5 -> 91.7, 1024 704 -> 700).
        if (__all(mask_row[lane] == 0x3f80)) {
            multiply(std::true_type{});
        } else {
            multiply(std::false_type{});
        }
        // 16 channels x eight 16-byte pieces of 8 positions; pieces past the last one repeat it.  A store: 16 channels x four pieces.
        const int last_piece = (positions - 1 - step * STEP) >> 3;
        char *const to = out + (int64_t)step * (2 * STEP);
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const uint32_t piece = (uint32_t)min(4 * half + chunk, last_piece);
            const lds_char *from = (const lds_char *)panel + (256u * piece + 32u * (col >> 2));
            const bf16x8 v = lds_transposed_fragment(from + 8 * (col & 3), from + (128 + 8 * ((col & 3) ^ 2)));
            *reinterpret_cast<uint4 *>(to + ((uint32_t)col * (uint32_t)plane * 2u + 16u * piece)) = as_uint4(v);
        }
        __syncthreads(); // the other stage is complete, this one no longer read
    };
    int step = first;
    while (true) {
        do_step(step, 0, odd, even);
        if (++step >= stop) {
            break;
        }
        do_step(step, 1, even, odd);
        if (++step >= stop) {
            break;
        }
    }
}

// x[i, j] += bf16(bf16(centre' . wo^T + bo) * sigmoid(bf16(y . wg^T + bg))), centre' the normalised centre of (i, j), y its
// normalised row of x.  Four waves, two workgroups per CU (the three barriers of a step of one are covered by the
// other); a wave owns 32 output features, keeps both 32 x 128 weight blocks in 64 registers and moves 16 of the step's 64
// positions: it normalises their rows of x, normalises their centre (which lies channel by channel in the stage; transposing
// LDS reads give a lane 32 channels of one position: exchanged between lanes the whole block took 94.7 us at 384 residues,
// 93.6 so, and 92.8 with the biases as the products' seeds), and finishes them with the
// residual, for which the rows of x have stayed in its registers.
// Four lanes hold a row of x: with sixteen, four rows a lane, their sums, scales, addresses and bounds were formed four times by each
// (1006 vector instructions a step and wave, 873 now, the pairs of rounded values among them).  This kernel, us: 384 residues 39.2 -> 37.5, 691
// 97.7 -> 93.3, 1024 203 -> 194.
constexpr int BACK_STAGE = STEP * ROW_SLOTS; // slots of each of the four stages: centre as it lies, y, centre', result
constexpr size_t BACK_LDS = (size_t)4 * BACK_STAGE * 16 + 6 * C * sizeof(float);

__global__ __launch_bounds__(256, 2) void triangle_back_kernel(const bf16_t *__restrict__ centre, int64_t plane, const float *__restrict__ c_gamma,
                                                               const float *__restrict__ c_beta, const bf16_t *__restrict__ wo,
                                                               const float *__restrict__ bo, const bf16_t *__restrict__ wg,
                                                               const float *__restrict__ bg, bf16_t *__restrict__ x,
                                                               const float *__restrict__ gamma, const float *__restrict__ beta, float eps,
                                                               int n, int np, int steps_per_group, int longer)
{
    extern __shared__ uint4 lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rv = lane & 31, gv = lane >> 5;
    uint4 *raw = lds, *ys = lds + BACK_STAGE, *cs = lds + 2 * BACK_STAGE, *res = lds + 3 * BACK_STAGE;
    float *params = reinterpret_cast<float *>(lds + 4 * BACK_STAGE); // gamma, beta, centre's gamma and beta, bo, bg
    // the first `longer` workgroups take one step more
    const int positions = n * np, id = (int)blockIdx.x;
    const int first = id * steps_per_group + min(id, longer), stop = first + steps_per_group + (id < longer ? 1 : 0);

    // rows of x: this wave's 16 positions of a step, four lanes each: lane l holds pieces l % 4 + 4 u of position 16 wave + l / 4
    struct RowOfX {
        uint4 r0, r1, r2, r3; // named members, so that they always live in registers
        uint32_t at;          // i n + j, of the position itself or of the last one in its place
        bool there;
    };
    Place at_lo = place_of((uint32_t)(first * STEP + 16 * wave), (uint32_t)np), at_hi = place_of((uint32_t)(first * STEP + 16 * wave + 8), (uint32_t)np);
    auto row_of_x = [&](uint32_t at, int ln) { return reinterpret_cast<char *>(x) + ((uint64_t)at * (2 * C) + 16u * (ln & 3)); };
    auto load_row = [&](RowOfX &t) {
        const int i = lane < 32 ? at_lo.i : at_hi.i, j = (lane < 32 ? at_lo.j : at_hi.j) + ((lane >> 2) & 7);
        t.there = i < n && j < n;
        t.at = (uint32_t)min(i, n - 1) * (uint32_t)n + (uint32_t)min(j, n - 1);
        const char *row = row_of_x(t.at, lane);
        t.r0 = *reinterpret_cast<const uint4 *>(row), t.r1 = *reinterpret_cast<const uint4 *>(row + 64);
        t.r2 = *reinterpret_cast<const uint4 *>(row + 128), t.r3 = *reinterpret_cast<const uint4 *>(row + 192);
        advance(at_lo, np), advance(at_hi, np);
    };
    // the centre: channels 32 wave + 8 i + lane / 8, positions 8 (lane % 8) .. + 7 of the step; past the end the last eight
    const uint32_t lane_plane = (uint32_t)(lane >> 3) * (uint32_t)plane * 2u;
    auto load_centre = [&](int step) {
        PanelRegs t;
        const uint32_t pos = (uint32_t)min(step * STEP + 8 * (lane & 7), positions - 8);
        const char *src = reinterpret_cast<const char *>(centre + (int64_t)(32 * wave) * plane);
        const int64_t eight = 16 * plane; // bytes of eight channels
        const uint32_t off = lane_plane + 2u * pos;
        t.r0 = *reinterpret_cast<const uint4 *>(src + off);
        t.r1 = *reinterpret_cast<const uint4 *>(src + eight + off);
        t.r2 = *reinterpret_cast<const uint4 *>(src + 2 * eight + off);
        t.r3 = *reinterpret_cast<const uint4 *>(src + 3 * eight + off);
        return t;
    };

    RowOfX row, next_row;
    PanelRegs ct = load_centre(first);
    load_row(row);
    next_row = row;
    bf16x8 wof[CK], wgf[CK];
    load_half_lines<CK>(wof, wo + wave * 32 * C, C, lane);
    load_half_lines<CK>(wgf, wg + wave * 32 * C, C, lane);
    half_lines_to_fragments<CK>(wof, res + 128 * wave, lane);
    half_lines_to_fragments<CK>(wgf, res + 128 * wave, lane);
    if (tid < C) {
        params[tid] = gamma[tid], params[C + tid] = beta[tid];
        params[2 * C + tid] = c_gamma[tid], params[3 * C + tid] = c_beta[tid];
        params[4 * C + tid] = bo[tid], params[5 * C + tid] = bg[tid];
    }
    __syncthreads();
    // waited for here, not at their first uses in the loop, where that is a wait for the next step's loads
#pragma unroll
    for (int ks = 0; ks < CK; ++ks) {
        asm volatile("" ::"v"(wof[ks]), "v"(wgf[ks]));
    }

    for (int step = first; step < stop; ++step) {
        int lv = lane; // opaque: LDS addresses are formed per step, not kept across the loop
        asm volatile("" : "+v"(lv));
        // the centre as it lies: [128 channels][8 slots], the slot XOR-ed with 2 (channel % 4) + channel / 4 % 2, under which the
        // transposing reads below (16 lanes: four channels, two slots) and these writes are free of bank conflicts
        {
            uint4 *mine = raw + (32 * wave + (lv >> 3)) * 8 + ((lv & 7) ^ (2 * ((lv >> 3) & 3) + (lv >> 5)));
            mine[0] = ct.r0, mine[64] = ct.r1, mine[128] = ct.r2, mine[192] = ct.r3;
        }
        if (step + 1 < stop) {
            ct = load_centre(step + 1);
        }
        {
            const bf16x8 v[4] = {as_bf16x8(row.r0), as_bf16x8(row.r1), as_bf16x8(row.r2), as_bf16x8(row.r3)};
            // the row's first element, in the first of its four lanes
            const float x0 = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(to_f32(v[0][0])), 0x00, 0xf, 0xf, false));
            float s1 = 0.f, s2 = 0.f, rstd, shift;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float d = to_f32(v[t][e]) - x0;
                    s1 += d;
                    s2 = fmaf(d, d, s2);
                }
            }
            s1 = dpp_add<0x4E>(dpp_add<0xB1>(s1)), s2 = dpp_add<0x4E>(dpp_add<0xB1>(s2)); // lanes ^ 1, ^ 2
            norm_from_sums<false>(s1, s2, x0, (float)C, eps, rstd, shift);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int chunk = 4 * t + (lv & 3);
                const float *gm = params + 8 * chunk, *bt = gm + C;
                bf16x8 o;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    o[e] = (bf16_t)fmaf(fmaf(to_f32(v[t][e]), rstd, shift), gm[e], bt[e]);
                }
                ys[row_slot(16 * wave + (lv >> 2), chunk)] = as_uint4(o);
            }
        }
        if (step + 1 < stop) {
            load_row(next_row);
        }
        __syncthreads();
        auto biases = [&](int which) { // of this wave's 32 features, in accumulator order: the seed of their products
            f32x16 b;
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const f32x4 v = *reinterpret_cast<const f32x4 *>(params + which * C + wave * 32 + 8 * a + 4 * (lv >> 5));
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    b[4 * a + c] = v[c];
                }
            }
            return b;
        };
        // gate: this wave's 32 features of all 64 positions, rounded to bf16
        bf16x8 gate[2][2];
        {
            f32x16 acc[2];
            acc[0] = acc[1] = biases(5);
#pragma unroll
            for (int ks = 0; ks < CK; ++ks) {
#pragma unroll
                for (int pb = 0; pb < 2; ++pb) {
                    acc[pb] = mfma(wgf[ks], as_bf16x8(ys[row_slot(32 * pb + (lv & 31), 2 * ks + (lv >> 5))]), acc[pb]);
                }
            }
#pragma unroll
            for (int pb = 0; pb < 2; ++pb) {
                gate[pb][0] = pack8(acc[pb], 0), gate[pb][1] = pack8(acc[pb], 8);
                asm volatile("" : "+v"(gate[pb][0]), "+v"(gate[pb][1])); // else each value is rounded by itself
            }
        }
        // the centre of this wave's positions: lane l takes channels 8 (l / 16) .. + 7 (+ 32 t) of position l % 16
        {
            const lds_char *from = (const lds_char *)raw + (lv >> 4) * 1024 + ((lv >> 2) & 3) * 128 + 8 * (lv & 1);
            const int slot = (2 * wave + ((lv >> 1) & 1)) ^ (2 * ((lv >> 2) & 3));
            bf16x8 v[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                v[t] = lds_transposed_fragment(from + t * 4096 + 16 * slot, from + t * 4096 + 512 + 16 * (slot ^ 1));
            }
            const float x0 = __shfl(to_f32(v[0][0]), lv & 15, 64);
            float s1 = 0.f, s2 = 0.f;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float d = to_f32(v[t][e]) - x0;
                    s1 += d;
                    s2 = fmaf(d, d, s2);
                }
            }
            float rstd, shift;
            norm_from_sums<true>(half_swap_sum(quarter_swap_sum(s1)), half_swap_sum(quarter_swap_sum(s2)), x0, (float)C, eps, rstd, shift);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const float *gm = params + 2 * C + 32 * t + 8 * (lv >> 4), *bt = gm + C;
                bf16x8 o;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    o[e] = (bf16_t)fmaf(fmaf(to_f32(v[t][e]), rstd, shift), gm[e], bt[e]);
                }
                cs[row_slot(16 * wave + (lv & 15), 4 * t + (lv >> 4))] = as_uint4(o);
            }
        }
        __syncthreads();
        {
            f32x16 acc[2];
            acc[0] = acc[1] = biases(4);
#pragma unroll
            for (int ks = 0; ks < CK; ++ks) {
#pragma unroll
                for (int pb = 0; pb < 2; ++pb) {
                    acc[pb] = mfma(wof[ks], as_bf16x8(cs[row_slot(32 * pb + (lv & 31), 2 * ks + (lv >> 5))]), acc[pb]);
                }
            }
#pragma unroll
            for (int pb = 0; pb < 2; ++pb) {
                bf16x8 rounded[2] = {pack8(acc[pb], 0), pack8(acc[pb], 8)};
                asm volatile("" : "+v"(rounded[0]), "+v"(rounded[1])); // else each value is rounded by itself
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    bf16x4 ov;
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        // bf16(out) * sigmoid(bf16(gate)), rounded to bf16: the reference's rounding points
                        const float o = to_f32(rounded[a >> 1][4 * (a & 1) + c]);
                        ov[c] = (bf16_t)(o * sigmoid_fast(to_f32(gate[pb][a >> 1][4 * (a & 1) + c])));
                    }
                    *(reinterpret_cast<bf16x4 *>(res + row_slot(32 * pb + (lv & 31), 4 * wave + a)) + (lv >> 5)) = ov;
                }
            }
        }
        __syncthreads();
        {
            char *to = row_of_x(row.at, lv);
            const uint4 raw_row[4] = {row.r0, row.r1, row.r2, row.r3};
            uint4 sum[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const bf16x8 d = as_bf16x8(res[row_slot(16 * wave + (lv >> 2), 4 * t + (lv & 3))]), z = as_bf16x8(raw_row[t]);
                bf16x8 o;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    o[e] = (bf16_t)(to_f32(z[e]) + to_f32(d[e]));
                }
                sum[t] = as_uint4(o);
            }
            if (row.there) {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    *reinterpret_cast<uint4 *>(to + 64 * t) = sum[t];
                }
            }
        }
        row = next_row;
    }
}

// runs of equally many steps for at most `cap` workgroups, the last one shorter
struct Split {
    unsigned groups;
    int per_group;
};
Split split_steps(int64_t n, int64_t np, int64_t cap)
{
    const int64_t steps = (n * np + STEP - 1) / STEP;
    const int64_t per = (steps + cap - 1) / cap;
    return Split{(unsigned)((steps + per - 1) / per), (int)per};
}
} // namespace

namespace kutacc_launch {

bool triangle_ends_support(const kutacc_hip_triangle_multiplication_args_t &a)
{
    // 16-byte loads of the activation's rows and of the weights; positions and sixteen planes' bytes (2^31 at
    // 8192 residues) in 32 bits
    return a.c_z == C && a.c_i == C && a.n_res <= 8192 && kutacc_hip_aligned16(a.pair_act) && kutacc_hip_aligned16(a.left_proj_w) &&
           kutacc_hip_aligned16(a.left_gate_w) && kutacc_hip_aligned16(a.right_proj_w) && kutacc_hip_aligned16(a.right_gate_w) &&
           kutacc_hip_aligned16(a.output_w) && kutacc_hip_aligned16(a.gating_w);
}

int triangle_front(const kutacc_hip_triangle_multiplication_args_t &a, void *left, void *right, int64_t rows, int64_t np, int64_t plane, hipStream_t stream)
{
    static size_t configured[KUTACC_DEVICE_SLOTS] = {};
    if (const hipError_t e = kutacc_opt_in_lds(reinterpret_cast<const void *>(&triangle_front_kernel), FRONT_LDS, configured)) {
        return kutacc_hip_status(e);
    }
    kutacc_prof::KernelTimer t("triangle_front_kernel", 8.0 * (double)(a.n_res * a.n_res) * C * C, stream);
    const Split s = split_steps(rows, np, kutacc_cu_count());
    const Side l = {(const bf16_t *)a.left_proj_w, (const bf16_t *)a.left_gate_w, a.left_proj_b, a.left_gate_b, (bf16_t *)left};
    const Side r = {(const bf16_t *)a.right_proj_w, (const bf16_t *)a.right_gate_w, a.right_proj_b, a.right_gate_b, (bf16_t *)right};
    triangle_front_kernel<<<dim3(s.groups), 64 * FRONT_WAVES, FRONT_LDS, stream>>>((const bf16_t *)a.pair_act, a.ln_in_gamma, a.ln_in_beta, a.ln_eps, l,
                                                                                  r, (const bf16_t *)a.pair_mask, plane, (int)a.n_res, (int)rows,
                                                                                  (int)np, s.per_group);
    return kutacc_hip_status(hipGetLastError());
}

int triangle_back(const kutacc_hip_triangle_multiplication_args_t &a, const void *centre, int64_t np, int64_t plane, hipStream_t stream)
{
    static size_t configured[KUTACC_DEVICE_SLOTS] = {};
    if (const hipError_t e = kutacc_opt_in_lds(reinterpret_cast<const void *>(&triangle_back_kernel), BACK_LDS, configured)) {
        return kutacc_hip_status(e);
    }
    kutacc_prof::KernelTimer t("triangle_back_kernel", 4.0 * (double)(a.n_res * a.n_res) * C * C, stream);
    // The workgroups that take a step more come first, one a CU: 384 residues give a CU nine steps, five and four, where equal runs of five gave
    // most ten (whole block, two activations in turn, 94.7 -> 92.3 us; 200 residues 41.6 -> 38.7).
    const int64_t steps = (a.n_res * np + STEP - 1) / STEP, groups = std::min(steps, 2 * (int64_t)kutacc_cu_count());
    triangle_back_kernel<<<dim3((unsigned)groups), 256, BACK_LDS, stream>>>(
        (const bf16_t *)centre, plane, a.ln_center_gamma, a.ln_center_beta, (const bf16_t *)a.output_w, a.output_b, (const bf16_t *)a.gating_w,
        a.gating_b, (bf16_t *)a.pair_act, a.ln_in_gamma, a.ln_in_beta, a.ln_eps, (int)a.n_res, (int)np, (int)(steps / groups), (int)(steps % groups));
    return kutacc_hip_status(hipGetLastError());
}

} // namespace kutacc_launch
