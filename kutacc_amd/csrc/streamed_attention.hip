// Gated attention of long batch rows for gfx950, bf16 storage, head size 32, 128 or 256 channels: the rows whose keys and
// values do not fit the LDS twice beside a head's weights (persistent_pair_kernel), in batches that fill the chip.
//
// Four kernels, of which a call runs three, with K, V, Q, the gate and the gated average in memory between them:
//
//   qkvg_projection_kernel    reads the input rows once, forms all four projections and writes them as the MFMA fragments
//       the attention loads -- 1 KB per store instruction, no layout change anywhere after it.
//   streamed_attention_kernel softmax(q.k^T + mask + pair bias).v * gate.  A wave owns the same 32 queries of several batch rows,
//       which share the pair bias (fp32 tiles in accumulator order, the C operand of every row's logits MFMAs, as in
//       persistent_pair_kernel); a workgroup of four waves walks all keys of the rows, their K and V staged
//       through a ring of key tiles in the LDS.
//   streamed_plain_kernel     the same without a pair bias, where a wave owns two blocks of queries of one row.
//   output_projection_kernel  multiplies the gated average, fragments as well, and adds the result to the activation.
//
// Against fused_head_kernel (one workgroup per row and head, K and V of the whole row in the LDS, projections in front):
// the pair bias costs no MFMAs and half the bytes, waves of every length work alike, the projections
// run at the rate of the memory instead of behind one barrier per workgroup, and a row's length decides nothing.  The price
// is the four projections and the average through memory, 10 bytes per channel and position.
//
// The order of positions, keys and head dims inside a fragment is that of the fused kernels (fused_attention.hip): lane r
// of a block of 32 positions stands for position pi(r), Q and K share their order of head dims, V and the probabilities
// their order of keys, so that accumulators are packed into operands as they are.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <climits>
#include <cstring>
#include <type_traits>

#include "attention_util.h"
#include "launch_internal.h"
#include "mfma_tiles.h"
#include "profiler.h"

namespace {
using namespace kutacc_dev;

constexpr int HEAD = 32;
constexpr uint32_t MIXED_WORDS = 1; // no word a row shares: a denormal mask bias
constexpr int BLOCK_SLOTS = 128; // 16-byte slots of a fragment pair: 32 positions x 32 head dims

struct StreamedParams {
    const bf16_t *x; // un-normalised
    int64_t x_ld, x_sb;
    const float *ln_gamma, *ln_beta;
    float ln_eps;
    const bf16_t *wq, *wk, *wv, *wg;
    const float *bg;
    const bf16_t *bias;
    int64_t bias_sb, bias_sk;
    int bias_is_mask;
    float qmul; // log2(e) / sqrt(head size)
    // [batch row][head][block of 32 positions][2 k-steps][64 lanes]; the gated average takes the place of the queries it was formed from
    uint4 *q, *g, *k, *v;
    // [batch row][block][32]: mask bias of key pi(i) in log2 units as two bf16 (mask_word).  Their 2^-17 moves no probability: the bias
    // is formed from a bf16 mask, so it is 0, or at least 3.9e6 in size and 2^-8 of that from any other: two keys' masks differ by
    // thousands or by nothing.  The fused kernels keep the bias in fp32; blocks of up to 1024 keys that run here instead get the same
    // probabilities.  (A third part was 7 % slower at 2048 residues, a tenth of them masked.)
    uint32_t *words;
    // [batch row][block]: 0, no key of the block has a mask; the word that all its keys have (those of the row, the tail is at -inf);
    // MIXED_WORDS otherwise
    uint32_t *flags;
    const f32x4 *tiles;   // pair bias: [head][query block][NT][4][64 lanes] (pair_bias_tiles_kernel)
    int B, S, H, NB, NT; // batch rows, positions, heads, blocks, key tiles of `tiles` per query block
    int query_groups, set_groups, groups, group_rows, plain_waves; // the attention's workgroups
};

// ---- the projections ----
//
// Bound by HBM: per position 2 C bytes in and 8 C out.  Eight waves, one workgroup per CU (and per 128 channels of outputs); a
// wave owns one head's two matrices -- Q and gate, or K and V -- whose 32 x C blocks stay in its registers, and stages
// eight of the 64 positions of a step into the shared stage, requested a step ahead and normalised on the way (a row's pieces lie
// in neighbouring lanes), so that no pass writes and reads a normalised copy.
template <int C>
constexpr size_t projection_lds() { return (size_t)2 * 64 * (C / 8) * 16 + 12 * C; }

template <int C>
__global__ __launch_bounds__(512, 1) void qkvg_projection_kernel(const StreamedParams p, int steps_per_group)
{
    constexpr int CK = C / 16, SLOTS = C / 8, LOADS = 8 * SLOTS / 64, ROWS = 64 / SLOTS; // rows per load instruction
    constexpr int AHEAD = 2; // fragments of the stage on their way to the products
    extern __shared__ uint4 lds[]; // two stages of [64 positions][SLOTS], gamma, beta, gating bias
    float *gamma = reinterpret_cast<float *>(lds + 2 * 64 * SLOTS), *beta = gamma + C, *gating = beta + C;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, g = lane >> 5;
    // Workgroup ids are dealt round robin over the 8 XCDs: with 256 channels the two workgroups that read the same rows, eight ids apart,
    // share an L2 whatever the number of runs (508 x 259, 127 runs: 279.5 -> 276 us).
    constexpr int HALVES = C / 128;
    const int id = (int)blockIdx.x, run = HALVES == 1 ? id : (id & 7) + 8 * (id >> 4), half_of_heads = HALVES == 1 ? 0 : (id >> 3) & 1;
    const int h = half_of_heads * 4 + (wave & 3);
    const bool forms_kv = wave >= 4;

    const int blocks = p.B * p.NB, total_steps = (blocks + 1) / 2;
    const int first = run * steps_per_group;
    const int stop = min(first + steps_per_group, total_steps);
    if (first >= stop) {
        return;
    }
    // The stage's rows lie in order of position; slot index XOR-ed so that the eight positions eight consecutive lanes of a
    // fragment read stand for (pi: 0-3 and 16-19, 4-7 and 20-23, ...) lie in different bank groups.
    auto slot = [](int pos, int chunk) { return pos * SLOTS + (chunk ^ ((pos & 3) | ((pos >> 2) & 4))); };

    // block of 32 positions this wave stages its eight of, as (batch row, block of the row)
    int load_b = (2 * first + (wave >> 2)) / p.NB, load_j = (2 * first + (wave >> 2)) % p.NB;
    auto advance = [&](int &b, int &j) {
        j += 2;
        while (j >= p.NB) {
            j -= p.NB, ++b;
        }
    };
    struct Rows {
        uint4 r[LOADS];
    };
    auto load = [&] {
        Rows t;
        const char *base = reinterpret_cast<const char *>(p.x + (int64_t)min(load_b, p.B - 1) * p.x_sb);
#pragma unroll
        for (int u = 0; u < LOADS; ++u) {
            const int pos = min(32 * load_j + 8 * (wave & 3) + ROWS * u + lane / SLOTS, p.S - 1);
            __builtin_memcpy(&t.r[u], base + ((int64_t)pos * p.x_ld * 2 + 16 * (lane % SLOTS)), 16); // on any address
        }
        advance(load_b, load_j);
        return t;
    };
    auto park = [&](int s, const Rows &t, int lane) {
        float gm[8], bt[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            gm[e] = gamma[lane % SLOTS * 8 + e], bt[e] = beta[lane % SLOTS * 8 + e];
        }
#pragma unroll
        for (int u = 0; u < LOADS; ++u) {
            const bf16x8 in = as_bf16x8(t.r[u]);
            float v[8], rstd, shift;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                v[e] = to_f32(in[e]);
            }
            group_stats<SLOTS>(v, __shfl(v[0], lane & ~(SLOTS - 1), 64), (float)C, p.ln_eps, rstd, shift);
            bf16x8 out;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                out[e] = (bf16_t)fmaf(fmaf(v[e], rstd, shift), gm[e], bt[e]);
            }
            lds[s * 64 * SLOTS + slot(8 * wave + ROWS * u + lane / SLOTS, lane % SLOTS)] = as_uint4(out);
        }
    };
    // The masks of a step's two blocks are the business of waves 0 and 3, one each.  Whatever a step uses is asked for a step ahead and in
    // front of the next rows: loads return in order, and a later one waited for would make the rows' wait a whole round trip.
    const bool forms_masks = half_of_heads == 0 && (wave == 0 || wave == 3);
    int mask_b = (2 * first + (wave == 3)) / p.NB, mask_j = (2 * first + (wave == 3)) % p.NB;
    auto load_mask = [&] {
        const int key = min(32 * mask_j + pi_row(r), p.S - 1);
        const bf16_t m = p.bias[(int64_t)min(mask_b, p.B - 1) * p.bias_sb + (int64_t)key * p.bias_sk];
        advance(mask_b, mask_j);
        return m;
    };
    bf16_t mask = (bf16_t)0.f;
    if (forms_masks) {
        mask = load_mask();
    }
    Rows rows = load();
    for (int c = tid; c < C; c += 512) {
        gamma[c] = p.ln_gamma[c], beta[c] = p.ln_beta[c], gating[c] = p.bg[c];
    }
    bf16x8 w0[CK], w1[CK]; // Q and gate, or K and V
    {
        const bf16_t *m0 = forms_kv ? p.wk : p.wq, *m1 = forms_kv ? p.wv : p.wg;
        load_half_lines<CK>(w0, m0 + h * HEAD * C, C, lane);
        load_half_lines<CK>(w1, m1 + h * HEAD * C, C, lane);
        half_lines_to_fragments<CK>(w0, lds + 128 * wave, lane); // on the stages, which are empty still
        half_lines_to_fragments<CK>(w1, lds + 128 * wave, lane);
    }
    __syncthreads();
    park(0, rows, lane);
    bf16_t next_mask = (bf16_t)0.f;
    if (first + 1 < stop) {
        next_mask = forms_masks ? load_mask() : next_mask;
        rows = load();
    }
    __syncthreads();
    // The weights are waited for here: waits that the compiler leaves to their first uses stand in the loop, where they are waits for
    // every load and store on its way (with the stores of a step counted below, 2048 residues 1289 -> 1165 us, 5.4 GB
    // at 4.6 TB/s; 1024 sequences x 384 residues of 256 channels 261 -> 240 us).
#pragma unroll
    for (int ks = 0; ks < CK; ++ks) {
        asm volatile("" ::"v"(w0[ks]), "v"(w1[ks]));
    }

    int b = (2 * first) / p.NB, j = (2 * first) % p.NB; // the block being multiplied
    auto steps = [&](auto kv) {
        for (int step = first; step < stop; ++step) {
            const int s = (step - first) & 1;
            // With 256 channels the lane index is opaque to the optimiser, so that addresses are formed per step: kept across the loop
            // beside the weights they would be spilled, and a reload waits for every load on its way.
            int lv = tid & 63;
            if constexpr (C == 256) {
                asm volatile("" : "+v"(lv));
            }
            const int r = lv & 31, g = lv >> 5, lane = lv;
            bf16_t after_next = (bf16_t)0.f;
            auto stage_next = [&] {
                if (step + 1 < stop) {
                    park(s ^ 1, rows, lane);
                    after_next = forms_masks ? load_mask() : after_next;
                    rows = load();
                }
            };
            // The two waves of a SIMD start a step together: one normalises while the other multiplies.
            if constexpr (!decltype(kv)::value) {
                stage_next();
            }
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                // Behind an odd number of blocks the last one again: every step has the same stores, so that the wait for the next rows lets
                // them be on their way.
                const uint4 *stage = lds + (s * 64 + (2 * step + half < blocks ? 32 * half : 0)) * SLOTS;
                // Fragment ks lies in slot(pi_row(r), 2 ks + g): four lane offsets, the rest of the slot is the same for all lanes.  With an
                // offset for each of 16 fragments and one fragment on its way, as the compiler had it, a pair of products waited for its operand:
                // 508 sequences x 259 residues 274.5 -> 269.4 us (projections 94.6 -> 90.0), 1024 x 384 843 -> 833.5 (236 -> 223); four, six and
                // eight on their way 90.3, 90.5 and 91.5 us.
                const uint4 *lane_slot[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    lane_slot[i] = stage + slot(pi_row(r), 2 * i + g);
                }
                bf16x8 xf[CK];
                auto fragment = [&](int ks) { xf[ks] = as_bf16x8(lane_slot[ks & 3][8 * (ks >> 2)]); };
#pragma unroll
                for (int ks = 0; ks < AHEAD; ++ks) {
                    fragment(ks);
                }
                f32x16 a0 = zero16(), a1 = zero16();
                const int64_t at = (((int64_t)b * p.H + h) * p.NB + j) * BLOCK_SLOTS + lane;
                if constexpr (decltype(kv)::value) {
#pragma unroll
                    for (int ks = 0; ks < CK; ++ks) {
                        a0 = mfma(w0[ks], xf[ks], a0);
                        a1 = mfma(xf[ks], w1[ks], a1); // V: rows = keys, columns = head dims
                        if (ks + AHEAD < CK) {
                            fragment(ks + AHEAD);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    p.k[at] = as_uint4(pack8(a0, 0)), p.k[at + 64] = as_uint4(pack8(a0, 8));
                    p.v[at] = as_uint4(pack8(a1, 0)), p.v[at + 64] = as_uint4(pack8(a1, 8));
                } else {
#pragma unroll
                    for (int ks = 0; ks < CK; ++ks) {
                        a0 = mfma(w0[ks], xf[ks], a0);
                        a1 = mfma(w1[ks], xf[ks], a1);
                        if (ks + AHEAD < CK) {
                            fragment(ks + AHEAD);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    const float *bg = gating + h * HEAD + 4 * g;
#pragma unroll
                    for (int a = 0; a < 4; ++a) {
                        const f32x4 bv = *reinterpret_cast<const f32x4 *>(bg + 8 * a);
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            a0[4 * a + c] *= p.qmul;
                            a1[4 * a + c] += bv[c]; // the gate is rounded in front of its sigmoid, as where the reference stores it
                        }
                    }
                    p.q[at] = as_uint4(pack8(a0, 0)), p.q[at + 64] = as_uint4(pack8(a0, 8));
                    p.g[at] = as_uint4(pack8(a1, 0)), p.g[at + 64] = as_uint4(pack8(a1, 8));
                }
                if (!decltype(kv)::value && forms_masks && wave == 3 * half && 2 * step + half < blocks) {
                    const int key = 32 * j + pi_row(r);
                    float mv = -INFINITY;
                    if (key < p.S) {
                        mv = to_f32(mask);
                        if (p.bias_is_mask) {
                            mv = to_f32((bf16_t)fmaf(mv, 1e9f, -1e9f));
                        }
                        mv = finite_bias(mv * LOG2E);
                    }
                    const uint32_t word = mask_word(mv), first_word = __builtin_amdgcn_readfirstlane(word); // lane 0: key 32 j
                    if (lane < 32) {
                        p.words[((int64_t)b * p.NB + j) * 32 + lane] = word;
                    }
                    const bool any = __ballot(mv != 0.f) != 0, mixed = __ballot(key < p.S && word != first_word) != 0 || first_word == 0;
                    if (lane == 0) {
                        p.flags[(int64_t)b * p.NB + j] = !any ? 0u : (mixed ? MIXED_WORDS : first_word);
                    }
                }
                if (2 * step + half + 1 < blocks && ++j == p.NB) {
                    j = 0, ++b;
                }
            }
            if constexpr (decltype(kv)::value) {
                stage_next();
            }
            mask = next_mask, next_mask = after_next;
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); // the next stage is complete, this one no longer read
        }
    };
    if (forms_kv) { // two loops, so that the waits of each are those of its own loads and stores
        steps(std::true_type{});
    } else {
        steps(std::false_type{});
    }
}

// ---- the attention ----
constexpr int WAVES = 4;                  // query blocks per workgroup
constexpr int PLAIN_BLOCKS = 2;           // query blocks of a wave without a pair bias
constexpr int RING = 3;                   // groups of tiles in the LDS
constexpr int TOGETHER = 8, MEMBERS = 64; // query groups and workgroups of a placement group, at most

// What a wave attends with one set of 32 queries' positions: ROWS batch rows, which share a tile of the pair bias.  A tile's keys and
// values are ROWS x 4 KB; tiles come in groups of which every wave brings four pieces of 1 KB.
template <int ROWS>
struct Walk {
    static constexpr int TILES_PER_GROUP = 4 / ROWS, TILE_SLOTS = ROWS * 2 * BLOCK_SLOTS, TILE_BYTES = TILE_SLOTS * 16;
    static constexpr int GROUP_BYTES = TILES_PER_GROUP * TILE_BYTES; // 4 KB a wave
    static constexpr size_t LDS = (size_t)RING * GROUP_BYTES;
};

// The gated average of 32 queries of one row in the place of their queries: o / l * sigmoid(gate).  Positions past the row's end are
// stored like the others: nobody reads them.  l lies within 1e-30 .. 1e30, or is of a repeated row: 1 .. 2^20.
__device__ __forceinline__ void store_average(uint4 *dst, uint4 gate0, uint4 gate1, const f32x16 &o, float l)
{
    const bf16x8 g0 = as_bf16x8(gate0), g1 = as_bf16x8(gate1);
    const float inv = reciprocal(l);
    float sigmoid[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        sigmoid[i] = to_f32(i < 8 ? g0[i & 7] : g1[i & 7]);
    }
    sigmoids_f32(sigmoid);
    f32x16 out;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        out[i] = o[i] * inv * sigmoid[i];
    }
    dst[0] = as_uint4(pack8(out, 0)), dst[64] = as_uint4(pack8(out, 8));
}

// Repeat of one row's 32 queries after an overflow or underflow of the unshifted exponentials (a sum outside 1e-30 .. 1e30): the
// true row maxima first, then the probabilities with them subtracted.  Not a hot path: one row, operands straight from memory, no
// barrier.  q: the queries, whose place the result takes.
template <bool HAS_NB>
__device__ __forceinline__ void attend_shifted(const uint4 *k, const uint4 *v, const uint32_t *words, const f32x4 *nbc, uint4 *q, const uint4 *gate,
                                               int NB, int lane)
{
    const bf16x8 q0 = as_bf16x8(q[lane]), q1 = as_bf16x8(q[64 + lane]);
    auto logits = [&](int t) {
        f32x16 x;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            f32x4 cv = {0.f, 0.f, 0.f, 0.f};
            if constexpr (HAS_NB) {
                cv = nbc[(t * 4 + a) * 64 + lane];
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                x[4 * a + c] = mask_word_value(words[32 * t + 8 * a + 4 * (lane >> 5) + c]) + cv[c];
            }
        }
        x = mfma(as_bf16x8(k[t * BLOCK_SLOTS + lane]), q0, x);
        return mfma(as_bf16x8(k[t * BLOCK_SLOTS + 64 + lane]), q1, x);
    };
    float mx = -INFINITY;
    for (int t = 0; t < NB; ++t) {
        const f32x16 x = logits(t);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            mx = fmaxf(mx, x[i]);
        }
    }
    mx = half_swap_max(mx); // finite: a fully masked row has -1e9*log2(e) everywhere
    f32x16 o = zero16();
    f32x4 sums = {0.f, 0.f, 0.f, 0.f};
    const bf16x8 ones_rows = rowsum_selector(lane);
    for (int t = 0; t < NB; ++t) {
        f32x16 x = logits(t);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            x[i] = __builtin_amdgcn_exp2f(x[i] - mx);
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const bf16x8 pv = pack8(x, 8 * s);
            o = mfma(as_bf16x8(v[t * BLOCK_SLOTS + 64 * s + lane]), pv, o);
            sums = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones_rows, pv, sums, 0, 0, 0);
        }
    }
    store_average(q + lane, gate[lane], gate[64 + lane], o, rowsum_fetch(sums, lane));
}

// Bound by the issue of the softmax (16 exponentials and 8 packs per lane, row and tile: 201 of the 268 clocks that a tile of 32 x 32
// logits takes a SIMD with no load in the loop) and next to it by what the loop loads.  Four rows a wave halve the loads of
// the pair bias, 4 KB a tile, and leave 256 registers to the two waves of a SIMD, against two rows on three waves of 168: 2048
// residues without padding 6.56 -> 5.84 ms, 1024 residues 1.00 -> 0.79 ms.
//
// Keys and values come straight into the LDS (global_load_lds_dwordx4), a group of tiles at a time, of which every wave brings four
// pieces of 1 KB: a ring of three groups, one barrier per group.  At the barrier in front of group G, group G + 1 has landed and group
// G - 1 has been left by every wave; its place takes group G + 2.
template <int ROWS>
__global__ __launch_bounds__(512) void streamed_attention_kernel(const StreamedParams p)
{
    using W = Walk<ROWS>;
    typedef __attribute__((address_space(3))) void *lds_ptr;
    extern __shared__ uint4 lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int NB = p.NB;

    // Workgroup ids are dealt round robin over the 8 XCDs; an XCD works on one group at a time: group_rows sets of rows x
    // up to eight query groups of one head, which sweep the keys together, so that the group's K and V and pair bias come
    // from memory once and from the XCD's L2 after that.
    const int members = p.group_rows * min(p.query_groups, TOGETHER);
    const int local = (int)(blockIdx.x >> 3);
    const int group = (int)(blockIdx.x & 7) + 8 * (local / members), member = local % members;
    if (group >= p.groups) {
        return;
    }
    const int set_group = group % p.set_groups, rest = group / p.set_groups;
    const int h = rest % p.H, query_part = rest / p.H;
    const int set = set_group * p.group_rows + member % p.group_rows, qg = query_part * TOGETHER + member / p.group_rows;
    if (ROWS * set >= p.B || qg >= p.query_groups) {
        return;
    }
    // The pieces u = 4 wave + i of a group of tiles: tile u / (4 ROWS), piece u % (4 ROWS) = [row][K, V][k-step].  Written out: as a builtin
    // the compiler takes every LDS read behind it for a reader of its data and waits for all loads in flight.
    const uint32_t ring = (uint32_t)(uintptr_t)(lds_ptr)lds, lane_bytes = 16u * (uint32_t)lane;
    const int own_row = ROWS == 4 ? wave : wave & 1; // all four pieces of a wave are of one row and tile
    const int64_t own = ((int64_t)min(ROWS * set + own_row, p.B - 1) * p.H + h) * NB;
    auto request = [&](int first_tile, int place) { // tiles first_tile .. into group `place` of the ring
        const int64_t from = (own + min(first_tile + (ROWS == 4 ? 0 : wave >> 1), NB - 1)) * BLOCK_SLOTS;
        const uint32_t to = ring + (uint32_t)place * W::GROUP_BYTES + (uint32_t)wave * 4096u;
        load_to_lds(to, p.k + from, lane_bytes);
        load_to_lds(to + 1024u, p.k + from + 64, lane_bytes);
        load_to_lds(to + 2048u, p.v + from, lane_bytes);
        load_to_lds(to + 3072u, p.v + from + 64, lane_bytes);
    };
    request(0, 0);
    request(W::TILES_PER_GROUP, 1);
    // Rows first .. first + N - 1 of the set, the queries of block j.
    auto attend = [&](int j, int first, auto rows_attended) __attribute__((always_inline)) {
        constexpr int N = decltype(rows_attended)::value;
        int b[N]; // past the last row: that one again, not stored
        int64_t row[N]; // first fragment block
#pragma unroll
        for (int i = 0; i < N; ++i) {
            b[i] = min(ROWS * set + first + i, p.B - 1);
            row[i] = ((int64_t)b[i] * p.H + h) * NB;
        }

        int fill = 2, fill_tile = 2 * W::TILES_PER_GROUP; // the next group to ask for: its place in the ring, its first tile
        // Behind the last keys each wave asks for the gates of its own queries, two rows at a time, four pieces as well, so that they wait
        // in the ring when the loop ends (asked for there, they were a round trip at the end of every workgroup).
        int gates = 0, gate_place = 0; // rows asked for; the place of the first two
        auto refill = [&] {
            if (fill_tile < NB) {
                request(fill_tile, fill);
            } else if (gates < N && j < NB) {
                gate_place = gates == 0 ? fill : gate_place;
                const uint32_t to = ring + (uint32_t)fill * W::GROUP_BYTES + (uint32_t)wave * 4096u;
                const uint4 *first = p.g + ((gates == 0 ? row[0] : row[N - 2]) + j) * BLOCK_SLOTS;
                const uint4 *second = p.g + ((gates == 0 ? row[1] : row[N - 1]) + j) * BLOCK_SLOTS;
                load_to_lds(to, first, lane_bytes);
                load_to_lds(to + 1024u, first + 64, lane_bytes);
                load_to_lds(to + 2048u, second, lane_bytes);
                load_to_lds(to + 3072u, second + 64, lane_bytes);
                gates += 2;
            }
            fill = fill == RING - 1 ? 0 : fill + 1;
            fill_tile += W::TILES_PER_GROUP;
        };
        if (j >= NB) { // a wave without queries brings its share of the keys
            for (int t = 0; t < NB; t += W::TILES_PER_GROUP) {
                asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
                refill();
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            return;
        }

        bf16x8 q[N][2];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const uint4 *src = p.q + (row[i] + j) * BLOCK_SLOTS;
            q[i][0] = as_bf16x8(src[lane]), q[i][1] = as_bf16x8(src[64 + lane]);
        }
        const f32x4 *nbc = p.tiles + ((int64_t)h * NB + j) * p.NT * 256;
        auto load_nb = [&](int t) {
            f32x16 c;
            const char *tile = reinterpret_cast<const char *>(nbc + min(t, NB - 1) * 256); // uniform; the lane's part in 32 bits
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const f32x4 v = *reinterpret_cast<const f32x4 *>(tile + (lane_bytes + 1024u * a));
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    c[4 * a + e] = v[e];
                }
            }
            return c;
        };
        f32x16 C0 = load_nb(0), C1 = load_nb(1);

        // first key tile in which a row has a mask (the ragged tail of a row counts: its keys are at -inf)
        int masked_from = NB;
        for (int t0 = 0; t0 < NB; t0 += 64) {
            uint32_t f = 0;
#pragma unroll
            for (int i = 0; i < N; ++i) {
                f |= t0 + lane < NB ? p.flags[(int64_t)b[i] * NB + t0 + lane] : 0u;
            }
            const unsigned long long any = __ballot(f != 0u);
            if (any != 0) {
                masked_from = t0 + __builtin_ctzll(any);
                break;
            }
        }

        // A row whose keys all have one mask (a padded residue's: -1e9 everywhere) would end with every exponential at zero.  Its logits
        // are taken against that mask from the start: x = (q.k + bias + mask) - mask, each sum rounded, so that the mask absorbs what
        // it absorbs in the reference.  shift: the word of the -mask, 0 for other rows.  Such rows used to be attended twice more, by
        // attend_shifted: 2048 residues, 4 % of them padding, 1.4 ms of 8.0.  The masked loop adds the shift of every row, zero or not (2048
        // residues without the first one 9.46 ms, whole 7.83; two rows a wave with one product 10.9 and 8.78).
        uint32_t shift[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            shift[i] = 0;
            if (masked_from == 0) {
                const uint32_t *flags = p.flags + (int64_t)b[i] * NB;
                const uint32_t f = flags[0];
                bool differs = f == MIXED_WORDS || f == 0;
                for (int t0 = 0; t0 < NB && !differs; t0 += 64) {
                    differs = __any(flags[min(t0 + lane, NB - 1)] != f);
                }
                shift[i] = __builtin_amdgcn_readfirstlane(differs ? 0u : f ^ 0x80008000u);
            }
        }

        // The mask of a row as a rank-one MFMA: A holds (hi, lo) of the key of accumulator row i in k-slots 0 and 1, B ones there,
        // all else zero, also in the lanes of the upper half, so that an infinite mask value never meets a zero.
        const uint32_t lower = lane < 32 ? 0xffffffffu : 0u;
        auto mask_word_of = [&](int i, int t) { return p.words[((int64_t)b[i] * NB + min(t, NB - 1)) * 32 + (lane & 31)] & lower; };
        auto add_mask = [&](f32x16 x, uint32_t w) {
            const bf16x8 ones = as_bf16x8(make_uint4(0x3f803f80u & lower, 0u, 0u, 0u));
            return mfma(as_bf16x8(make_uint4(w, 0u, 0u, 0u)), ones, x);
        };

        asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory"); // groups 0 and 1 have landed, every wave's part of them
        refill();
        int left = W::TILES_PER_GROUP; // tiles of the current group still to come, this one included
        const uint4 *cur = lds, *const end = lds + RING * W::TILES_PER_GROUP * W::TILE_SLOTS, *next = lds + W::TILE_SLOTS; // tiles t and t + 1
        auto keys = [&](const uint4 *tile, int i) { return tile + (first + i) * 2 * BLOCK_SLOTS + lane; };
        auto values = [&](const uint4 *tile, int i) { return tile + (first + i) * 2 * BLOCK_SLOTS + BLOCK_SLOTS + lane; };
        uint4 k0 = keys(cur, 0)[0], k1 = keys(cur, 0)[64], v0, v1;
        f32x16 x[2]; // logits: of row i in x[i & 1]
        x[0] = mfma(as_bf16x8(k0), q[0][0], C0);
        x[0] = mfma(as_bf16x8(k1), q[0][1], x[0]);
        k0 = keys(cur, 1)[0], k1 = keys(cur, 1)[64];
        v0 = values(cur, 0)[0], v1 = values(cur, 0)[64];
        f32x16 o[N];
        f32x4 sums[N]; // the row sums on the matrix pipe: see rowsum_selector
        uint32_t m[N]; // the mask words of a row's next logits
#pragma unroll
        for (int i = 0; i < N; ++i) {
            o[i] = zero16(), sums[i] = f32x4{0.f, 0.f, 0.f, 0.f}, m[i] = 0;
        }
        const bf16x8 ones_rows = rowsum_selector(lane);

        auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
        // Tile t with seed C: finishes row i = 0 .. N - 1, each time softmax and P.V of the finished logits, the logits of the next row (of
        // the first one and tile t + 1, from seed Cn, behind the last), and the fragments of the row behind that.  The fences deal the
        // exponentials between the MFMAs.  The empty asm keeps C live past the MFMA that reads it, so that the logits get registers of their own.
        auto tile = [&](int t, f32x16 &C, f32x16 &Cn, auto masked) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < N; ++i) {
                constexpr int LAST = N - 1;
                const int n = i == LAST ? 0 : i + 1, nn = (i + 2) % N; // the next row, the one behind it
                f32x16 &xc = x[i & 1], &xn = x[n & 1];
                auto exp4 = [&](int base) {
#pragma unroll
                    for (int e = base; e < base + 4; ++e) {
                        xc[e] = __builtin_amdgcn_exp2f(xc[e]);
                    }
                };
                exp4(0);
                if (i == LAST) {
                    xn = mfma(as_bf16x8(k0), q[n][0], Cn);
                    asm volatile("" ::"v"(Cn));
                } else {
                    xn = mfma(as_bf16x8(k0), q[n][0], C);
                    asm volatile("" ::"v"(C));
                }
                fence();
                exp4(4);
                const bf16x8 p0 = pack8(xc, 0);
                xn = mfma(as_bf16x8(k1), q[n][1], xn);
                if constexpr (decltype(masked)::value) {
                    xn = add_mask(add_mask(xn, m[n]), shift[n] & lower);
                }
                const uint4 *kf = keys(i + 2 < N ? cur : next, nn);
                k0 = kf[0], k1 = kf[64];
                fence();
                exp4(8);
                o[i] = mfma(as_bf16x8(v0), p0, o[i]);
                fence();
                exp4(12);
                const bf16x8 p1 = pack8(xc, 8);
                sums[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones_rows, p0, sums[i], 0, 0, 0);
                o[i] = mfma(as_bf16x8(v1), p1, o[i]);
                sums[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones_rows, p1, sums[i], 0, 0, 0);
                fence();
                const uint4 *vf = values(i == LAST ? next : cur, n);
                v0 = vf[0], v1 = vf[64];
                fence(); // the loads stay behind the last reader of the registers they fill
                if (i == LAST - 1) {
                    C = load_nb(t + 2);
                }
                if constexpr (decltype(masked)::value) {
                    m[n] = mask_word_of(n, t + (i == LAST ? 2 : 1));
                }
                fence();
            }
            cur = next;
            next += W::TILE_SLOTS;
            next = next == end ? lds : next;
            if (--left == 0) {
                // This wave's pieces of the group behind the next one have landed: it asked for them a group ago, and its
                // youngest loads are those of the group's tiles' bias, issued since.
                asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(4 * W::TILES_PER_GROUP) : "memory");
                refill();
                left = W::TILES_PER_GROUP;
            }
        };
        auto run = [&](int from, int to, auto masked) __attribute__((always_inline)) {
            int t = from;
            for (; t + 1 < to; t += 2) {
                tile(t, C0, C1, masked);
                tile(t + 1, C1, C0, masked);
            }
            if (t < to) {
                tile(t, C0, C1, masked);
                const f32x16 swap = C0;
                C0 = C1, C1 = swap;
            }
        };
        run(0, masked_from, std::false_type{});
        if (masked_from < NB) {
            x[0] = add_mask(add_mask(x[0], mask_word_of(0, masked_from)), shift[0] & lower);
#pragma unroll
            for (int i = 0; i < N; ++i) {
                m[i] = mask_word_of(i, masked_from + (i == 0 ? 1 : 0));
            }
            run(masked_from, NB, std::true_type{});
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the gates, and requests past the last tile before the LDS is given back
        uint32_t again = 0; // rows whose sums ran out of range
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const float l = rowsum_fetch(sums[i], lane);
            const bool stored = ROWS * set + first + i < p.B;
            if (__any(!(l > 1e-30f && l < 1e30f))) {
                again |= stored ? 1u << i : 0u;
            } else if (stored) {
                const int place = i < 2 ? gate_place : (gate_place == RING - 1 ? 0 : gate_place + 1);
                const uint4 *gate = lds + place * (W::GROUP_BYTES / 16) + wave * 256 + (i & 1) * 128 + lane;
                store_average(p.q + (row[i] + j) * BLOCK_SLOTS + lane, gate[0], gate[64], o[i], l);
            }
        }
        while (again != 0) {
            const int i = __builtin_ctz(again), bi = ROWS * set + first + i;
            again &= again - 1;
            const int64_t at = ((int64_t)bi * p.H + h) * NB;
            attend_shifted<true>(p.k + at * BLOCK_SLOTS, p.v + at * BLOCK_SLOTS, p.words + (int64_t)bi * NB * 32, nbc, p.q + (at + j) * BLOCK_SLOTS,
                                   p.g + (at + j) * BLOCK_SLOTS, NB, lane);
        }
    };
    // One or two query blocks behind the last whole workgroup: its waves share out the rows, two each, and are done in half the time; with four
    // rows a wave two or three of the four only brought keys.  508 sequences x 259 residues (nine blocks) 281 -> 276 us and padded
    // 296 -> 283, 300 x 420 301 -> 289, triangle attention of 1200 residues 2139 -> 2080.
    if constexpr (ROWS == 4) {
        const int left = NB % WAVES;
        if (qg == p.query_groups - 1 && (left == 1 || left == 2)) {
            attend(qg * WAVES + (wave >> 1), 2 * (wave & 1), std::integral_constant<int, 2>{});
            return;
        }
    }
    attend(qg * WAVES + wave, 0, std::integral_constant<int, ROWS>{});
}

// The same without a pair bias, where batch rows share nothing: a wave attends two blocks of 32 queries of one row, which share its
// keys, values and masks.  A workgroup walks the row's keys once for all its blocks; each of its waves brings one tile (4 KB) of a group.
// Bound by issue and power: 1024 sequences x 384 residues x 8 heads 520 us, 295 clocks a tile of 32 x 32 logits and SIMD, at the
// 1.8 GHz that the chip holds under it (some 10 us more with the rounded quotients behind the loop).  Two rows a wave, which share nothing, 541 us; four blocks a wave on two waves a SIMD 526; two
// blocks on four waves of 128 registers 523.  3000 x 60 685 -> 605, 700 x 256 211 -> 192, 300 x 100 25.2 -> 26.2 us.
__global__ __launch_bounds__(768) void streamed_plain_kernel(const StreamedParams p)
{
    typedef __attribute__((address_space(3))) void *lds_ptr;
    extern __shared__ uint4 lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int NB = p.NB, W = p.plain_waves;
    constexpr int BLOCKS = PLAIN_BLOCKS, TILE = 2 * BLOCK_SLOTS; // slots of a tile in the LDS: K, V

    // Workgroup ids are dealt round robin over the 8 XCDs: a row and head's workgroups run side by side on one, whose L2 has its keys.
    const int local = (int)(blockIdx.x >> 3), part = local % p.query_groups;
    const int row_head = (local / p.query_groups) * 8 + (int)(blockIdx.x & 7);
    if (row_head >= p.groups) {
        return;
    }
    const int b = row_head / p.H;
    const int64_t row = (int64_t)row_head * NB; // first fragment block
    const int j = (part * W + wave) * BLOCKS;

    const uint32_t ring = (uint32_t)(uintptr_t)(lds_ptr)lds, lane_bytes = 16u * (uint32_t)lane;
    auto request = [&](uint32_t place, int first_tile) { // this wave's one of the tiles first_tile ..
        const int64_t from = (row + min(first_tile + wave, NB - 1)) * BLOCK_SLOTS;
        const uint32_t to = ring + (place * W + wave) * 4096u;
        load_to_lds(to, p.k + from, lane_bytes);
        load_to_lds(to + 1024u, p.k + from + 64, lane_bytes);
        load_to_lds(to + 2048u, p.v + from, lane_bytes);
        load_to_lds(to + 3072u, p.v + from + 64, lane_bytes);
    };
    request(0, 0);
    request(1, W);
    int fill = 2, fill_tile = 2 * W;
    int gate_place = -1; // of this wave's gates, which follow the last keys as in streamed_attention_kernel
    auto refill = [&] {
        if (fill_tile < NB) {
            request(fill, fill_tile);
        } else if (gate_place < 0 && j < NB) {
            gate_place = fill;
            const uint32_t to = ring + (uint32_t)(fill * W + wave) * 4096u;
            const uint4 *first = p.g + (row + j) * BLOCK_SLOTS, *second = p.g + (row + min(j + 1, NB - 1)) * BLOCK_SLOTS;
            load_to_lds(to, first, lane_bytes);
            load_to_lds(to + 1024u, first + 64, lane_bytes);
            load_to_lds(to + 2048u, second, lane_bytes);
            load_to_lds(to + 3072u, second + 64, lane_bytes);
        }
        fill = fill == RING - 1 ? 0 : fill + 1;
        fill_tile += W;
    };
    if (j >= NB) { // a wave without queries brings its share of the keys
        for (int t = 0; t < NB; t += W) {
            asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
            refill();
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        return;
    }

    bf16x8 q[BLOCKS][2]; // past the last block: that one again, not stored
#pragma unroll
    for (int i = 0; i < BLOCKS; ++i) {
        const uint4 *src = p.q + (row + min(j + i, NB - 1)) * BLOCK_SLOTS;
        q[i][0] = as_bf16x8(src[lane]), q[i][1] = as_bf16x8(src[64 + lane]);
    }

    const uint32_t *flags = p.flags + (int64_t)b * NB;
    int masked_from = NB; // first key tile that has a mask (the ragged tail counts: its keys are at -inf)
    for (int t0 = 0; t0 < NB; t0 += 64) {
        const unsigned long long any = __ballot(t0 + lane < NB && flags[min(t0 + lane, NB - 1)] != 0u);
        if (any != 0) {
            masked_from = t0 + __builtin_ctzll(any);
            break;
        }
    }
    uint32_t shift = 0; // one mask on all keys: see streamed_attention_kernel
    if (masked_from == 0) {
        const uint32_t f = flags[0];
        bool differs = f == MIXED_WORDS;
        for (int t0 = 0; t0 < NB && !differs; t0 += 64) {
            differs = __any(flags[min(t0 + lane, NB - 1)] != f);
        }
        shift = __builtin_amdgcn_readfirstlane(differs ? 0u : f ^ 0x80008000u);
    }
    const uint32_t lower = lane < 32 ? 0xffffffffu : 0u; // the mask as a rank-one MFMA
    auto mask_word_of = [&](int t) { return p.words[((int64_t)b * NB + min(t, NB - 1)) * 32 + (lane & 31)] & lower; };
    auto add_mask = [&](f32x16 x, uint32_t w) {
        const bf16x8 ones = as_bf16x8(make_uint4(0x3f803f80u & lower, 0u, 0u, 0u));
        return mfma(as_bf16x8(make_uint4(w, 0u, 0u, 0u)), ones, x);
    };

    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory"); // groups 0 and 1 have landed, every wave's part of them
#pragma unroll
    for (int i = 0; i < BLOCKS; ++i) { // waited for here, not at their first uses in the loop, where that is a wait for the next tiles
        asm volatile("" ::"v"(q[i][0]), "v"(q[i][1]));
    }
    refill();
    int left = W; // tiles of the current group still to come, this one included
    const uint4 *const end = lds + RING * W * TILE, *next = lds + TILE; // tile t + 1
    uint4 k0 = lds[lane], k1 = lds[64 + lane], v0 = lds[128 + lane], v1 = lds[192 + lane];
    f32x16 x[2]; // logits: of block i in x[i & 1]
    x[0] = mfma(as_bf16x8(k0), q[0][0], zero16());
    x[0] = mfma(as_bf16x8(k1), q[0][1], x[0]);
    f32x16 o[BLOCKS];
    f32x4 sums[BLOCKS];
#pragma unroll
    for (int i = 0; i < BLOCKS; ++i) {
        o[i] = zero16(), sums[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    uint32_t m = 0, mn = 0; // mask words of this tile and of the next
    const bf16x8 ones_rows = rowsum_selector(lane);

    auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
    auto tile = [&](int t, auto masked) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < BLOCKS; ++i) {
            constexpr int LAST = BLOCKS - 1;
            const int n = i == LAST ? 0 : i + 1;
            f32x16 &xc = x[i & 1], &xn = x[n & 1];
            auto exp4 = [&](int base) {
#pragma unroll
                for (int e = base; e < base + 4; ++e) {
                    xc[e] = __builtin_amdgcn_exp2f(xc[e]);
                }
            };
            exp4(0);
            xn = mfma(as_bf16x8(k0), q[n][0], zero16());
            fence();
            exp4(4);
            const bf16x8 p0 = pack8(xc, 0);
            xn = mfma(as_bf16x8(k1), q[n][1], xn);
            if constexpr (decltype(masked)::value) {
                xn = add_mask(add_mask(xn, i == LAST ? mn : m), shift & lower);
            }
            if (i == LAST - 1) {
                k0 = next[lane], k1 = next[64 + lane];
            }
            fence();
            exp4(8);
            o[i] = mfma(as_bf16x8(v0), p0, o[i]);
            fence();
            exp4(12);
            const bf16x8 p1 = pack8(xc, 8);
            sums[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones_rows, p0, sums[i], 0, 0, 0);
            o[i] = mfma(as_bf16x8(v1), p1, o[i]);
            sums[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones_rows, p1, sums[i], 0, 0, 0);
            fence();
            if (i == LAST) {
                v0 = next[128 + lane], v1 = next[192 + lane];
                if constexpr (decltype(masked)::value) {
                    m = mn, mn = mask_word_of(t + 2);
                }
            }
            fence();
        }
        next += TILE;
        next = next == end ? lds : next;
        if (--left == 0) {
            asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory"); // this wave's tile of the group behind the next one: asked for a group ago
            refill();
            left = W;
        }
    };
    for (int t = 0; t < masked_from; ++t) {
        tile(t, std::false_type{});
    }
    if (masked_from < NB) {
        m = mask_word_of(masked_from), mn = mask_word_of(masked_from + 1);
        x[0] = add_mask(add_mask(x[0], m), shift & lower);
        for (int t = masked_from; t < NB; ++t) {
            tile(t, std::true_type{});
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the gates, and requests past the last tile before the LDS is given back
    uint32_t again = 0; // blocks whose sums ran out of range
#pragma unroll
    for (int i = 0; i < BLOCKS; ++i) {
        const float l = rowsum_fetch(sums[i], lane);
        const bool stored = j + i < NB;
        if (__any(!(l > 1e-30f && l < 1e30f))) {
            again |= stored ? 1u << i : 0u;
        } else if (stored) {
            const uint4 *gate = lds + (gate_place * W + wave) * TILE + i * BLOCK_SLOTS + lane;
            store_average(p.q + (row + j + i) * BLOCK_SLOTS + lane, gate[0], gate[64], o[i], l);
        }
    }
    while (again != 0) {
        const int i = __builtin_ctz(again);
        again &= again - 1;
        attend_shifted<false>(p.k + row * BLOCK_SLOTS, p.v + row * BLOCK_SLOTS, p.words + (int64_t)b * NB * 32, nullptr,
                              p.q + (row + j + i) * BLOCK_SLOTS, p.g + (row + j + i) * BLOCK_SLOTS, NB, lane);
    }
}

// ---- the output projection ----
//
// act += avg . Wo^T + bo, row (b, s) of the product to row (b, s) of act, or transposed to row (s, b).  Bound by HBM: 2 C bytes a
// position in, and 4 C of act.  A wave keeps the weights of 32 features in registers, their head dims in the order of the fragments in which the
// gated average arrives; a workgroup of all features walks blocks of 32 positions, which its waves share in the LDS, the next block
// and its activations under way; with 256 channels, one workgroup a CU, the next two (medians of this kernel: MSA columns of
// 1024 x 384 125 -> 119 us, of 2000 x 300 186 -> 176, rows of 508 x 259 47 -> 45; with 128, two workgroups a CU, 2048 residues 617 -> 638).  The product (rows = features, columns = positions) crosses the LDS to meet the activation in whole
// cache lines.  act, weights and bias lie on any address.  With the weights in the LDS, read for every block by waves that walked
// alone, MSA rows of 508 x 259 took 52 us of this kernel, now 45, 300 x 300 39 and 31, columns of 500 x 100 27 and 21, of 1024 x 384 122 and 119,
// triangle attention of 2048 residues 650 and 618, of 1200 193 and 176.
template <int C>
__global__ __launch_bounds__(2 * C, 2) void output_projection_kernel(
    const uint4 *__restrict__ avg, const bf16_t *__restrict__ wo, const float *__restrict__ bo, bf16_t *__restrict__ act, int64_t ld,
    int B, int S, int H, int NB, int transposed)
{
    constexpr int CK = C / 16, THREADS = 2 * C, LOADS = CK * 64 / THREADS, PIECES = C / 8, AHEAD = C / 128;
    __shared__ uint4 block[CK * 64], result[32 * PIECES]; // a position's pieces XOR-ed with position % 16
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, g = lane >> 5;
    const int units = B * NB;
    const int64_t step = (transposed ? (int64_t)B : 1) * ld * 2;
    const int pos[2] = {tid / PIECES, tid / PIECES + 16}; // the thread's pieces of 8 features of the activation
    struct Block {
        bf16x8 in[LOADS], z[2];
        char *to[2];
    };
    auto fetch = [&](Block &t, int unit) __attribute__((always_inline)) {
        const int b = unit / NB, j = unit - b * NB, last = min(31, S - 1 - 32 * j); // last position of the block that is one
        const uint4 *src = avg + ((int64_t)b * H * NB + j) * BLOCK_SLOTS;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) { // k-steps 2 h and 2 h + 1 = head h
            const int at = tid + THREADS * i;
            t.in[i] = *reinterpret_cast<const bf16x8 *>(src + (int64_t)(at / BLOCK_SLOTS) * NB * BLOCK_SLOTS + at % BLOCK_SLOTS);
        }
        const int64_t row = transposed ? (int64_t)32 * j * B + b : (int64_t)b * S + 32 * j;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            t.to[i] = reinterpret_cast<char *>(act) + row * ld * 2 + min(pos[i], last) * step + tid % PIECES * 16;
            __builtin_memcpy(&t.z[i], t.to[i], 16);
        }
    };
    Block even, odd;
    fetch(even, blockIdx.x);
    if (AHEAD == 2) {
        fetch(odd, min((int)(blockIdx.x + gridDim.x), units - 1));
    }
    bf16x8 w[CK];
    load_half_lines<CK>(w, wo + 32 * wave * C, C, lane);
    f32x4 bv[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        __builtin_memcpy(&bv[a], bo + 32 * wave + 8 * a + 4 * g, 16);
    }
    {
        // elements e of lane half g: head dims 16 ks + 4 g + e (e < 4), 16 ks + 8 + 4 g + e - 4; through 2 KB that are the wave's own
        uint4 *own = result + 128 * wave;
#pragma unroll
        for (int ks = 0; ks < CK; ks += 2) {
            own[half_line_slot(lane >> 2, lane & 3)] = as_uint4(w[ks]);
            own[half_line_slot(16 + (lane >> 2), lane & 3)] = as_uint4(w[ks + 1]);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                uint2 lo, hi;
                __builtin_memcpy(&lo, reinterpret_cast<const char *>(own + half_line_slot(r, 2 * k)) + 8 * g, 8);
                __builtin_memcpy(&hi, reinterpret_cast<const char *>(own + half_line_slot(r, 2 * k + 1)) + 8 * g, 8);
                w[ks + k] = as_bf16x8(make_uint4(lo.x, lo.y, hi.x, hi.y));
            }
        }
    }
    auto do_block = [&](int unit, Block &now) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            block[tid + THREADS * i] = as_uint4(now.in[i]);
        }
        const int last = min(31, S - 1 - 32 * (unit % NB));
        const bf16x8 z[2] = {now.z[0], now.z[1]};
        char *const to[2] = {now.to[0], now.to[1]};
        __syncthreads(); // (the previous result has been read, too)
        if (unit + AHEAD * (int)gridDim.x < units) {
            fetch(now, unit + AHEAD * gridDim.x);
        }
        f32x16 acc;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            acc[v] = bv[v >> 2][v & 3];
        }
#pragma unroll
        for (int ks = 0; ks < CK; ++ks) {
            acc = mfma(w[ks], as_bf16x8(block[ks * 64 + lane]), acc);
        }
        const int p = pi_row(r);
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            bf16x4 ov;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                ov[c] = (bf16_t)acc[4 * a + c];
            }
            *(reinterpret_cast<bf16x4 *>(result + p * PIECES + ((4 * wave + a) ^ (p & 15))) + g) = ov;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const bf16x8 o = as_bf16x8(result[pos[i] * PIECES + (tid % PIECES ^ (pos[i] & 15))]);
            bf16x8 sum;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                sum[e] = (bf16_t)(to_f32(z[i][e]) + to_f32(o[e]));
            }
            if (pos[i] <= last) {
                __builtin_memcpy(to[i], &sum, 16);
            }
        }
    };
    for (int unit = blockIdx.x; unit < units; unit += AHEAD * gridDim.x) {
        do_block(unit, even);
        if (AHEAD == 2 && unit + (int)gridDim.x < units) {
            do_block(unit + gridDim.x, odd);
        }
    }
}

template <int C>
int launch_projection(const StreamedParams &p, hipStream_t stream)
{
    static size_t configured[KUTACC_DEVICE_SLOTS] = {};
    if (const hipError_t e = kutacc_opt_in_lds(reinterpret_cast<const void *>(&qkvg_projection_kernel<C>), projection_lds<C>(), configured)) {
        return kutacc_hip_status(e);
    }
    const int halves = C / 128; // workgroups that share a step, one per 128 channels of outputs
    const int64_t steps = ((int64_t)p.B * p.NB + 1) / 2, cap = std::max(1, kutacc_cu_count() / halves);
    const int64_t per = (steps + cap - 1) / cap;
    kutacc_prof::KernelTimer t("qkvg_projection_kernel", 8.0 * (double)p.B * p.S * C * C, stream);
    const int64_t runs = (steps + per - 1) / per;
    qkvg_projection_kernel<C><<<dim3((unsigned)(halves == 1 ? runs : (runs + 7) / 8 * 16)), 512, projection_lds<C>(), stream>>>(p, (int)per);
    return kutacc_hip_status(hipGetLastError());
}

template <int ROWS>
int launch_attention(StreamedParams p, hipStream_t stream)
{
    const int sets = (p.B + ROWS - 1) / ROWS;
    p.query_groups = (p.NB + WAVES - 1) / WAVES;
    const int parts = (p.query_groups + TOGETHER - 1) / TOGETHER, together = std::min(p.query_groups, TOGETHER);
    p.group_rows = std::min(sets, MEMBERS / together);
    p.set_groups = (sets + p.group_rows - 1) / p.group_rows;
    p.groups = p.set_groups * p.H * parts;
    const int64_t blocks = (int64_t)(p.groups + 7) / 8 * 8 * p.group_rows * together;
    kutacc_prof::KernelTimer t("streamed_attention_kernel", 4.0 * (double)p.B * p.S * p.S * p.H * HEAD, stream);
    streamed_attention_kernel<ROWS><<<dim3((unsigned)blocks), 64 * WAVES, Walk<ROWS>::LDS, stream>>>(p);
    return kutacc_hip_status(hipGetLastError());
}

int launch_plain(StreamedParams p, hipStream_t stream)
{
    // Three waves a workgroup instead of four where that leaves a tenth fewer queries past the row's end, as 9 .. 12 blocks do (300
    // sequences x 100 residues 27.9 -> 26.2 us; 900 x 300, 30 blocks for 32, 373 -> 382).
    const auto slots = [&](int waves) { return (p.NB + PLAIN_BLOCKS * waves - 1) / (PLAIN_BLOCKS * waves) * waves; };
    p.plain_waves = 10 * slots(3) < 9 * slots(4) ? 3 : 4;
    p.query_groups = slots(p.plain_waves) / p.plain_waves;
    p.groups = p.B * p.H;
    const int64_t blocks = ((int64_t)p.groups + 7) / 8 * 8 * p.query_groups;
    kutacc_prof::KernelTimer t("streamed_attention_kernel", 4.0 * (double)p.B * p.S * p.S * p.H * HEAD, stream);
    streamed_plain_kernel<<<dim3((unsigned)blocks), 64 * p.plain_waves, (size_t)RING * p.plain_waves * 4096, stream>>>(p);
    return kutacc_hip_status(hipGetLastError());
}

// workgroups a CU, as the registers allow with 256 channels; with 128, columns of 2048 x 2048 pairs 621 us, with three 658, with four 682, and
// no difference up to 1000 x 1000
template <int C>
constexpr int OUTPUT_PER_CU = C == 128 ? 2 : 1;
template <int C>
int launch_output(const StreamedParams &p, const void *wo, const float *bo, void *act, int64_t ld, bool transposed, hipStream_t stream)
{
    kutacc_prof::KernelTimer t("output_projection_kernel<residual>", 2.0 * (double)p.B * p.S * C * C, stream);
    const int64_t units = (int64_t)p.B * p.NB, full = (int64_t)kutacc_cu_count() * OUTPUT_PER_CU<C>;
    output_projection_kernel<C><<<dim3((unsigned)std::min(full, units)), 2 * C, 0, stream>>>(
        p.q, (const bf16_t *)wo, bo, (bf16_t *)act, ld, p.B, p.S, p.H, p.NB, transposed ? 1 : 0);
    return kutacc_hip_status(hipGetLastError());
}
} // namespace

namespace kutacc_launch {

namespace {
std::atomic<int> g_forced{0};
inline int64_t align256(int64_t v) { return (v + 255) / 256 * 256; }
int64_t blocks_of(int64_t S) { return (S + 31) / 32; }
int64_t row_bytes(int64_t S, int64_t C) { return blocks_of(S) * 32 * C * 2; } // one of q, k, v, gate of a batch row
int64_t tile_bytes(int64_t S, int64_t heads) { return align256(heads * blocks_of(S) * ((blocks_of(S) + 1) & ~(int64_t)1) * 4096); }
int64_t word_bytes(int64_t B, int64_t S) { return align256(B * blocks_of(S) * 132); } // mask words and flags
} // namespace

bool streamed_attention_forced() { return g_forced.load(std::memory_order_relaxed) != 0; }

int streamed_attention_tuning(const char *name, const char *value)
{
    if (std::strcmp(name, "streamed")) {
        return KUTACC_HIP_EINVAL;
    }
    g_forced.store(value && value[0] == '1' ? 1 : 0);
    return 0;
}

int64_t streamed_workspace_bytes(int64_t B, int64_t S, int64_t heads, bool pair_bias)
{
    return (pair_bias ? tile_bytes(S, heads) : 0) + word_bytes(B, S) + 4 * B * row_bytes(S, heads * HEAD);
}

bool streamed_attention_supports(const kutacc_hip_attention_args_t &a)
{
    const int64_t C = a.nheads * a.head_size;
    return a.dtype == KUTACC_DTYPE_BF16 && a.head_size == HEAD && (C == 128 || C == 256) && a.seq_len > 0 && a.seq_len <= (1 << 20) &&
           a.batch > 0 && a.batch <= (1 << 24) && a.batch * blocks_of(a.seq_len) <= INT32_MAX / 4;
}

int gating_attention_streamed(const kutacc_hip_attention_args_t &a, const FusedAttentionOptions &opt, void *workspace, int64_t bytes,
                              hipStream_t stream)
{
    const int64_t C = a.nheads * a.head_size, S = a.seq_len;
    const bool has_nb = a.nonbatched_bias != nullptr;
    if (!streamed_attention_supports(a) || opt.out_mode == FUSED_OUT_STORE || opt.ln_gamma == nullptr) {
        return KUTACC_HIP_EUNSUPPORTED;
    }
    if (bytes < streamed_workspace_bytes(a.batch, S, a.nheads, has_nb)) {
        return KUTACC_HIP_EINVAL;
    }
    char *ws = static_cast<char *>(workspace), *words = ws + (has_nb ? tile_bytes(S, a.nheads) : 0), *data = words + word_bytes(a.batch, S);
    int rc = has_nb && !opt.nb_tiles_ready ? pair_bias_tiles(a, ws, stream) : 0;
    if (rc != 0) {
        return rc;
    }
    StreamedParams p;
    std::memset(&p, 0, sizeof(p));
    p.x = (const bf16_t *)a.input, p.x_ld = a.input_ld, p.x_sb = opt.input_stride_b != 0 ? opt.input_stride_b : S * a.input_ld;
    p.ln_gamma = opt.ln_gamma, p.ln_beta = opt.ln_beta, p.ln_eps = opt.ln_eps;
    p.wq = (const bf16_t *)a.query_w, p.wk = (const bf16_t *)a.key_w, p.wv = (const bf16_t *)a.value_w, p.wg = (const bf16_t *)a.gating_w;
    p.bg = a.gating_b;
    p.bias = (const bf16_t *)a.bias, p.bias_sb = a.bias_stride_b, p.bias_sk = opt.bias_stride_k, p.bias_is_mask = opt.bias_is_mask ? 1 : 0;
    // (float)(1/sqrt(head_size)) as the reference forms it (gating_attention.cpp:68)
    p.qmul = (float)(1.0 / sqrt((double)HEAD)) * LOG2E;
    const int64_t each = a.batch * row_bytes(S, C);
    p.q = (uint4 *)data, p.k = (uint4 *)(data + each), p.v = (uint4 *)(data + 2 * each), p.g = (uint4 *)(data + 3 * each);
    p.tiles = has_nb ? (const f32x4 *)ws : nullptr;
    p.B = (int)a.batch, p.S = (int)S, p.H = (int)a.nheads, p.NB = (int)blocks_of(S), p.NT = (p.NB + 1) & ~1;
    p.words = (uint32_t *)words, p.flags = p.words + (int64_t)p.B * p.NB * 32;
    rc = C == 128 ? launch_projection<128>(p, stream) : launch_projection<256>(p, stream);
    if (rc == 0) {
        // Two rows a wave where four would leave CUs idle, below three workgroups to two CUs (8 heads of 1100 residues, whole block: 4, 8
        // and 16 sequences 155, 167 and 187 us against 165, 172 and 192 on four rows a wave; 24 and 64: 223 and 347 against 206 and 336).
        const int64_t fours = (a.batch + 3) / 4 * a.nheads * ((p.NB + WAVES - 1) / WAVES);
        rc = !has_nb                             ? launch_plain(p, stream)
             : 2 * fours >= 3 * kutacc_cu_count() ? launch_attention<4>(p, stream)
                                                  : launch_attention<2>(p, stream);
    }
    if (rc != 0) {
        return rc;
    }
    const bool transposed = opt.out_mode == FUSED_OUT_ADD_TRANSPOSED;
    return C == 128 ? launch_output<128>(p, a.output_w, a.output_b, a.out, a.out_ld, transposed, stream)
                    : launch_output<256>(p, a.output_w, a.output_b, a.out, a.out_ld, transposed, stream);
}

} // namespace kutacc_launch
