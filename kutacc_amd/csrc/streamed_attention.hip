// Gated attention of long batch rows for gfx950, bf16 storage, head size 32, 128 or 256 channels: the rows whose keys and
// values do not fit the LDS twice beside a head's weights (persistent_pair_kernel), in batches that fill the chip.
//
// Two kernels share the work, with K, V, Q and the gate in memory between them:
//
//   qkvg_projection_kernel    reads the input rows once, forms all four projections and writes them as the MFMA fragments
//       the attention loads -- 1 KB per store instruction, no layout change anywhere after it.
//   streamed_attention_kernel softmax(q.k^T + mask + pair bias).v * gate.  A wave owns the same 32 queries of two batch rows,
//       which share the pair bias (fp32 tiles in accumulator order, the C operand of both rows' logits MFMAs, as in
//       persistent_pair_kernel); a workgroup of four waves walks all keys of the two rows, its K and V staged
//       through a ring of three key tiles in the LDS.
//
// Against fused_head_kernel (one workgroup per row and head, K and V of the whole row in the LDS, projections in front):
// the pair bias costs no MFMAs and half the bytes, three waves per SIMD at every length instead of two, the projections
// run at the rate of the memory instead of behind one barrier per workgroup, and a row's length decides nothing.  The price
// is the four projections through memory, 8 bytes per channel and position.
//
// The order of positions, keys and head dims inside a fragment is that of the fused kernels (fused_attention.hip): lane r
// of a block of 32 positions stands for position pi(r), Q and K share their order of head dims, V and the probabilities
// their order of keys, so that accumulators are packed into operands as they are.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <climits>
#include <cstring>

#include "attention_util.h"
#include "launch_internal.h"
#include "mfma_tiles.h"
#include "profiler.h"

namespace {
using namespace kutacc_dev;

constexpr int HEAD = 32;
constexpr int BLOCK_SLOTS = 128; // 16-byte slots of a fragment pair: 32 positions x 32 head dims

struct StreamedParams {
    const bf16_t *x; // first batch row of the slice
    int64_t x_ld, x_sb;
    const bf16_t *wq, *wk, *wv, *wg;
    const float *bg;
    const bf16_t *bias;
    int64_t bias_sb, bias_sk;
    int bias_is_mask;
    float qmul; // log2(e) / sqrt(head size)
    uint4 *q, *g, *k, *v; // [batch row][head][block of 32 positions][2 k-steps][64 lanes]
    // [batch row][block][32]: mask bias of key pi(i) in log2 units as two bf16 (mask_word).  Their 2^-17 moves no probability: the bias
    // is formed from a bf16 mask, so it is 0, or at least 3.9e6 in size and 2^-8 of that from any other.  (A third part was 7 %
    // slower at 2048 residues, a tenth of them masked.)
    uint32_t *words;
    uint32_t *flags;      // [batch row][block]: some word of the block is not zero
    const f32x4 *tiles;   // pair bias: [head][query block][NT][4][64 lanes] (pair_bias_tiles_kernel)
    bf16_t *avg;          // first batch row of the slice
    int64_t avg_sb, avg_ss;
    int B, S, H, NB, NT; // batch rows of the slice, positions, heads, blocks, key tiles of `tiles` per query block
    int query_groups, pair_groups, groups, group_rows; // placement of the attention's workgroups
};

// ---- the projections ----
//
// Bound by HBM: per position 2 C bytes in and 8 C out.  Eight waves, one workgroup per CU (and per 128 channels of outputs); a
// wave owns one head's two matrices -- Q and gate, or K and V -- whose 32 x C blocks stay in its registers, and stages
// eight of the 64 positions of a step into the shared stage, requested a step ahead.
template <int C>
constexpr size_t projection_lds() { return (size_t)2 * 64 * (C / 8) * 16; }

template <int C>
__global__ __launch_bounds__(512, 1) void qkvg_projection_kernel(const StreamedParams p, int steps_per_group)
{
    constexpr int CK = C / 16, SLOTS = C / 8, LOADS = 8 * SLOTS / 64, ROWS = 64 / SLOTS; // rows per load instruction
    extern __shared__ uint4 lds[];                                                      // two stages of [64 positions][SLOTS]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, g = lane >> 5;
    const int h = (int)blockIdx.y * 4 + (wave & 3);
    const bool forms_kv = wave >= 4;

    const int blocks = p.B * p.NB, total_steps = (blocks + 1) / 2;
    const int first = (int)blockIdx.x * steps_per_group;
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
            t.r[u] = *reinterpret_cast<const uint4 *>(base + ((int64_t)pos * p.x_ld * 2 + 16 * (lane % SLOTS)));
        }
        advance(load_b, load_j);
        return t;
    };
    auto park = [&](int s, const Rows &t) {
#pragma unroll
        for (int u = 0; u < LOADS; ++u) {
            lds[s * 64 * SLOTS + slot(8 * wave + ROWS * u + lane / SLOTS, lane % SLOTS)] = t.r[u];
        }
    };
    Rows rows = load();
    bf16x8 w0[CK], w1[CK]; // Q and gate, or K and V
    {
        const bf16_t *m0 = forms_kv ? p.wk : p.wq, *m1 = forms_kv ? p.wv : p.wg;
#pragma unroll
        for (int ks = 0; ks < CK; ++ks) {
            const int at = (h * HEAD + r) * C + ks * 16 + g * 8;
            w0[ks] = as_bf16x8(load8_any(m0, at)), w1[ks] = as_bf16x8(load8_any(m1, at)); // once per workgroup: on any address
        }
    }
    park(0, rows);
    if (first + 1 < stop) {
        rows = load();
    }
    __syncthreads();

    int b = (2 * first) / p.NB, j = (2 * first) % p.NB; // the block being multiplied
    for (int step = first; step < stop; ++step) {
        const int s = (step - first) & 1;
        if (step + 1 < stop) {
            park(s ^ 1, rows);
            if (step + 2 < stop) {
                rows = load();
            }
        }
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            if (2 * step + half >= blocks) {
                break;
            }
            const uint4 *stage = lds + (s * 64 + 32 * half) * SLOTS;
            f32x16 a0 = zero16(), a1 = zero16();
            const int64_t at = (((int64_t)b * p.H + h) * p.NB + j) * BLOCK_SLOTS + lane;
            if (forms_kv) {
#pragma unroll
                for (int ks = 0; ks < CK; ++ks) {
                    const bf16x8 xf = as_bf16x8(stage[slot(pi_row(r), 2 * ks + g)]);
                    a0 = mfma(w0[ks], xf, a0);
                    a1 = mfma(xf, w1[ks], a1); // V: rows = keys, columns = head dims
                }
                p.k[at] = as_uint4(pack8(a0, 0)), p.k[at + 64] = as_uint4(pack8(a0, 8));
                p.v[at] = as_uint4(pack8(a1, 0)), p.v[at + 64] = as_uint4(pack8(a1, 8));
            } else {
#pragma unroll
                for (int ks = 0; ks < CK; ++ks) {
                    const bf16x8 xf = as_bf16x8(stage[slot(pi_row(r), 2 * ks + g)]);
                    a0 = mfma(w0[ks], xf, a0);
                    a1 = mfma(w1[ks], xf, a1);
                }
                const float *bg = p.bg + h * HEAD + 4 * g;
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    f32x4 bv;
                    __builtin_memcpy(&bv, bg + 8 * a, 16); // on any address
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        a0[4 * a + c] *= p.qmul;
                        a1[4 * a + c] += bv[c]; // the gate is rounded in front of its sigmoid, as where the reference stores it
                    }
                }
                p.q[at] = as_uint4(pack8(a0, 0)), p.q[at + 64] = as_uint4(pack8(a0, 8));
                p.g[at] = as_uint4(pack8(a1, 0)), p.g[at + 64] = as_uint4(pack8(a1, 8));
            }
            if (wave == 3 * half && blockIdx.y == 0) { // the mask of the block, by two waves in turn
                const int key = 32 * j + pi_row(r);
                float mv = -INFINITY;
                if (key < p.S) {
                    mv = to_f32(p.bias[(int64_t)b * p.bias_sb + (int64_t)key * p.bias_sk]);
                    if (p.bias_is_mask) {
                        mv = to_f32((bf16_t)fmaf(mv, 1e9f, -1e9f));
                    }
                    mv *= LOG2E;
                }
                if (lane < 32) {
                    p.words[((int64_t)b * p.NB + j) * 32 + lane] = mask_word(mv);
                }
                const bool any = __ballot(mv != 0.f) != 0;
                if (lane == 0) {
                    p.flags[(int64_t)b * p.NB + j] = any ? 1u : 0u;
                }
            }
            if (++j == p.NB) {
                j = 0, ++b;
            }
        }
        __syncthreads(); // the next stage is complete, this one no longer read
    }
}

// ---- the attention ----
constexpr int WAVES = 4;                      // query blocks per workgroup
constexpr int TILES_PER_GROUP = WAVES / 2;    // key tiles per barrier: four pieces of 1 KB for every wave
constexpr int RING = 3;                       // groups of tiles in the LDS
constexpr int TOGETHER = 8, MEMBERS = 64;     // query groups and workgroups of a placement group, at most
constexpr int TILE_SLOTS = 4 * BLOCK_SLOTS;   // K and V of one key tile of the two rows: [row][K, V][2][64]
constexpr int TILE_BYTES = TILE_SLOTS * 16;

// Repeat of one row's 32 queries after an overflow or underflow of the unshifted exponentials (a sum outside 1e-30 .. 1e30, a
// row with every key masked): the true row maxima first, then the probabilities with them subtracted.  Not a hot path:
// one row, operands straight from memory, no barrier.
template <bool HAS_NB>
__device__ __forceinline__ void attend_shifted(const uint4 *k, const uint4 *v, const uint32_t *words, const f32x4 *nbc, bf16x8 q0, bf16x8 q1,
                                               int NB, int lane, f32x16 &o_out, float &l_out)
{
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
    o_out = o;
    l_out = rowsum_fetch(sums, lane);
}

// Keys and values come straight into the LDS (global_load_lds_dwordx4), two key tiles at a time, so that every wave brings
// four pieces of 1 KB per group of tiles: a ring of three groups, one barrier per group.  At the barrier in front of group G,
// group G + 1 has landed and group G - 1 has been left by every wave; its place takes group G + 2.  Three workgroups share
// a CU: three waves per SIMD (the launch bound asks for 168 registers), 48 KB of ring each.
template <bool HAS_NB>
__global__ __launch_bounds__(768) void streamed_attention_kernel(const StreamedParams p)
{
    typedef __attribute__((address_space(3))) void *lds_ptr;
    extern __shared__ uint4 lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int NB = p.NB;

    // Workgroup ids are dealt round robin over the 8 XCDs; an XCD works on one group at a time: group_rows pairs of rows x
    // up to eight query groups of one head, which sweep the keys together, so that the group's K and V and pair bias come
    // from memory once and from the XCD's L2 after that.
    const int members = p.group_rows * min(p.query_groups, TOGETHER);
    const int local = (int)(blockIdx.x >> 3);
    const int group = (int)(blockIdx.x & 7) + 8 * (local / members), member = local % members;
    if (group >= p.groups) {
        return;
    }
    const int pair_group = group % p.pair_groups, rest = group / p.pair_groups;
    const int h = rest % p.H, query_part = rest / p.H;
    const int pair = pair_group * p.group_rows + member % p.group_rows, qg = query_part * TOGETHER + member / p.group_rows;
    if (2 * pair >= p.B || qg >= p.query_groups) {
        return;
    }
    const int bA = 2 * pair, bB = min(bA + 1, p.B - 1);
    const int j = qg * WAVES + wave;
    const int64_t rowA = ((int64_t)bA * p.H + h) * NB, rowB = ((int64_t)bB * p.H + h) * NB; // first fragment block of either row

    // The pieces u = 4 wave + i of a group of tiles: tile u / 8, piece u % 8 = [row][K, V][k-step].  Written out: as a builtin
    // the compiler takes every LDS read behind it for a reader of its data and waits for all loads in flight.
    const uint32_t ring = (uint32_t)(uintptr_t)(lds_ptr)lds, lane_bytes = 16u * (uint32_t)lane;
    auto request = [&](int first_tile, int place) { // tiles first_tile .. into group `place` of the ring
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int u = 4 * wave + i;
            const int t = min(first_tile + (u >> 3), NB - 1);
            const uint4 *src = ((u & 2) ? p.v : p.k) + (((u & 4) ? rowB : rowA) + t) * BLOCK_SLOTS + (u & 1) * 64;
            const uint32_t to = ring + (uint32_t)(place * TILES_PER_GROUP) * TILE_BYTES + (uint32_t)u * 1024u;
            load_to_lds(to, src, lane_bytes);
        }
    };
    request(0, 0);
    request(TILES_PER_GROUP, 1);
    int fill = 2, fill_tile = 2 * TILES_PER_GROUP; // the next group to ask for: its place in the ring, its first tile
    auto refill = [&] {
        request(fill_tile, fill);
        fill = fill == 2 ? 0 : fill + 1;
        fill_tile += TILES_PER_GROUP;
    };
    if (j >= NB) { // a wave without queries brings its share of the keys
        for (int t = 0; t < NB; t += TILES_PER_GROUP) {
            asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
            refill();
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        return;
    }

    const uint4 *qa = p.q + (rowA + j) * BLOCK_SLOTS, *qb = p.q + (rowB + j) * BLOCK_SLOTS;
    const bf16x8 qA0 = as_bf16x8(qa[lane]), qA1 = as_bf16x8(qa[64 + lane]), qB0 = as_bf16x8(qb[lane]), qB1 = as_bf16x8(qb[64 + lane]);
    const f32x4 *nbc = HAS_NB ? p.tiles + ((int64_t)h * NB + j) * p.NT * 256 : nullptr;
    const uint32_t *wordsA = p.words + (int64_t)bA * NB * 32, *wordsB = p.words + (int64_t)bB * NB * 32;
    auto load_nb = [&](int t) {
        f32x16 c = zero16();
        if constexpr (HAS_NB) {
            const int tc = min(t, NB - 1);
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const f32x4 v = nbc[(tc * 4 + a) * 64 + lane];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    c[4 * a + e] = v[e];
                }
            }
        }
        return c;
    };
    f32x16 C0 = load_nb(0), C1 = load_nb(1);

    // first key tile in which either row has a mask (the ragged tail of a row counts: its keys are at -inf)
    int masked_from = NB;
    for (int t0 = 0; t0 < NB; t0 += 64) {
        const int t = t0 + lane;
        const uint32_t f = t < NB ? (p.flags[(int64_t)bA * NB + t] | p.flags[(int64_t)bB * NB + t]) : 0u;
        const unsigned long long any = __ballot(f != 0u);
        if (any != 0) {
            masked_from = t0 + __builtin_ctzll(any);
            break;
        }
    }

    // The mask of a row as a rank-one MFMA: A holds (hi, lo) of the key of accumulator row i in k-slots 0 and 1, B ones there,
    // all else zero, also in the lanes of the upper half, so that an infinite mask value never meets a zero.
    const uint32_t lower = lane < 32 ? 0xffffffffu : 0u;
    auto mask_word_of = [&](const uint32_t *words, int t) { return words[min(t, NB - 1) * 32 + (lane & 31)] & lower; };
    auto add_mask = [&](f32x16 x, uint32_t w) {
        const bf16x8 ones = as_bf16x8(make_uint4(0x3f803f80u & lower, 0u, 0u, 0u));
        return mfma(as_bf16x8(make_uint4(w, 0u, 0u, 0u)), ones, x);
    };

    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory"); // groups 0 and 1 have landed, every wave's part of them
    refill();
    int left = TILES_PER_GROUP;                              // tiles of the current group still to come, this one included
    const uint4 *cur = lds, *const end = lds + RING * TILES_PER_GROUP * TILE_SLOTS, *next = lds + TILE_SLOTS; // tiles t and t + 1
    next = next == end ? lds : next;
    uint4 k0 = cur[lane], k1 = cur[64 + lane], v0, v1;
    f32x16 xa, xb;
    xa = mfma(as_bf16x8(k0), qA0, C0);
    xa = mfma(as_bf16x8(k1), qA1, xa);
    k0 = cur[2 * BLOCK_SLOTS + lane], k1 = cur[2 * BLOCK_SLOTS + 64 + lane];
    v0 = cur[BLOCK_SLOTS + lane], v1 = cur[BLOCK_SLOTS + 64 + lane];
    f32x16 oA = zero16(), oB = zero16();
    f32x4 sumsA = {0.f, 0.f, 0.f, 0.f}, sumsB = {0.f, 0.f, 0.f, 0.f}; // the row sums on the matrix pipe: see rowsum_selector
    const bf16x8 ones_rows = rowsum_selector(lane);
    uint32_t mA = 0, mB = 0; // mask words of (A, t + 1) and (B, t)

    auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
    // softmax and P.V of the finished logits xc (into o, sums); the logits of the next row and tile into xn from seed C with
    // query fragments q0, q1; then k0, k1 <- knext.  The fences deal the exponentials between the MFMAs.  The empty asm keeps C
    // live past the MFMA that reads it, so that xn gets registers of its own.
    auto half_step = [&](f32x16 &xc, f32x16 &xn, const f32x16 &C, bf16x8 q0, bf16x8 q1, f32x16 &o, f32x4 &sums, const uint4 *knext,
                         uint32_t mask_next, auto masked) {
        auto exp4 = [&](int base) {
#pragma unroll
            for (int e = base; e < base + 4; ++e) {
                xc[e] = __builtin_amdgcn_exp2f(xc[e]);
            }
        };
        exp4(0);
        xn = mfma(as_bf16x8(k0), q0, C);
        asm volatile("" ::"v"(C));
        fence();
        exp4(4);
        const bf16x8 p0 = pack8(xc, 0);
        xn = mfma(as_bf16x8(k1), q1, xn);
        if constexpr (decltype(masked)::value) {
            xn = add_mask(xn, mask_next);
        }
        k0 = knext[lane], k1 = knext[64 + lane];
        fence();
        exp4(8);
        o = mfma(as_bf16x8(v0), p0, o);
        fence();
        exp4(12);
        const bf16x8 p1 = pack8(xc, 8);
        sums = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones_rows, p0, sums, 0, 0, 0);
        o = mfma(as_bf16x8(v1), p1, o);
        sums = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones_rows, p1, sums, 0, 0, 0);
        fence();
    };
    // Tile t: finishes (A, t) and (B, t), forms the logits of (B, t) from C and of (A, t + 1) from Cn
    auto tile = [&](int t, f32x16 &C, f32x16 &Cn, auto masked) {
        half_step(xa, xb, C, qB0, qB1, oA, sumsA, next, mB, masked);
        v0 = cur[3 * BLOCK_SLOTS + lane], v1 = cur[3 * BLOCK_SLOTS + 64 + lane];
        fence(); // the loads stay behind the last reader of the registers they fill
        C = load_nb(t + 2);
        if constexpr (decltype(masked)::value) {
            mB = mask_word_of(wordsB, t + 1);
        }
        fence();
        half_step(xb, xa, Cn, qA0, qA1, oB, sumsB, next + 2 * BLOCK_SLOTS, mA, masked);
        v0 = next[BLOCK_SLOTS + lane], v1 = next[BLOCK_SLOTS + 64 + lane];
        if constexpr (decltype(masked)::value) {
            mA = mask_word_of(wordsA, t + 2);
        }
        cur = next;
        next += TILE_SLOTS;
        next = next == end ? lds : next;
        if (--left == 0) {
            // This wave's pieces of the group behind the next one have landed: it asked for them a group ago, and with a
            // pair bias its eight youngest loads are those of the last two tiles' bias, issued since.
            if constexpr (HAS_NB) {
                asm volatile("s_waitcnt vmcnt(8)\n\ts_barrier" ::: "memory");
            } else {
                asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
            }
            refill();
            left = TILES_PER_GROUP;
        }
    };
    auto run = [&](int from, int to, auto masked) {
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
        mB = mask_word_of(wordsB, masked_from), mA = mask_word_of(wordsA, masked_from + 1);
        xa = add_mask(xa, mask_word_of(wordsA, masked_from));
        run(masked_from, NB, std::true_type{});
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // requests past the last tile: let them land before the LDS is given back
    float lA = rowsum_fetch(sumsA, lane), lB = rowsum_fetch(sumsB, lane);
    if (__any(!(lA > 1e-30f && lA < 1e30f))) {
        attend_shifted<HAS_NB>(p.k + rowA * BLOCK_SLOTS, p.v + rowA * BLOCK_SLOTS, wordsA, nbc, qA0, qA1, NB, lane, oA, lA);
    }
    if (__any(!(lB > 1e-30f && lB < 1e30f))) {
        attend_shifted<HAS_NB>(p.k + rowB * BLOCK_SLOTS, p.v + rowB * BLOCK_SLOTS, wordsB, nbc, qB0, qB1, NB, lane, oB, lB);
    }
    const int qpos = j * 32 + pi_row(lane & 31);
    if (qpos < p.S) {
        auto store = [&](int b, int64_t row, const f32x16 &o, float l) {
            const uint4 *gf = p.g + (row + j) * BLOCK_SLOTS;
            const bf16x8 g0 = as_bf16x8(gf[lane]), g1 = as_bf16x8(gf[64 + lane]);
            f32x16 gv;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                gv[i] = sigmoid_f32(to_f32(g0[i])), gv[8 + i] = sigmoid_f32(to_f32(g1[i]));
            }
            store_gated(p.avg + (int64_t)b * p.avg_sb + (int64_t)qpos * p.avg_ss + h * HEAD + 4 * (lane >> 5), o, 1.0f / l, gv);
        };
        store(bA, rowA, oA, lA);
        if (bB != bA) {
            store(bB, rowB, oB, lB);
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
    qkvg_projection_kernel<C><<<dim3((unsigned)((steps + per - 1) / per), halves), 512, projection_lds<C>(), stream>>>(p, (int)per);
    return kutacc_hip_status(hipGetLastError());
}

template <bool HAS_NB>
int launch_attention(StreamedParams p, hipStream_t stream)
{
    constexpr size_t lds_bytes = (size_t)RING * TILES_PER_GROUP * TILE_BYTES;
    const int pairs = (p.B + 1) / 2;
    p.query_groups = (p.NB + WAVES - 1) / WAVES;
    const int parts = (p.query_groups + TOGETHER - 1) / TOGETHER, together = std::min(p.query_groups, TOGETHER);
    p.group_rows = std::min(pairs, MEMBERS / together);
    p.pair_groups = (pairs + p.group_rows - 1) / p.group_rows;
    p.groups = p.pair_groups * p.H * parts;
    const int64_t blocks = (int64_t)(p.groups + 7) / 8 * 8 * p.group_rows * together;
    kutacc_prof::KernelTimer t("streamed_attention_kernel", 4.0 * (double)p.B * p.S * p.S * p.H * HEAD, stream);
    streamed_attention_kernel<HAS_NB><<<dim3((unsigned)blocks), 64 * WAVES, lds_bytes, stream>>>(p);
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
           a.batch > 0 && a.batch <= (1 << 24) && a.batch * blocks_of(a.seq_len) <= INT32_MAX / 4 && a.input_ld % 8 == 0 &&
           kutacc_hip_aligned16(a.input) && a.avg_stride_h == HEAD && a.avg_stride_s % 8 == 0 && a.avg_stride_b == a.seq_len * a.avg_stride_s &&
           kutacc_hip_aligned16(a.avg);
}

int gating_attention_streamed(const kutacc_hip_attention_args_t &a, const FusedAttentionOptions &opt, void *workspace, int64_t bytes,
                              hipStream_t stream)
{
    const int64_t C = a.nheads * a.head_size, S = a.seq_len;
    const bool has_nb = a.nonbatched_bias != nullptr;
    if (!streamed_attention_supports(a) || opt.out_mode == FUSED_OUT_STORE || opt.ln_gamma != nullptr) {
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
    p.wq = (const bf16_t *)a.query_w, p.wk = (const bf16_t *)a.key_w, p.wv = (const bf16_t *)a.value_w, p.wg = (const bf16_t *)a.gating_w;
    p.bg = a.gating_b;
    p.bias = (const bf16_t *)a.bias, p.bias_sb = a.bias_stride_b, p.bias_sk = opt.bias_stride_k, p.bias_is_mask = opt.bias_is_mask ? 1 : 0;
    // (float)(1/sqrt(head_size)) as the reference forms it (gating_attention.cpp:68)
    p.qmul = (float)(1.0 / sqrt((double)HEAD)) * LOG2E;
    const int64_t each = a.batch * row_bytes(S, C);
    p.q = (uint4 *)data, p.k = (uint4 *)(data + each), p.v = (uint4 *)(data + 2 * each), p.g = (uint4 *)(data + 3 * each);
    p.tiles = has_nb ? (const f32x4 *)ws : nullptr;
    p.avg = (bf16_t *)a.avg, p.avg_sb = a.avg_stride_b, p.avg_ss = a.avg_stride_s;
    p.B = (int)a.batch, p.S = (int)S, p.H = (int)a.nheads, p.NB = (int)blocks_of(S), p.NT = (p.NB + 1) & ~1;
    p.words = (uint32_t *)words, p.flags = p.words + (int64_t)p.B * p.NB * 32;
    rc = C == 128 ? launch_projection<128>(p, stream) : launch_projection<256>(p, stream);
    if (rc == 0) {
        rc = has_nb ? launch_attention<true>(p, stream) : launch_attention<false>(p, stream);
    }
    if (rc != 0) {
        return rc;
    }
    // The projection adds its result to the activation on the way out (2048 residues: 411 us and 674 us of residual pass
    // before, 664 us together now).  Where it cannot (the activation, the output weights or bias not on 16 bytes), it leaves its result
    // where q was, which no kernel reads any more, and a pass of its own adds it.
    const int64_t M = a.batch * S;
    const bool transposed = opt.out_mode == FUSED_OUT_ADD_TRANSPOSED;
    if (row_projection_supports(a.avg, a.avg_stride_s, a.output_w, a.output_b, a.out, a.out_ld, M, C, C)) {
        return row_projection_residual(a.avg, a.avg_stride_s, a.output_w, a.output_b, a.out, a.out_ld, M, C, C, transposed ? S : 0, stream);
    }
    kutacc_hip_gemm_args_t g = {};
    g.m = M, g.n = g.k = C, g.batches = 1, g.dtype = KUTACC_DTYPE_BF16, g.path = KUTACC_HIP_PATH_AUTO;
    g.a = a.avg, g.a_stride_m = a.avg_stride_s, g.a_stride_k = 1, g.b = a.output_w, g.b_stride_n = C, g.b_stride_k = 1;
    g.c = p.q, g.c_stride_m = C, g.bias = a.output_b, g.bias_axis = 1;
    rc = pair_gemm(g, stream);
    return rc != 0 ? rc : residual_add(a.out, p.q, transposed ? S : a.batch, transposed ? a.batch : S, C, transposed, KUTACC_DTYPE_BF16, stream);
}

} // namespace kutacc_launch
