// Global (extra-MSA column) attention for gfx950, bf16 storage, 64 channels
// (reference src/attention/global_attention.cpp:30-164; nchannels == 64 is hard-wired there, :172).
//
// Per batch row b there is ONE query per head, the masked mean of the row's tokens, and ONE key/value
// head shared by all heads:
//   q_avg = sum_s mask[s] x[s,:] / (sum_s mask[s] + 1e-10);  q = q_avg.Wq^T  viewed [H, d]
//   logit[h,s] = q[h].(Wk x[s]) / sqrt(d) + (mask[s]*1e9 - 1e9);  p = softmax_s
//   wavg[h,:] = sum_s p[h,s] (Wv x[s]);  out[s,:] = (sigmoid(x[s].Wg^T + bg) * wavg).Wo^T + bo
// One workgroup owns a batch row and walks it in 32-token tiles in three phases: (A) masked mean, (B) logits, online
// softmax and weighted average, (C) gate, gating and output projection.  A wave keeps the fragments of its first tiles in
// registers after phase A -- all of them up to 1024 tokens, 80 tiles of a longer row's -- and what is left of a longer row
// is read again in phases B and C, straight into the LDS.  Nothing but q_avg and out is written to memory.  All
// contractions are v_mfma_f32_32x32x16_bf16:
//   B: logits^T[s, h] = X[s, :] . QK^T with QK[h, :] = q[h].Wk / sqrt(d) folded per batch row (heads are the
//      columns, 8 of 32 used for H = 8); V[s, e] = X . Wv^T; O^T[e, h] += V^T . P^T -- the accumulators
//      of the first two products are directly the operands of the third, as in the gated attention
//      kernels (rows of a tile are the contraction index of the third product on both sides).
//   C: G^T[c, s] = Wg . X^T with the rows of Wg ordered so that a lane's accumulators are the k-slots of
//      the next product's B operand; OUT^T[o, s] = Wo . gated^T with the rows of Wo ordered so that a lane
//      holds 16 consecutive output features of its token (two 16-byte stores).
// The -1e9 mask bias is the accumulator's initial value and absorbs the logit in fp32, so a row whose mask
// is all zero attends uniformly, as in the reference.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "device_util.h"
#include "launch_internal.h"
#include "mfma_tiles.h"
#include "profiler.h"

using namespace kutacc_dev;

namespace {

constexpr int GC = 64;        // channels
constexpr int MAX_PARTS = 8;  // workgroups of a batch row
constexpr int PANEL_SLOTS = 288; // of a wave: 32 rows of 128 bytes, or 64 lanes of MERGE_LD floats
constexpr int MERGE_LD = 18;  // floats per lane in the cross-wave merge area: m, l, 16 accumulators

struct GlobalParams {
    const bf16_t *x, *mask, *wq, *wk, *wv, *wg, *wo;
    const float *bg, *bo;
    bf16_t *q_avg, *out;
    int64_t x_sb, x_ss, mask_sb, qavg_sb, out_sb, out_ss;
    int B, S, H, d, NT;
    int whole, parts; // batch rows that have one workgroup each; workgroups of each row behind them
    float scale;
};

// channel that accumulator register v of lane half g holds in row block rb of the gate product
__device__ __forceinline__ int gate_channel(int rb, int v, int g)
{
    const int idx = rb * 16 + v;
    return 16 * (idx >> 3) + 8 * g + (idx & 7);
}

// A wave keeps the fragments of its first KEEP tiles in registers from phase A on.  STREAM: the row may have more tiles than
// NW * KEEP; the rest is read again in every phase, straight into the LDS, two tiles of a wave ahead.
// What bounds it: in phase C the vector ALU (two transcendentals per gate element, 67 % busy on a row that has the chip to
// itself), in phases A and B the memory.  Measured at 5120 tokens x 384 rows: phases 48 + 36 + 100 us; 220 us with every
// phase streaming the whole row through registers, 189 with 64 of its 160 tiles kept, 186.5 with 80, for which gate bias and average are read
// from the LDS per tile (4000 x 300 146.5 -> 144).  1508 x 107: 32.4 -> 24.9 us.
template <int NW, int KEEP, bool STREAM>
__global__ __launch_bounds__(64 * NW, 2) void global_attention_kernel(GlobalParams p)
{
    constexpr int NTHR = 64 * NW;
    bf16x8 xs[KEEP][4];
    extern __shared__ uint4 lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, g = lane >> 5;
    const int S = p.S, NT = p.NT, H = p.H, d = p.d;
    // Workgroup ids are dealt round robin over the 8 XCDs: the parts of a row are eight ids apart, so that its tiles come from one L2.
    int b = (int)blockIdx.x, put_from = 0, put_to = NT; // the tiles it puts out
    if (NW == 8 && b >= p.whole) { // (rows of four waves are never shared)
        const int idx = b - p.whole, part = (idx >> 3) % p.parts;
        b = p.whole + (idx >> 3) / p.parts * 8 + (idx & 7);
        if (b >= p.B) {
            return;
        }
        put_from = NT * part / p.parts, put_to = NT * (part + 1) / p.parts;
    }
    // A wave's tiles are wave + NW * i.  All workgroups of a row take them in the same order, so that they have the same sums, and find in one L2
    // what another has just read; a part keeps those from the first one on that it puts out (or the last KEEP).  Beginning with its own tiles, each
    // part had sums of its own: tokens of a row differed by a bf16 unit of the average, 5120 x 60 took 52.5 us and takes 45.0, 4000 x 300 115.5 and 117.5.
    const int count = (NT - wave + NW - 1) / NW;
    const int kept_from = STREAM ? max(0, min((put_from - wave + NW - 1) / NW, count - KEEP)) : 0;
    auto kept_tile = [&](int i) { return wave + NW * (kept_from + i); };
    const int spad = NT * 32;
    // STREAM: ten tiles leave no registers beside them for constants and weights, which are read per tile, and tiles are kept from one another
    // (rows that are kept whole have them, and lose by it: 300 tokens x 100 rows 11.3 -> 11.8 us, 512 x 300 19.5 -> 20.3, 1024 x 384 33.6 -> 34.2).
    auto per_tile_lane = [&] {
        int l = lane;
        if constexpr (STREAM) {
            asm volatile("" : "+v"(l)); // opaque: what is addressed with it stays where it is read
        }
        return l;
    };
    auto fence = [] {
        if constexpr (STREAM) {
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    uint4 *qk_frag = lds;            // [4 k-steps][64 lanes]
    uint4 *wv_frag = qk_frag + 256;  // [4][64]
    uint4 *wg_frag = wv_frag + 256;  // [2 row blocks][4][64]
    uint4 *wo_frag = wg_frag + 512;  // [2 row blocks][4][64]
    uint4 *wk_rows = wo_frag + 512;  // the key weights as they lie in memory, [d][64 channels] bf16 (d <= 32)
    uint4 *panels = wk_rows + 256;                  // [NW][PANEL_SLOTS]: a panel of phase A, the merge area of phase B
    uint4 *panel = panels + wave * PANEL_SLOTS;
    uint4 *ring = panels + NW * PANEL_SLOTS + wave * 512; // STREAM: two tiles per wave
    bf16_t *mask16 = reinterpret_cast<bf16_t *>(panels + NW * (PANEL_SLOTS + (STREAM ? 512 : 0))); // per token, -inf past S
    float *part = reinterpret_cast<float *>(mask16 + spad); // [NW waves][68]: channel sums, mask sum
    float *qavg = part + NW * 68;                           // [64]
    float *qv = qavg + GC;                                  // [64] q, bf16-rounded
    float *wavg = qv + GC;                                  // [64]
    float *bos = wavg + GC;                                 // [64] output bias
    float *bgs = bos + GC;                                  // [64] gate bias (eight waves)
    float *merge = reinterpret_cast<float *>(panels);       // [NW waves][64 lanes][MERGE_LD]

    const bf16_t *xb = p.x + (int64_t)b * p.x_sb;
    const uint32_t x_pitch = (uint32_t)p.x_ss; // tokens of a row by 32-bit byte offsets from xb (the launcher checks the range)

    // Requested before anything else, so that their latency passes under the staging of the weights: the first tiles of
    // the row (all of a wave's tiles when they are kept in registers and there are at most four) and this thread's slice
    // of the query weights (output o = tid / TPR, channels part * 64 / TPR ...).
    constexpr int PRE = STREAM ? 1 : 4; // beside ten tiles there are no registers for more
    PanelRegs ahead[PRE];
#pragma unroll
    for (int i = 0; i < PRE; ++i) {
        const int t = kept_tile(i);
        ahead[i] = panel_load_near(xb, x_pitch, (t < NT ? t : NT - 1) * 32, S - 1, 0, lane);
    }
    // The tiles that are not kept: the n-th of them.  In phases A and B they come through the ring around the kept ones, in phase C behind them.
    const int streamed = max(0, count - KEEP);
    auto streamed_tile = [&](int n) { return wave + NW * (n < kept_from ? n : n + KEEP); };
    const uint32_t ring_lds = (uint32_t)(uintptr_t)(const lds_char *)ring;
    auto ask = [&](int n) { // the n-th streamed tile into its slot of the ring, in the panel's layout
        const int at = streamed_tile(n), slot = n & 1;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int rl = lane >> 3, row = min(at * 32 + 8 * i + rl, S - 1);
            load_to_lds(ring_lds + slot * 4096u + i * 1024u, xb, __umul24((uint32_t)row, 2u * x_pitch) + 16u * (uint32_t)((lane & 7) ^ rl ^ (i >> 1)));
        }
    };
    auto stream_start = [&](int from, int end) {
        if (STREAM && from < end) {
            ask(from);
            if (from + 1 < end) {
                ask(from + 1);
            }
        }
    };
    struct Tile {
        bf16x8 f[4];
    };
    auto ring_tile = [&](int n, int end) { // out of the ring, and the tile after the next one asked for in its place
        const int slot = n & 1;
        Tile x;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            x.f[ks] = as_bf16x8(ring[slot * 256 + panel_slot(r, 2 * ks + g)]);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (n + 2 < end) {
            ask(n + 2);
        }
        return x;
    };
    // ... of which those up to this one are put out, from kept_from on: a part that has more than the kept tiles keeps its first ones
    const int put_streamed = max(0, (put_to - wave + NW - 1) / NW - KEEP);
    stream_start(0, streamed);
    auto walk = [&](int from, int to, auto f) __attribute__((always_inline)) { // f(t, fragments) of streamed tiles, all of which are asked for in turn
#pragma unroll 1
        for (int n = from; n < to; ++n) {
            if (n + 1 < streamed) {
                wait_for_loads<4>(); // all but the next tile's
            } else {
                wait_for_loads<0>();
            }
            const Tile x = ring_tile(n, streamed);
            f(streamed_tile(n), x.f);
        }
    };
    constexpr int TPR = NTHR / GC, WQV = GC / TPR / 8; // threads per output of q, 16-byte pieces per thread
    uint4 wq_part[WQV];
#pragma unroll
    for (int v = 0; v < WQV; ++v) {
        wq_part[v] = *reinterpret_cast<const uint4 *>(p.wq + (tid / TPR) * GC + (tid % TPR) * (GC / TPR) + v * 8);
    }

    // ---- weights of phases B and C as MFMA fragments; mask ----
    for (int idx = tid; idx < d * 8; idx += NTHR) {
        wk_rows[idx] = reinterpret_cast<const uint4 *>(p.wk)[idx];
    }
    for (int idx = tid; idx < 256; idx += NTHR) {
        const int ks = idx >> 6, l = idx & 63, e = l & 31, gg = l >> 5;
        uint4 v = {0u, 0u, 0u, 0u};
        if (e < d) {
            v = *reinterpret_cast<const uint4 *>(p.wv + e * GC + ks * 16 + gg * 8);
        }
        wv_frag[idx] = v;
    }
    for (int idx = tid; idx < 512; idx += NTHR) {
        const int rb = idx >> 8, ks = (idx >> 6) & 3, l = idx & 63, i = l & 31, gg = l >> 5;
        const int ch = gate_channel(rb, 4 * (i >> 3) + (i & 3), (i >> 2) & 1);
        wg_frag[idx] = *reinterpret_cast<const uint4 *>(p.wg + ch * GC + ks * 16 + gg * 8);
        const int o = 32 * rb + pi_row(i);
        wo_frag[idx] = *reinterpret_cast<const uint4 *>(p.wo + o * GC + ks * 16 + gg * 8);
    }
    for (int s = tid; s < spad; s += NTHR) {
        mask16[s] = s < S ? p.mask[(int64_t)b * p.mask_sb + s] : (bf16_t)-INFINITY;
    }
    if (tid < GC) {
        bos[tid] = p.bo[tid];
        if constexpr (NW == 8) {
            bgs[tid] = p.bg[tid];
        }
    }
    __syncthreads();

    // ---- phase A: masked mean of the row, q, and the folded query-key matrix ----
    {
        float acc[4][8];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                acc[ks][e] = 0.f;
            }
        }
        float msum = 0.f;
        auto add_tile = [&](int t, const bf16x8 (&xf)[4]) {
            float m = to_f32(mask16[t * 32 + r]);
            m = m == -INFINITY ? 0.f : m;
            msum += g == 0 ? m : 0.f;
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    acc[ks][e] = fmaf(m, to_f32(xf[ks][e]), acc[ks][e]);
                }
            }
        };
        if constexpr (STREAM) {
            walk(0, kept_from, add_tile);
        }
        // the loads of the next PRE tiles are in flight while this one is summed
#pragma unroll
        for (int i = 0; i < KEEP; ++i) {
            const int t = kept_tile(i);
            if (t >= NT) {
                break;
            }
            panel_store(panel, lane, ahead[i % PRE]);
            if (i + PRE < KEEP) {
                const int tn = t + NW * PRE;
                ahead[i % PRE] = panel_load_near(xb, x_pitch, (tn < NT ? tn : NT - 1) * 32, S - 1, 0, lane);
            }
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                xs[i][ks] = as_bf16x8(panel[panel_slot(r, 2 * ks + g)]);
            }
            add_tile(t, xs[i]);
            fence();
        }
        if constexpr (STREAM) {
            walk(kept_from, streamed, add_tile);
            stream_start(0, streamed);
        }
        // sum over the 32 lanes of each half (they hold different tokens of the same channels)
        msum = group_sum<32>(msum);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                acc[ks][e] = group_sum<32>(acc[ks][e]);
            }
        }
        if (r == 0) {
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    part[wave * 68 + ks * 16 + g * 8 + e] = acc[ks][e];
                }
            }
            if (g == 0) {
                part[wave * 68 + 64] = msum;
            }
        }
    }
    __syncthreads();
    if (tid < GC) {
        float tot = 0.f, ms = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            tot += part[w * 68 + tid];
            ms += part[w * 68 + 64];
        }
        const bf16_t qa = (bf16_t)(tot * (1.0f / (ms + 1e-10f))); // reference :66-74
        qavg[tid] = to_f32(qa);
        if (p.q_avg != nullptr && put_from == 0) {
            p.q_avg[(int64_t)b * p.qavg_sb + tid] = qa;
        }
    }
    __syncthreads();
    {
        // q[o] = sum_c q_avg[c] wq[o][c]: TPR neighbouring threads share an output, each with the slice it fetched at the start
        float a = 0.f;
#pragma unroll
        for (int v = 0; v < WQV; ++v) {
            const bf16x8 w8 = as_bf16x8(wq_part[v]);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                a = fmaf(qavg[(tid % TPR) * (GC / TPR) + v * 8 + e], to_f32(w8[e]), a);
            }
        }
#pragma unroll
        for (int off = TPR / 2; off > 0; off >>= 1) {
            a += __shfl_xor(a, off, 64);
        }
        if (tid % TPR == 0) {
            qv[tid / TPR] = to_f32((bf16_t)a); // the reference stores q as bf16 (:76-80)
        }
    }
    __syncthreads();
    if (tid < 256) {
        // B operand of the logits product: column h (zero for h >= H), 8 channels per lane and k-step
        const int ks = tid >> 6, h = r;
        float a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (h < H) {
            for (int e = 0; e < d; ++e) {
                const bf16x8 w8 = as_bf16x8(wk_rows[e * 8 + ks * 2 + g]); // channels ks*16 + g*8 .. +8 of key row e
                const float qe = qv[h * d + e];
#pragma unroll
                for (int e8 = 0; e8 < 8; ++e8) {
                    a[e8] = fmaf(qe, to_f32(w8[e8]), a[e8]);
                }
            }
        }
        bf16x8 f;
#pragma unroll
        for (int e8 = 0; e8 < 8; ++e8) {
            f[e8] = (bf16_t)(a[e8] * p.scale);
        }
        qk_frag[ks * 64 + lane] = as_uint4(f);
    }
    __syncthreads();

    // ---- phase B: logits, online softmax, weighted average of V; one (m, l, O^T) state per wave ----
    {
        f32x16 o = zero16();
        float m_run = -1e30f, lsum = 0.f;
        auto attend = [&](int t, const bf16x8 (&xf)[4]) {
            const int lane = per_tile_lane(), g = lane >> 5;
            f32x16 x1, vv = zero16();
            const bf16x4 *mb4 = reinterpret_cast<const bf16x4 *>(mask16 + t * 32 + 4 * g);
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const bf16x4 mv = mb4[2 * a];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    x1[4 * a + c] = fmaf(to_f32(mv[c]), 1e9f, -1e9f); // reference :120-121
                }
            }
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                x1 = mfma(xf[ks], as_bf16x8(qk_frag[ks * 64 + lane]), x1);
                vv = mfma(xf[ks], as_bf16x8(wv_frag[ks * 64 + lane]), vv);
            }
            float mx = x1[0];
#pragma unroll
            for (int v = 1; v < 16; ++v) {
                mx = fmaxf(mx, x1[v]);
            }
            mx = half_swap_max(mx);
            const float m_new = fmaxf(m_run, mx);
            const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * LOG2E);
            lsum *= alpha;
            const float ml = -m_new * LOG2E;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                o[v] *= alpha;
                x1[v] = __builtin_amdgcn_exp2f(fmaf(x1[v], LOG2E, ml));
            }
            m_run = m_new;
            const bf16x8 p0 = pack8(x1, 0), p1 = pack8(x1, 8);
#pragma unroll
            for (int v = 0; v < 8; ++v) {
                lsum += to_f32(p0[v]) + to_f32(p1[v]);
            }
            o = mfma(pack8(vv, 0), p0, o);
            o = mfma(pack8(vv, 8), p1, o);
            fence();
        };
        if constexpr (STREAM) {
            walk(0, kept_from, attend);
        }
#pragma unroll
        for (int i = 0; i < KEEP; ++i) {
            if (kept_tile(i) >= NT) {
                break;
            }
            attend(kept_tile(i), xs[i]);
        }
        if constexpr (STREAM) {
            walk(kept_from, streamed, attend);
            stream_start(kept_from, put_streamed);
        }
        float *mine = merge + (wave * 64 + lane) * MERGE_LD;
        mine[0] = m_run;
        mine[1] = half_swap_sum(lsum);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            mine[2 + v] = o[v];
        }
    }
    __syncthreads();
    if (wave == 0) {
        float mw[NW], lw[NW];
        float M = -1e30f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            mw[w] = merge[(w * 64 + lane) * MERGE_LD];
            lw[w] = merge[(w * 64 + lane) * MERGE_LD + 1];
            M = fmaxf(M, mw[w]);
        }
        float L = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            mw[w] = __builtin_amdgcn_exp2f((mw[w] - M) * LOG2E);
            L = fmaf(lw[w], mw[w], L);
        }
        const float inv = 1.0f / L;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            float a = 0.f;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                a = fmaf(merge[(w * 64 + lane) * MERGE_LD + 2 + v], mw[w], a);
            }
            const int e = 8 * (v >> 2) + 4 * g + (v & 3);
            if (r < H && e < d) {
                wavg[r * d + e] = to_f32((bf16_t)(a * inv)); // the reference stores the weighted average as bf16 (:126-130)
            }
        }
    }
    __syncthreads();

    // ---- phase C: gate, gating, output projection ----
    {
        // per-channel constants of the gating, in the order the accumulators hold them
        constexpr int KEPT = STREAM ? 1 : 32;
        float bgv[KEPT], wv_[KEPT];
        if constexpr (!STREAM) {
#pragma unroll
            for (int i = 0; i < 32; ++i) {
                const int ch = gate_channel(i >> 4, i & 15, g);
                bgv[i] = NW == 8 ? bgs[ch] : p.bg[ch], wv_[i] = wavg[ch];
            }
        }
        auto put_out = [&](int t, const bf16x8 (&xf)[4]) {
            const int lane = per_tile_lane(), r = lane & 31, g = lane >> 5;
            auto four = [&](const float *at, const float (&kept)[KEPT], int rb, int a) { // constants 4 a .. 4 a + 3 of row block rb
                f32x4 v;
                if constexpr (STREAM) { // gate_channel(rb, 4 a, g) and the three behind it
                    v = *reinterpret_cast<const f32x4 *>(at + 32 * rb + 8 * g + 16 * (a >> 1) + 4 * (a & 1));
                } else {
                    v = f32x4{kept[16 * rb + 4 * a], kept[16 * rb + 4 * a + 1], kept[16 * rb + 4 * a + 2], kept[16 * rb + 4 * a + 3]};
                }
                return v;
            };
            bf16x8 gf[4];
#pragma unroll
            for (int rb = 0; rb < 2; ++rb) {
                f32x16 ga;
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    const f32x4 bv = four(bgs, bgv, rb, a);
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        ga[4 * a + c] = bv[c];
                    }
                }
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) {
                    ga = mfma(as_bf16x8(wg_frag[(rb * 4 + ks) * 64 + lane]), xf[ks], ga);
                }
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    const f32x4 wv = four(wavg, wv_, rb, a);
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        ga[4 * a + c] = wv[c] * sigmoid_fast(ga[4 * a + c]);
                    }
                }
                gf[2 * rb] = pack8(ga, 0);
                gf[2 * rb + 1] = pack8(ga, 8);
            }
            const int s = t * 32 + r;
#pragma unroll
            for (int ob = 0; ob < 2; ++ob) {
                f32x16 oa;
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    const f32x4 bv = *reinterpret_cast<const f32x4 *>(bos + 32 * ob + 16 * g + 4 * a);
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        oa[4 * a + c] = bv[c];
                    }
                }
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) {
                    oa = mfma(as_bf16x8(wo_frag[(ob * 4 + kk) * 64 + lane]), gf[kk], oa);
                }
                if (s < S) {
                    char *row_out = reinterpret_cast<char *>(p.out + (int64_t)b * p.out_sb + 32 * ob); // uniform
                    uint4 *dst = reinterpret_cast<uint4 *>(row_out + (__umul24((uint32_t)s, 2u * (uint32_t)p.out_ss) + 32u * g));
                    dst[0] = as_uint4(pack8(oa, 0));
                    dst[1] = as_uint4(pack8(oa, 8));
                }
            }
            fence();
        };
#pragma unroll
        for (int i = 0; i < KEEP; ++i) {
            if (kept_tile(i) >= put_to) {
                break;
            }
            if (NW == 4 || kept_tile(i) >= put_from) {
                put_out(kept_tile(i), xs[i]);
            }
        }
        if constexpr (STREAM) {
            for (int n = kept_from; n < put_streamed; ++n) {
                // younger than the tile's loads are the stores of the two tiles before it, four each (of kept ones, for the
                // first two tiles)
                wait_for_loads<8>();
                const Tile x = ring_tile(n, put_streamed);
                put_out(streamed_tile(n), x.f);
            }
        }
    }
}

// Dynamic LDS of global_attention_kernel for NT tiles: staged weights, the waves' panels and rings (16-byte units), mask
// (bf16), then per-wave sums and the vectors of the row (floats).
constexpr size_t LDS_PER_WORKGROUP = 160 * 1024;
constexpr size_t lds_bytes_for(int nw, bool stream, int nt)
{
    return (size_t)(256 + 256 + 512 + 512 + 256 + nw * (PANEL_SLOTS + (stream ? 512 : 0))) * 16 + (size_t)nt * 64 + (size_t)(nw * 68 + 5 * GC) * 4;
}
constexpr int MAX_SEQ_LEN = 12288;
static_assert(lds_bytes_for(8, true, MAX_SEQ_LEN / 32) <= LDS_PER_WORKGROUP);

template <int NW, int KEEP, bool STREAM>
hipError_t launch(const GlobalParams &p, hipStream_t stream)
{
    static size_t configured[KUTACC_DEVICE_SLOTS] = {};
    const size_t lds_bytes = lds_bytes_for(NW, STREAM, p.NT);
    const auto kernel = &global_attention_kernel<NW, KEEP, STREAM>;
    if (const hipError_t e = kutacc_opt_in_lds(reinterpret_cast<const void *>(kernel), lds_bytes, configured)) {
        return e;
    }
    const int64_t rest = p.B - p.whole;
    kernel<<<dim3((unsigned)(p.whole + (rest + 7) / 8 * 8 * p.parts)), 64 * NW, lds_bytes, stream>>>(p);
    return hipGetLastError();
}

} // namespace

namespace kutacc_launch {

int global_attention(const kutacc_hip_global_attention_args_t &a, hipStream_t stream)
{
    if (a.batch <= 0 || a.seq_len <= 0 || a.nheads <= 0 || a.head_size <= 0 || !a.q_data || !a.q_mask || !a.query_w ||
        !a.key_w || !a.value_w || !a.gating_w || !a.output_w || !a.gating_b || !a.output_b || !a.out) {
        return KUTACC_HIP_EINVAL;
    }
    if (a.dtype != KUTACC_DTYPE_BF16 || a.nheads * a.head_size != GC || a.nheads > 32 || a.head_size > 32 ||
        a.batch > INT32_MAX || a.seq_len > MAX_SEQ_LEN) {
        return KUTACC_HIP_EUNSUPPORTED;
    }
    // tokens of a batch row are addressed by 32-bit byte offsets from its first one
    if (a.q_data_stride_s <= 0 || a.out_stride_s <= 0 || a.q_data_stride_s >= (1 << 22) || a.out_stride_s >= (1 << 22) ||
        a.seq_len >= (1 << 23) || (a.seq_len + 32) * a.q_data_stride_s * 2 >= ((int64_t)1 << 31) ||
        (a.seq_len + 32) * a.out_stride_s * 2 >= ((int64_t)1 << 31)) {
        return KUTACC_HIP_EUNSUPPORTED;
    }
    // 16-byte row loads of x and the weights, 16-byte stores of out rows
    if (a.q_data_stride_s % 8 != 0 || a.q_data_stride_b % 8 != 0 || a.out_stride_s % 8 != 0 || a.out_stride_b % 8 != 0 ||
        !kutacc_hip_aligned16(a.q_data) || !kutacc_hip_aligned16(a.out) || !kutacc_hip_aligned16(a.query_w) || !kutacc_hip_aligned16(a.key_w) ||
        !kutacc_hip_aligned16(a.value_w) || !kutacc_hip_aligned16(a.gating_w) || !kutacc_hip_aligned16(a.output_w)) {
        return KUTACC_HIP_EUNSUPPORTED;
    }
    GlobalParams p;
    p.x = (const bf16_t *)a.q_data, p.mask = (const bf16_t *)a.q_mask;
    p.wq = (const bf16_t *)a.query_w, p.wk = (const bf16_t *)a.key_w, p.wv = (const bf16_t *)a.value_w;
    p.wg = (const bf16_t *)a.gating_w, p.wo = (const bf16_t *)a.output_w;
    p.bg = a.gating_b, p.bo = a.output_b;
    p.q_avg = (bf16_t *)a.q_avg, p.out = (bf16_t *)a.out;
    p.x_sb = a.q_data_stride_b, p.x_ss = a.q_data_stride_s, p.mask_sb = a.q_mask_stride_b;
    p.qavg_sb = a.q_avg_stride_b, p.out_sb = a.out_stride_b, p.out_ss = a.out_stride_s;
    p.B = (int)a.batch, p.S = (int)a.seq_len, p.H = (int)a.nheads, p.d = (int)a.head_size;
    p.NT = (int)((a.seq_len + 31) / 32);
    p.scale = (float)(1.0 / sqrt((double)a.head_size)); // reference :98
    // A batch row is one workgroup and its three phases follow one another (load and mean, logits, gate and output), so what
    // overlaps them is other rows on the same CU.  With the row kept in registers (up to 1024 positions) four waves hold
    // 128 + 107 registers and two rows share a CU; eight waves hold half the tiles each (171 registers) and one row has the
    // CU to itself, which is faster only while there is no second row to put there -- batch <= CUs: 28.1 against 30.7 us at
    // 256 x 1024, 48.3 against 39.3 us at 384 x 1024.  Longer rows take eight waves with 80 tiles kept.
    const double BS = (double)a.batch * (double)a.seq_len;
    kutacc_prof::KernelTimer t("global_attention_kernel", BS * (4.0 * GC * a.head_size + 4.0 * GC * GC + 4.0 * GC), stream);
    const bool eight_waves = p.NT > 32 || (p.NT >= 16 && a.batch <= kutacc_cu_count());
    // Rows of eight waves that would leave half of the CUs or more without one are shared by up to eight workgroups each: all form the
    // mean and the average, the same bits in each, from one L2, and a part of the result (us, one workgroup a row with 64 tiles kept against this: 5120
    // positions x 384 rows 184 -> 173, x 128 69.1 -> 58.4, x 60 66.0 -> 45.0; 4000 x 300 136 -> 117, 2500 x 100 38.1 -> 30.1, 1024 x 128 19.4 -> 17.3,
    // x 60 18.5 -> 14.6, 700 x 100 15.7 -> 14.2).  Two rows of four waves a CU gain nothing (400 x 200 16.4 -> 17.3).  Not where the result lies over the input: one
    // workgroup would put out what another still reads.
    const int64_t room = kutacc_cu_count(), rest = eight_waves ? a.batch % room : 0;
    const uintptr_t in = reinterpret_cast<uintptr_t>(a.q_data), out = reinterpret_cast<uintptr_t>(a.out);
    const int64_t in_bytes = 2 * ((a.batch - 1) * a.q_data_stride_b + (a.seq_len - 1) * a.q_data_stride_s + GC);
    const int64_t out_bytes = 2 * ((a.batch - 1) * a.out_stride_b + (a.seq_len - 1) * a.out_stride_s + GC);
    const bool apart = a.q_data_stride_b >= 0 && a.out_stride_b >= 0 && (in + (uintptr_t)in_bytes <= out || out + (uintptr_t)out_bytes <= in);
    p.parts = rest > 0 && apart ? (int)std::min<int64_t>(MAX_PARTS, std::max<int64_t>(1, room / rest)) : 1;
    p.whole = (int)(p.parts > 1 ? a.batch - rest : a.batch);
    const hipError_t e = p.NT > 32 ? launch<8, 10, true>(p, stream) : eight_waves ? launch<8, 4, false>(p, stream) : launch<4, 8, false>(p, stream);
    return kutacc_hip_status(e);
}

} // namespace kutacc_launch
