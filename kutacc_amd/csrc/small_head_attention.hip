// Attention with heads of 8 (the extra-MSA row attention: 64 channels, eight heads) for gfx950: the middle step of the tiled
// route (tiled_attention.hip), reading q, k, v and gate as its projections leave them.
//
// A head of 8 leaves the matrix cores a quarter of a product's rows: 33 M logits take 4 % of a GFLOP and the exponential
// decides.  What the vector ALU does per logit is therefore kept to that exponential, half a packed conversion and a fourth
// of the pair bias's conversion:
//   * logits in log2 units straight from the MFMA.  q * log2(e)/sqrt(d) needs more than the eight bits of a bf16 operand to
//     keep the reference's product of bf16 q and k: the unused half of the 16 k-slots carries the rest, q = hi + lo
//     against the same keys, exact to 2^-17;
//   * the pair bias is the C operand of four batch rows' logits (a wave attends the same 32 queries of four rows at once);
//   * a row's mask is one more MFMA, only for key tiles that have one; ragged ends are keys at -inf;
//   * p.v with 16x16x32 MFMAs whose sixteen rows are the eight values of queries n and of queries n + 16 (the probability
//     fragment of the 32-query layout holds both): half the matrix-pipe time of the 32x32 form and four registers
//     instead of sixteen; row sums likewise (rowsum_selector).
// K, V and masks of a head's four rows lie in the LDS for the whole workgroup (128 bytes per key and 16 of mask words).
// Measured on 1024 rows x 301 keys x 8 heads: 505 us on the general attention_tiles_kernel, 200 us here (exponentials alone: 85).
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>

#include "attention_util.h"
#include "launch_internal.h"
#include "mfma_tiles.h"
#include "profiler.h"

namespace {
using namespace kutacc_dev;

constexpr int CU_LDS_BYTES = 160 * 1024;
constexpr int D = 8, ROWS = 4, TILE = ROWS * 32; // slots of a key tile's rows

struct SmallHeadParams {
    const bf16_t *q, *k, *v, *gate, *bias, *nb;
    bf16_t *avg;
    int64_t q_ss, k_ss, g_ss, a_ss; // rows of the [batch * seq, channels] matrices
    int64_t v_se, bias_sb, nb_sh, nb_sq;
    int B, S, H, NB, sets, splits; // blocks of 32 positions, sets of four rows, workgroups that share a set's queries
    float scale2;                  // log2(e) / sqrt(8)
};

// slot of key i of a tile of 32: accumulator row r of the logits stands for key pi(r), so that a lane holds 16 consecutive keys
__device__ __forceinline__ int key_slot(int i) { return (i & 3) | (((i >> 4) & 1) << 2) | (((i >> 2) & 3) << 3); }

template <bool HAS_NB>
__global__ __launch_bounds__(512, 3) void small_head_attention_kernel(const SmallHeadParams p)
{
    extern __shared__ uint4 lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = (int)blockDim.x >> 6;
    const int S = p.S, NB = p.NB, keys = 32 * NB;
    // Workgroup ids are dealt round robin over the 8 XCDs: a set's heads, whose q, k, gate and avg share cache lines, and its
    // query parts follow each other on one XCD.
    const int per_set = p.H * p.splits, local = (int)(blockIdx.x >> 3);
    const int set = (int)(blockIdx.x & 7) + 8 * (local / per_set), h = local % per_set / p.splits, split = local % p.splits;
    if (set >= p.sets) {
        return;
    }
    const int b0 = set * ROWS;
    auto row_of = [&](int i) { return min(b0 + i, p.B - 1); }; // past the last row: that one again

    // LDS, a tile's four rows together so that a lane's one offset serves them all: K [tile][row][32] (in key_slot order), V
    // [tile][row][k-step][half][value], a tile of zeros, mask words [tile][row][32]
    uint4 *ks = lds, *vs = lds + ROWS * keys, *zeros = vs + ROWS * keys;
    uint32_t *words = reinterpret_cast<uint32_t *>(zeros + TILE), *first_masked = words + ROWS * keys;
    for (int idx = tid; idx < TILE; idx += 64 * waves) {
        zeros[idx] = zero_u4();
    }
    if (tid == 0) {
        *first_masked = (uint32_t)NB;
    }
    __syncthreads();
    for (int idx = tid; idx < ROWS * keys; idx += 64 * waves) {
        const int i = idx / keys, key = idx % keys, b = row_of(i);
        const int64_t pos = (int64_t)b * S + min(key, S - 1);
        const uint4 kv = *reinterpret_cast<const uint4 *>(p.k + pos * p.k_ss + h * D);
        const int slot = (key >> 5) * TILE + i * 32 + key_slot(key & 31);
        ks[slot] = key < S ? kv : zero_u4();
        const float mv = key < S ? to_f32(p.bias[(int64_t)b * p.bias_sb + key]) * LOG2E : -INFINITY;
        words[slot] = mask_word(mv);
        if (mv != 0.f) {
            atomicMin(first_masked, (uint32_t)(key >> 5));
        }
    }
    for (int idx = tid; idx < ROWS * keys; idx += 64 * waves) { // eight keys of one value: as many pieces as keys
        const int i = idx / keys, rest = idx % keys, d = rest / (keys >> 3), kp = rest % (keys >> 3), key = 8 * kp;
        uint4 vv = zero_u4();
        if (key < S) {
            vv = load8_checked(p.v + (int64_t)(h * D + d) * p.v_se + (int64_t)row_of(i) * S, key, S);
        }
        vs[(kp >> 2) * TILE + i * 32 + ((kp & 1) * 2 + ((kp >> 1) & 1)) * 8 + d] = vv;
    }
    __syncthreads();
    const int masked_from = (int)*first_masked;

    const int r = lane & 31, g = lane >> 5;
    const uint32_t lower = lane < 32 ? 0xffffffffu : 0u;
    const bf16x8 onesf = as_bf16x8(make_uint4(0x3f803f80u & lower, 0u, 0u, 0u)), ones_rows = rowsum_selector(lane);
    // V operand of the 16x16x32 MFMA: lane (row i, chunk c) of the 64; rows 0-7 are the values for queries n, which chunks 0
    // and 2 of the probabilities belong to, rows 8-15 those for queries n + 16 (chunks 1 and 3); elsewhere zeros
    const int vi = lane & 15, vc = lane >> 4;
    const bool v_real = (vi >> 3) == (vc & 1);
    const uint32_t v_first = v_real ? 8u * (vc >> 1) + (vi & 7) : (uint32_t)(zeros - vs), v_tile = v_real ? (uint32_t)TILE : 0u;

    for (int j = split * waves + wave; j < NB; j += waves * p.splits) {
        int lv = lane; // opaque: the addresses of a query block's rows are formed where they are used, not kept over the keys
        asm volatile("" : "+v"(lv));
        const int query = min(32 * j + (lv & 31), S - 1);
        bf16x8 q[ROWS];
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            const bf16x8 raw = *reinterpret_cast<const bf16x8 *>(p.q + ((int64_t)row_of(i) * S + query) * p.q_ss + h * D);
#pragma unroll
            for (int e = 0; e < D; ++e) {
                const float x = to_f32(raw[e]) * p.scale2;
                const bf16_t hi = (bf16_t)x;
                q[i][e] = g == 0 ? hi : (bf16_t)(x - to_f32(hi));
            }
        }
        const bf16_t *nb_head = HAS_NB ? p.nb + (int64_t)h * p.nb_sh : nullptr;
        const uint32_t nb_row = HAS_NB ? (uint32_t)query * (uint32_t)p.nb_sq : 0u; // elements, within 2^30 (the launcher checks)
        struct Raw {
            uint4 lo, hi; // 16 consecutive keys of this lane's query
        };
        auto load_nb = [&](int t) {
            Raw w = {zero_u4(), zero_u4()};
            if constexpr (HAS_NB) {
                const int key = 32 * min(t, NB - 1) + 16 * g;
                if (32 * t + 32 <= S) {
                    w.lo = load8_any(nb_head, nb_row + key), w.hi = load8_any(nb_head, nb_row + key + 8);
                } else {
                    w.lo = load8_checked(nb_head + nb_row, key, S), w.hi = load8_checked(nb_head + nb_row, key + 8, S);
                }
            }
            return w;
        };
        auto convert_nb = [&](const Raw &w) {
            f32x16 c = zero16();
            if constexpr (HAS_NB) {
                const bf16x8 lo = as_bf16x8(w.lo), hi = as_bf16x8(w.hi);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    c[e] = to_f32(lo[e]) * LOG2E, c[8 + e] = to_f32(hi[e]) * LOG2E;
                }
            }
            return c;
        };
        auto logits = [&](int i, int t, const f32x16 &C) { // of row i, tile t, without the mask
            return mfma(as_bf16x8(ks[t * TILE + i * 32 + r]), q[i], C);
        };
        auto add_mask = [&](int i, int t, f32x16 x) {
            return mfma(as_bf16x8(make_uint4(words[t * TILE + i * 32 + r] & lower, 0u, 0u, 0u)), onesf, x);
        };
        f32x4 o[ROWS], sums[ROWS];
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            o[i] = sums[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        auto values = [&](int i, int t, int s) { return as_bf16x8(vs[v_first + t * v_tile + i * 32 + s * 16]); };
        auto finish = [&](int i, int t, f32x16 &x, float shift, auto shifted) { // softmax and p.v of row i, tile t
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                x[e] = __builtin_amdgcn_exp2f(decltype(shifted)::value ? x[e] - shift : x[e]);
            }
            const bf16x8 p0 = pack8(x, 0), p1 = pack8(x, 8);
            o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(values(i, t, 0), p0, o[i], 0, 0, 0);
            sums[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones_rows, p0, sums[i], 0, 0, 0);
            o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(values(i, t, 1), p1, o[i], 0, 0, 0);
            sums[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones_rows, p1, sums[i], 0, 0, 0);
        };
        Raw raw = load_nb(0);
        for (int t = 0; t < NB; ++t) {
            const f32x16 C = convert_nb(raw);
            if (t + 1 < NB) {
                raw = load_nb(t + 1);
            }
            // Two rows in flight: the logits of one are in the matrix pipe while the other's exponentials run.  The fences keep
            // it at two: left to itself the compiler starts all four and needs 235 registers, two waves per SIMD.
            auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
            auto rows = [&](auto masked) {
                auto next = [&](int i) {
                    const f32x16 x = logits(i, t, C);
                    return decltype(masked)::value ? add_mask(i, t, x) : x;
                };
                f32x16 xa = next(0);
                fence();
                f32x16 xb = next(1);
                finish(0, t, xa, 0.f, std::false_type{});
                fence();
                xa = next(2);
                finish(1, t, xb, 0.f, std::false_type{});
                fence();
                xb = next(3);
                finish(2, t, xa, 0.f, std::false_type{});
                fence();
                finish(3, t, xb, 0.f, std::false_type{});
                fence();
            };
            if (t < masked_from) {
                rows(std::false_type{});
            } else {
                rows(std::true_type{});
            }
        }
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            float l = rowsum_fetch(sums[i], lane);
            if (__any(!(l > 1e-30f && l < 1e30f))) {
                // Some probability overflowed or a whole row underflowed (every key masked: -1e9 log2(e) everywhere, which is
                // finite): the row's true maxima first, then the probabilities with them subtracted.
                float mx = -INFINITY;
                for (int t = 0; t < NB; ++t) {
                    const f32x16 x = add_mask(i, t, logits(i, t, convert_nb(load_nb(t))));
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        mx = fmaxf(mx, x[e]);
                    }
                }
                mx = half_swap_max(mx);
                mx = mx == -INFINITY ? 0.f : mx;
                o[i] = sums[i] = f32x4{0.f, 0.f, 0.f, 0.f};
                for (int t = 0; t < NB; ++t) {
                    f32x16 x = add_mask(i, t, logits(i, t, convert_nb(load_nb(t))));
                    finish(i, t, x, mx, std::true_type{});
                }
                l = rowsum_fetch(sums[i], lane);
            }
            // o: lane (column n, group c) holds values 4 (c & 1) .. + 3 of query n + 16 (c >> 1); its sum lies in the lane of
            // that query
            int le = lane;
            asm volatile("" : "+v"(le));
            const int qi = (le & 15) + 16 * (le >> 5), pos = 32 * j + qi, d0 = 4 * ((le >> 4) & 1);
            const float inv = 1.0f / __shfl(l, qi, 64);
            if (pos < S && b0 + i < p.B) {
                const int64_t row = (int64_t)(b0 + i) * S + pos;
                const bf16x4 gv = *reinterpret_cast<const bf16x4 *>(p.gate + row * p.g_ss + h * D + d0);
                bf16x4 ov;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const float wavg = to_f32((bf16_t)(o[i][c] * inv));
                    ov[c] = (bf16_t)(wavg * sigmoid_f32(to_f32(gv[c])));
                }
                *reinterpret_cast<bf16x4 *>(p.avg + row * p.a_ss + h * D + d0) = ov;
            }
        }
    }
}

size_t lds_bytes(int NB) { return (size_t)(2 * NB + 1) * TILE * 16 + (size_t)(TILE * NB + 1) * 4; }

template <bool HAS_NB>
int launch(SmallHeadParams p, hipStream_t stream)
{
    static size_t configured[KUTACC_DEVICE_SLOTS] = {};
    const size_t lds = lds_bytes(p.NB);
    if (const hipError_t e = kutacc_opt_in_lds(reinterpret_cast<const void *>(&small_head_attention_kernel<HAS_NB>), lds, configured)) {
        return kutacc_hip_status(e);
    }
    // Four waves while three workgroups' keys fit a CU (the registers' limit of 12 waves), else eight.  A number that is no
    // multiple of four leaves SIMDs without their share: 1024 rows of 301 took 288 us at five waves, 240 at eight, 200 at four.
    const int waves = std::min(p.NB, 3 * lds <= (size_t)CU_LDS_BYTES ? 4 : 8);
    // a set's queries are dealt to several workgroups, each staging the keys again, only while the chip has room for them
    const int turns = (p.NB + waves - 1) / waves, room = 2 * kutacc_cu_count() / std::max(1, p.sets * p.H);
    p.splits = std::max(1, std::min(turns, room));
    const int64_t blocks = (int64_t)(p.sets + 7) / 8 * 8 * p.H * p.splits;
    small_head_attention_kernel<HAS_NB><<<dim3((unsigned)blocks), 64 * waves, lds, stream>>>(p);
    return kutacc_hip_status(hipGetLastError());
}
} // namespace

namespace kutacc_launch {

bool small_head_attention_supports(const kutacc_hip_attention_args_t &a)
{
    static int table[KUTACC_DEVICE_SLOTS] = {};
    const int64_t NB = (a.seq_len + 31) / 32, sets = (a.batch + ROWS - 1) / ROWS;
    return a.head_size == D && NB <= 64 && lds_bytes((int)NB) <= (size_t)kutacc_device_attribute(hipDeviceAttributeMaxSharedMemoryPerBlock, 64 * 1024, table) &&
           a.nb_stride_q >= 0 && a.seq_len * a.nb_stride_q < (1 << 30) && (sets + 7) * a.nheads * 8 <= INT32_MAX;
}

int small_head_attention(const kutacc_hip_attention_args_t &a, hipStream_t stream)
{
    SmallHeadParams p;
    p.q = (const bf16_t *)a.q, p.k = (const bf16_t *)a.k, p.v = (const bf16_t *)a.v, p.gate = (const bf16_t *)a.gate;
    p.bias = (const bf16_t *)a.bias, p.nb = (const bf16_t *)a.nonbatched_bias, p.avg = (bf16_t *)a.avg;
    p.q_ss = a.q_stride_s, p.k_ss = a.k_stride_s, p.g_ss = a.gate_stride_s, p.a_ss = a.avg_stride_s;
    p.v_se = a.v_stride_e, p.bias_sb = a.bias_stride_b, p.nb_sh = a.nb_stride_h, p.nb_sq = a.nb_stride_q;
    p.B = (int)a.batch, p.S = (int)a.seq_len, p.H = (int)a.nheads, p.NB = (p.S + 31) / 32, p.sets = (p.B + ROWS - 1) / ROWS, p.splits = 1;
    // (float)(1 / sqrt(head_size)) as the reference forms it (gating_attention.cpp:68)
    p.scale2 = (float)(1.0 / sqrt((double)D)) * LOG2E;
    return p.nb ? launch<true>(p, stream) : launch<false>(p, stream);
}

} // namespace kutacc_launch
