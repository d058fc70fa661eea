// Attention with heads of 8 (the extra-MSA row attention: 64 channels, eight heads) for gfx950: the middle step of the tiled
// route (tiled_attention.hip), reading q, k, v and gate as its projections leave them.
//
// A head of 8 fills little of a matrix product: the 742 M logits of 1024 rows x 301 keys x 8 heads are 24 GFLOP of products, 71 as
// they fill the tiles, 57 us of the matrix cores; their exponentials take 85 us of the vector ALU.  What that does per logit is
// kept to the exponential, half a packed conversion and a fourth of the pair bias's conversion:
//   * logits in log2 units straight from a 16x16x32 MFMA.  q * log2(e)/sqrt(d) has 24 significant bits: three parts of eight, exact,
//     in three of the four chunks of k-slots, against the same keys in each;
//   * the pair bias is the C operand of four batch rows' logits (a wave attends the same 32 queries of four rows at once), with the
//     keys past the end at -inf; masks are added to it in fp32, only in key tiles that have one;
//   * p.v with 16x16x32 MFMAs of 32 keys whose rows are the eight values and ones, which give the sums of the probabilities.
// K, V and masks of a head's four rows lie in the LDS for the whole workgroup (128 bytes per key and 16 of masks).
// Measured on 1024 rows x 301 keys x 8 heads: 505 us on the general attention_tiles_kernel, 177 to 189 us here (vector
// issue 69 %).  With the queries and
// the masks in two parts (16 bits, an error of up to 8 % in a probability at logits of 11 000) and 32x32x16 products it was 199.
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

// slot of key i of a tile of 32: row m of half a of the logits products stands for key 8 (m / 4) + 4 a + m % 4, so that a lane's
// four accumulator rows of both halves are eight consecutive keys, the chunk of p.v's k-slots that the lane supplies
__device__ __forceinline__ int key_slot(int i) { return 16 * ((i >> 2) & 1) + 4 * (i >> 3) + (i & 3); }

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
    // [tile][row][chunk of eight keys][value], a tile of constants (slots 32 i zeros, 32 i + 1 ones), masks in log2 units [tile][row][32]
    uint4 *ks = lds, *vs = lds + ROWS * keys, *constants = vs + ROWS * keys;
    float *masks = reinterpret_cast<float *>(constants + TILE);
    uint32_t *first_masked = reinterpret_cast<uint32_t *>(masks + ROWS * keys);
    for (int idx = tid; idx < TILE; idx += 64 * waves) {
        const uint32_t one = idx % 32 == 1 ? 0x3f803f80u : 0u;
        constants[idx] = make_uint4(one, one, one, one);
    }
    if (tid == 0) {
        *first_masked = (uint32_t)NB;
    }
    __syncthreads();
    // A wave brings 64 keys of one row at a time, the next ones requested before these are stored: of K and the mask a key a lane, of V
    // eight keys of one value.  (Keys dealt to threads by division, K and V in loops of their own, one round trip after the other: whole
    // operator 2000 rows of 384 660 us, 627 so, of 170 206 and 200.)
    struct Piece {
        uint4 k, v;
        bf16_t mask;
    };
    const int units = ROWS * ((NB + 1) / 2); // row unit % 4, keys 64 (unit / 4) ..
    const bf16_t *v_lane = p.v + (int64_t)(h * D + (lane >> 3)) * p.v_se;
    auto fetch = [&](int unit) {
        const int64_t pos = (int64_t)row_of(unit & 3) * S;
        const int key0 = 64 * (unit >> 2), key = min(key0 + lane, S - 1);
        Piece w;
        w.k = *reinterpret_cast<const uint4 *>(p.k + pos * p.k_ss + h * D + (uint32_t)key * (uint32_t)p.k_ss);
        w.mask = (p.bias + (int64_t)row_of(unit & 3) * p.bias_sb)[(uint32_t)key];
        w.v = load8_checked(v_lane + pos, min(key0 + 8 * (lane & 7), S), S);
        return w;
    };
    Piece piece = fetch(min(wave, units - 1));
    for (int unit = wave; unit < units; unit += waves) {
        const Piece w = piece;
        piece = fetch(min(unit + waves, units - 1));
        const int i = unit & 3, key = 64 * (unit >> 2) + lane;
        const float mask = key < S ? to_f32(w.mask) * LOG2E : 0.f;
        if (key < keys) {
            const int tile_row = (key >> 5) * TILE + i * 32;
            ks[tile_row + key_slot(key & 31)] = key < S ? w.k : zero_u4();
            masks[tile_row + (key & 31)] = mask;
        }
        const int kp = 8 * (unit >> 2) + (lane & 7);
        if (8 * kp < keys) {
            vs[(kp >> 2) * TILE + i * 32 + (kp & 3) * 8 + (lane >> 3)] = w.v;
        }
        if (mask != 0.f) {
            atomicMin(first_masked, (uint32_t)(key >> 5));
        }
    }
    __syncthreads();
    const int masked_from = (int)*first_masked;

    // Operands of the 16x16x32 MFMA: lane (row or column n, chunk c of eight k-slots).
    //   logits: rows are sixteen keys, columns sixteen queries; chunks 0, 1, 2 hold the same keys against the three parts of the
    //           queries, chunk 3 nothing (zeros in the queries);
    //   p.v:    rows 0-7 are the values, row 8 ones (the row sums), the rest zeros; the k-slots of chunk c are keys 8 c .. 8 c + 7.
    const int n = lane & 15, c = lane >> 4;
    const uint32_t v_first = n < D ? 8u * c + n : (uint32_t)(constants - vs) + (n == D ? 1u : 0u), v_tile = n < D ? (uint32_t)TILE : 0u;
    auto product = [](bf16x8 a, bf16x8 b, f32x4 x) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, x, 0, 0, 0); };

    for (int j = split * waves + wave; j < NB; j += waves * p.splits) {
        int lv = lane; // opaque: the addresses of a query block's rows are formed where they are used, not kept over the keys
        asm volatile("" : "+v"(lv));
        bf16x8 q[ROWS][2]; // queries 32 j + 16 u + n
        uint32_t query[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            query[u] = (uint32_t)min(32 * j + 16 * u + (lv & 15), S - 1);
        }
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                // a lane splits dims 2 c and 2 c + 1 of its query, then the four lanes of the query exchange: parts for dims
                const uint32_t raw = *reinterpret_cast<const uint32_t *>(p.q + (int64_t)row_of(i) * S * p.q_ss + h * D +
                                                                         (query[u] * (uint32_t)p.q_ss + 2u * (uint32_t)(lv >> 4)));
                uint32_t part[4] = {0u, 0u, 0u, 0u};
                float x0 = __uint_as_float(raw << 16) * p.scale2, x1 = __uint_as_float(raw & 0xffff0000u) * p.scale2;
#pragma unroll
                for (int w = 0; w < 3; ++w) {
                    part[w] = __builtin_amdgcn_perm(__float_as_uint(x1), __float_as_uint(x0), 0x07060302u); // the upper halves
                    x0 -= __uint_as_float(__float_as_uint(x0) & 0xffff0000u), x1 -= __uint_as_float(__float_as_uint(x1) & 0xffff0000u);
                }
                q[i][u] = as_bf16x8(transpose4x4_lanes(part));
            }
        }
        const bf16_t *nb_head = HAS_NB ? p.nb + (int64_t)h * p.nb_sh : nullptr;
        uint32_t nb_row[2] = {0u, 0u}; // elements, within 2^30 (the launcher checks)
#pragma unroll
        for (int u = 0; HAS_NB && u < 2; ++u) {
            nb_row[u] = query[u] * (uint32_t)p.nb_sq;
        }
        struct Raw {
            uint4 r[2]; // keys 8 c .. 8 c + 7 of this lane's two queries
        };
        // eight keys of a row of the bias, the row's last eight where it ends before them (and rows of fewer than eight are not read here)
        auto load_nb = [&](int t) {
            Raw w = {zero_u4(), zero_u4()};
            if constexpr (HAS_NB) {
                const int key = min(32 * t + 8 * c, S - 8);
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    w.r[u] = load8_any(nb_head, nb_row[u] + (uint32_t)key);
                }
            }
            return w;
        };
        auto load_tail = [&] { // of the last tile, where it has fewer than 32 keys; keys past the end zero
            Raw w = {zero_u4(), zero_u4()};
            if constexpr (HAS_NB) {
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    w.r[u] = load8_checked(nb_head + nb_row[u], 32 * (NB - 1) + 8 * c, S);
                }
            }
            return w;
        };
        struct Tile {
            f32x4 x[2][2]; // [query half][key half]
        };
        auto seeds = [&](const Raw &w, auto tail) { // of the four rows' logits: the pair bias, -inf past the last key
            Tile s;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const bf16x8 raw = as_bf16x8(w.r[u]);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    s.x[u][e >> 2][e & 3] = HAS_NB ? to_f32(raw[e]) * LOG2E : 0.f;
                }
            }
            if constexpr (decltype(tail)::value) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    if (32 * (NB - 1) + 8 * c + e >= S) {
                        s.x[0][e >> 2][e & 3] = s.x[1][e >> 2][e & 3] = -INFINITY;
                    }
                }
            }
            return s;
        };
        auto logits = [&](int i, int t, const Tile &C, auto masked) { // of row i, tile t
            Tile l;
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                const bf16x8 k = as_bf16x8(ks[t * TILE + i * 32 + a * 16 + n]);
                f32x4 c0 = C.x[0][a], c1 = C.x[1][a];
                if constexpr (decltype(masked)::value) {
                    const f32x4 m = *reinterpret_cast<const f32x4 *>(masks + t * TILE + i * 32 + 8 * c + 4 * a);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        c0[e] += m[e], c1[e] += m[e];
                    }
                }
                l.x[0][a] = product(k, q[i][0], c0);
                l.x[1][a] = product(k, q[i][1], c1);
            }
            return l;
        };
        // rows 0-7: the values' sums, in lanes of chunks 0 and 1; row 8: the sums of the probabilities, in lanes of chunk 2
        f32x4 o[ROWS][2];
        auto clear = [&](int i) { o[i][0] = o[i][1] = f32x4{0.f, 0.f, 0.f, 0.f}; };
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            clear(i);
        }
        auto finish = [&](int i, int t, const Tile &l, const float (&shift)[2], auto shifted) { // softmax and p.v of row i, tile t
            const bf16x8 v = as_bf16x8(vs[v_first + t * v_tile + i * 32]);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                bf16x8 pr;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float x = l.x[u][e >> 2][e & 3];
                    pr[e] = (bf16_t)__builtin_amdgcn_exp2f(decltype(shifted)::value ? x - shift[u] : x);
                }
                o[i][u] = product(v, pr, o[i][u]);
            }
        };
        const float unshifted[2] = {0.f, 0.f};
        // Two rows in flight: the logits of one are in the matrix pipe while the other's exponentials run.  The fences keep
        // it at two: left to itself the compiler starts all four and needs registers for two waves per SIMD only.
        auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
        auto rows = [&](int t, const Tile &C, auto masked) __attribute__((always_inline)) {
            Tile xa = logits(0, t, C, masked);
            fence();
            Tile xb = logits(1, t, C, masked);
            finish(0, t, xa, unshifted, std::false_type{});
            fence();
            xa = logits(2, t, C, masked);
            finish(1, t, xb, unshifted, std::false_type{});
            fence();
            xb = logits(3, t, C, masked);
            finish(2, t, xa, unshifted, std::false_type{});
            fence();
            finish(3, t, xb, unshifted, std::false_type{});
            fence();
        };
        // Tiles without a mask, tiles with one, and the ragged last one, each in a loop of its own: with their choice inside one loop
        // a tile cost 76 vector instructions and 16 moves of register pairs more than the 160 that it needs (the whole operator, us: 1024
        // rows of 301 237 -> 221, 1000 of 420 432 -> 381).
        const int full = S >> 5, plain = min(masked_from, full);
        Raw raw = {zero_u4(), zero_u4()};
        if (S >= 8) {
            raw = load_nb(0);
        }
        auto run = [&](int from, int to, auto masked) __attribute__((always_inline)) {
            for (int t = from; t < to; ++t) {
                const Tile C = seeds(raw, std::false_type{});
                raw = load_nb(t + 1);
                rows(t, C, masked);
            }
        };
        run(0, plain, std::false_type{});
        run(plain, full, std::true_type{});
        if (full < NB) {
            if constexpr (HAS_NB) {
                if (S >= 8) {
                    const int drop = min(max(32 * full + 8 * c - (S - 8), 0), 8);
                    raw.r[0] = drop_first(raw.r[0], drop), raw.r[1] = drop_first(raw.r[1], drop);
                } else {
                    raw = load_tail();
                }
            }
            rows(full, seeds(raw, std::true_type{}), std::true_type{});
        }
        // the two query halves side by side: lane l then has values 4 (l / 16 % 2) .. + 3 of query 16 (l / 32) + l % 16
        int le = lane;
        asm volatile("" : "+v"(le));
        const int pos = 32 * j + 16 * (le >> 5) + (le & 15);
        const uint32_t d0 = 4 * ((le >> 4) & 1), gate_at = (uint32_t)min(pos, S - 1) * (uint32_t)p.g_ss + d0, avg_at = (uint32_t)pos * (uint32_t)p.a_ss + d0;
        bf16x4 gates[ROWS]; // of all rows at once, one round trip (2000 rows of 384 627 -> 622 us, of 170 200 -> 195)
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            gates[i] = *reinterpret_cast<const bf16x4 *>(p.gate + (int64_t)row_of(i) * S * p.g_ss + h * D + gate_at);
        }
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            f32x4 values;
            float l;
            auto collect = [&] {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(o[i][0][e]), __float_as_uint(o[i][1][e]), false, false);
                    values[e] = __uint_as_float(sw[0]);
                    if (e == 0) {
                        l = __shfl(__uint_as_float(sw[1]), le & 47, 64);
                    }
                }
            };
            collect();
            if (__any(!(l > 1e-30f && l < 1e30f))) {
                // Some probability overflowed or a whole row underflowed (every key masked: -1e9 log2(e) everywhere, which is
                // finite): the row's true maxima first, then the probabilities with them subtracted.
                auto again = [&](int t) { return logits(i, t, t < full ? seeds(load_nb(t), std::false_type{}) : seeds(load_tail(), std::true_type{}), std::true_type{}); };
                float mx[2] = {-INFINITY, -INFINITY};
                for (int t = 0; t < NB; ++t) {
                    const Tile x = again(t);
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        mx[e >> 3] = fmaxf(mx[e >> 3], x.x[e >> 3][(e >> 2) & 1][e & 3]);
                    }
                }
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    mx[u] = half_swap_max(mx[u]);
                    mx[u] = fmaxf(mx[u], __shfl_xor(mx[u], 16, 64));
                    mx[u] = mx[u] == -INFINITY ? 0.f : mx[u];
                }
                clear(i);
                for (int t = 0; t < NB; ++t) {
                    finish(i, t, again(t), mx, std::true_type{});
                }
                collect();
            }
            const float inv = reciprocal(l);
            if (pos < S && b0 + i < p.B) {
                float gate[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    gate[e] = to_f32(gates[i][e]);
                }
                sigmoids_f32(gate);
                bf16x4 ov;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float wavg = to_f32((bf16_t)(values[e] * inv));
                    ov[e] = (bf16_t)(wavg * gate[e]);
                }
                *reinterpret_cast<bf16x4 *>(p.avg + (int64_t)(b0 + i) * S * p.a_ss + h * D + avg_at) = ov;
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
    const auto in_reach = [&](int64_t stride) { return stride >= 0 && stride < (1 << 30) && a.seq_len * stride < (1 << 30); }; // of 32-bit byte offsets
    const int64_t NB = (a.seq_len + 31) / 32, sets = (a.batch + ROWS - 1) / ROWS;
    return a.head_size == D && NB <= 64 && lds_bytes((int)NB) <= (size_t)kutacc_device_attribute(hipDeviceAttributeMaxSharedMemoryPerBlock, 64 * 1024, table) &&
           in_reach(a.nb_stride_q) && in_reach(a.q_stride_s) && in_reach(a.k_stride_s) && in_reach(a.gate_stride_s) && in_reach(a.avg_stride_s) && (sets + 7) * a.nheads * 8 <= INT32_MAX;
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
