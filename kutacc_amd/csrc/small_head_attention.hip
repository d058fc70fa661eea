// Attention with heads of 8 (the extra-MSA row attention: 64 channels, eight heads) for gfx950: the middle step of the tiled
// route (tiled_attention.hip), reading q, k, v and gate as its projections leave them, or forming them itself (64 channels).
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
// Measured on 1024 rows x 301 keys x 8 heads: 505 us on the general attention_tiles_kernel, 177 to 189 us here behind a pass that
// projects, 168 to 204 from card to card with the projections inside (vector issue 73 %), 4 to 8 % less of them with the bias's rows, which start on any
// address, brought into the lanes' order by a pass of its own (seed_tiles_kernel).  With the queries and the masks in two parts (16 bits, an error of up to 8 % in a probability at logits of 11 000) and 32x32x16 products it was 199.
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
constexpr int PROJECTED = 64; // channels of the calls whose projections are formed here
constexpr int D = 8, ROWS = 4, TILE = ROWS * 32; // slots of a key tile's rows

struct SmallHeadParams {
    const bf16_t *q, *k, *v, *gate, *bias, *nb;
    bf16_t *avg;
    // ... and its queries and gates: of a set and head [row][tile][queries, gates][64 lanes] of 8 bytes, in one of three of the scratch tensors
    uint2 *stash[3];
    f32x4 *tiles;   // pair bias, where it has been put in the logits' order (seed_tiles_kernel): [head][query block][key tile][4][64 lanes]
    const bf16_t *x, *wq, *wk, *wv, *wg; // the kernel that projects: input rows of 64 channels, weights
    const float *bg;
    int64_t x_ss;
    int64_t q_ss, k_ss, g_ss, a_ss; // rows of the [batch * seq, channels] matrices
    int64_t v_se, bias_sb, nb_sh, nb_sq;
    int B, S, H, NB, sets, splits; // blocks of 32 positions, sets of four rows, workgroups that share a set's queries
    float scale2;                  // log2(e) / sqrt(8)
    int stash_each;                // sets and heads per tensor of the stash
};
// The size of a workgroup, which the kernel reads, comes 12 bytes behind these: in a fifth line of arguments a call waits 0.2 to 0.3 us longer (whole operator,
// us: 64 x 77 14.5 14.1, 600 x 77 30.15 29.9, 1000 x 63 30.7 30.4).
static_assert(sizeof(SmallHeadParams) <= 240, "four lines with the size of the launch");

// slot of key i of a tile of 32: row m of half a of the logits products stands for key 8 (m / 4) + 4 a + m % 4, so that a lane's
// four accumulator rows of both halves are eight consecutive keys, the chunk of p.v's k-slots that the lane supplies
__device__ __forceinline__ int key_slot(int i) { return 16 * ((i >> 2) & 1) + 4 * (i >> 3) + (i & 3); }

// The seeds of the logits of all batch rows: the pair bias in log2 units, -inf past the last key, tile by tile as the lanes hold them,
// pieces 2 u + a of query half u and key half a.  5 us with the launch; 4 KB a tile instead of 2 in the attention's loop, but whole lines and no
// conversion (a seventh of its vector instructions).
__global__ __launch_bounds__(256) void seed_tiles_kernel(const SmallHeadParams p)
{
    const int lane = threadIdx.x & 63, n = lane & 15, c = lane >> 4;
    const int tile = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6), t = tile % p.NB, j = tile / p.NB % p.NB, h = tile / (p.NB * p.NB);
    if (h >= p.H) {
        return;
    }
    f32x4 *to = p.tiles + (int64_t)tile * 256 + lane;
    const int key0 = 32 * t + 8 * c;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int query = min(32 * j + 16 * u + n, p.S - 1);
        const bf16x8 raw = as_bf16x8(load8_checked(p.nb + (int64_t)h * p.nb_sh + (uint32_t)query * (uint32_t)p.nb_sq, min(key0, p.S), p.S));
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = key0 + 4 * a + e < p.S ? finite_bias(to_f32(raw[4 * a + e]) * LOG2E) : -INFINITY;
            }
            to[(2 * u + a) * 64] = v;
        }
    }
}

template <bool HAS_NB, bool PROJECTS, bool TILES>
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
    // Operands of the 16x16x32 MFMA: lane (row or column n, chunk c of eight k-slots); results: lane (column n, rows 4 c .. 4 c + 3).
    const int n = lane & 15, c = lane >> 4;
    const int unit_of_stash = set * p.H + h;
    uint2 *const stash = PROJECTS ? p.stash[unit_of_stash / p.stash_each] + (int64_t)(unit_of_stash % p.stash_each) * ROWS * NB * 128 : nullptr;
    auto product = [](bf16x8 a, bf16x8 b, f32x4 x) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, x, 0, 0, 0); };
    if constexpr (PROJECTS) {
        // The head's four projections from the input rows, 16 features as they fill a product.  Keys and values go to the LDS: the
        // keys from rows of a product, so that a lane has four dims of a position, the values from the columns of the product the other
        // way round, so that it has four positions of a value.  Queries and gates wait in memory, as the lanes that use them hold
        // them (1 KB a row and tile in two stores; four bytes a lane in the layout of q and gate cost 25 us of 209): rows 4 c, 4 c + 1 of a third
        // product are the queries' dims 2 c, 2 c + 1, rows 4 c + 2, 4 c + 3 the gates' dims 2 d, 2 d + 1, d being c with its two bits exchanged, which an
        // exchange of the halves of the wave turns into the order of the average.
        // A wave takes the tiles whose queries it attends later, all four rows of them, a row's inputs of the next tile requested where those
        // of this one have left their registers.  They are read in whole lines and cross the lanes in the place of the tile's
        // values, which are written when all four rows have passed: read as the products want them, 16 bytes from each of 16 lines side
        // by side, they kept the address unit busy for three quarters of the kernel (whole operator, us: 1024 rows of
        // 301 181 -> 173, 3576 of 107 175 -> 154, 5120 of 128 281 -> 246).
        auto load_piece = [&](int i, int tile, int q) { // positions 8 q + lane / 8 of a tile of 32, channels 8 (lane % 8) .. + 7
            const uint32_t at = (uint32_t)min(32 * tile + 8 * q + (lane >> 3), S - 1) * (uint32_t)p.x_ss + 8u * (lane & 7);
            return *reinterpret_cast<const uint4 *>(p.x + (int64_t)row_of(i) * S * p.x_ss + at);
        };
        auto load_mask = [&](int i, int tile) { return (p.bias + (int64_t)row_of(i) * p.bias_sb)[(uint32_t)min(32 * tile + (lane & 31), S - 1)]; };
        uint4 in[ROWS][4];
        bf16_t mask_in[ROWS];
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                in[i][q] = load_piece(i, min(wave, NB - 1), q);
            }
            mask_in[i] = load_mask(i, min(wave, NB - 1));
        }
        bf16x8 kv[2], qg[2];
        {
            const int pair = n >> 2, dim = 2 * ((n & 2) == 0 ? pair : 2 * (pair & 1) + (pair >> 1)) + (n & 1);
            const bf16_t *from_kv = n < D ? p.wk + (h * D + n) * PROJECTED : p.wv + (h * D + n - D) * PROJECTED;
            const bf16_t *from_qg = ((n & 2) == 0 ? p.wq : p.wg) + (h * D + dim) * PROJECTED;
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                kv[ks] = as_bf16x8(*reinterpret_cast<const uint4 *>(from_kv + 32 * ks + 8 * c));
                qg[ks] = as_bf16x8(*reinterpret_cast<const uint4 *>(from_qg + 32 * ks + 8 * c));
            }
        }
        const int gate_pair = 2 * (c & 1) + (c >> 1);
        const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f}, gate_bias = {0.f, 0.f, p.bg[h * D + 2 * gate_pair], p.bg[h * D + 2 * gate_pair + 1]};
        for (int t = wave; t < NB; t += waves) {
            uint4 *const k_tile = ks + t * TILE, *const v_tile = vs + t * TILE;
            bf16x4 v4[ROWS][2];
#pragma unroll
            for (int i = 0; i < ROWS; ++i) {
                uint32_t q2[2], g2[2];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    // 128 slots for 16 positions, the pieces of 8 positions in other banks each
                    v_tile[(lane >> 3) * 8 + ((lane ^ (lane >> 3)) & 7)] = in[i][2 * u];
                    v_tile[64 + (lane >> 3) * 8 + ((lane ^ (lane >> 3)) & 7)] = in[i][2 * u + 1];
                    f32x4 kk = zero4, vv = zero4, qq = gate_bias;
#pragma unroll
                    for (int ks = 0; ks < 2; ++ks) {
                        const bf16x8 x = as_bf16x8(v_tile[n * 8 + ((4 * ks + c) ^ (n & 7))]);
                        kk = product(kv[ks], x, kk);
                        vv = product(x, kv[ks], vv);
                        qq = product(qg[ks], x, qq);
                    }
                    bf16x4 k4;
#pragma unroll
                    for (int e = 0; e < 4; ++e) { // zeros past the last key
                        k4[e] = (bf16_t)(32 * t + 16 * u + n < S ? kk[e] : 0.f);
                        v4[i][u][e] = (bf16_t)(32 * t + 16 * u + 4 * c + e < S ? vv[e] : 0.f);
                    }
                    if (c < 2) {
                        reinterpret_cast<bf16x4 *>(k_tile + i * 32 + key_slot(16 * u + n))[c] = k4;
                    }
                    const bf16x2 qp = {(bf16_t)qq[0], (bf16_t)qq[1]}, gp = {(bf16_t)qq[2], (bf16_t)qq[3]};
                    q2[u] = __builtin_bit_cast(uint32_t, qp), g2[u] = __builtin_bit_cast(uint32_t, gp);
                }
                const float mask_here = to_f32(mask_in[i]);
                if (t + waves < NB) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        in[i][q] = load_piece(i, t + waves, q);
                    }
                    mask_in[i] = load_mask(i, t + waves);
                }
                const auto sw = __builtin_amdgcn_permlane32_swap(g2[0], g2[1], false, false);
                uint2 *to = stash + (i * NB + t) * 128;
                to[lane] = make_uint2(q2[0], q2[1]), to[64 + lane] = make_uint2(sw[0], sw[1]);
                const int key = 32 * t + lane;
                const float mask = key < S ? finite_bias(mask_here * LOG2E) : 0.f;
                if (lane < 32) {
                    masks[t * TILE + i * 32 + lane] = mask;
                    if (mask != 0.f) {
                        atomicMin(first_masked, (uint32_t)t);
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < ROWS; ++i) {
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    if (n >= D) {
                        reinterpret_cast<bf16x4 *>(v_tile + i * 32 + (2 * u + (c >> 1)) * 8 + n - D)[c & 1] = v4[i][u];
                    }
                }
            }
        }
    } else {
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
            const float mask = key < S ? finite_bias(to_f32(w.mask) * LOG2E) : 0.f;
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
    }
    __syncthreads();
    const int masked_from = (int)*first_masked;

    //   logits: rows are sixteen keys, columns sixteen queries; chunks 0, 1, 2 hold the same keys against the three parts of the
    //           queries, chunk 3 nothing (zeros in the queries);
    //   p.v:    rows 0-7 are the values, row 8 ones (the row sums), the rest zeros; the k-slots of chunk c are keys 8 c .. 8 c + 7.
    const uint32_t v_first = n < D ? 8u * c + n : (uint32_t)(constants - vs) + (n == D ? 1u : 0u), v_tile = n < D ? (uint32_t)TILE : 0u;

    for (int j = split * waves + wave; j < NB; j += waves * p.splits) {
        int lv = lane; // opaque: the addresses of a query block's rows are formed where they are used, not kept over the keys
        asm volatile("" : "+v"(lv));
        bf16x8 q[ROWS][2]; // queries 32 j + 16 u + n
        uint32_t query[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            query[u] = (uint32_t)min(32 * j + 16 * u + (lv & 15), S - 1);
        }
        uint2 kept[ROWS];
        if constexpr (PROJECTS) {
#pragma unroll
            for (int i = 0; i < ROWS; ++i) {
                kept[i] = stash[(i * NB + j) * 128 + lv];
            }
        }
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                // a lane splits dims 2 c and 2 c + 1 of its query, then the four lanes of the query exchange: parts for dims
                const uint32_t raw = PROJECTS ? (u == 0 ? kept[i].x : kept[i].y) : *reinterpret_cast<const uint32_t *>(p.q + (int64_t)row_of(i) * S * p.q_ss + h * D +
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
        auto seeds = [&](const Raw &w, auto tail, auto finite) { // of the four rows' logits: the pair bias (finite: as finite_bias), -inf past the last key
            Tile s;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const bf16x8 raw = as_bf16x8(w.r[u]);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float x = HAS_NB ? to_f32(raw[e]) * LOG2E : 0.f;
                    s.x[u][e >> 2][e & 3] = decltype(finite)::value ? finite_bias(x) : x;
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
                    const f32x4 m = *reinterpret_cast<const f32x4 *>(masks + t * TILE + i * 32 + 8 * (TILES ? lv >> 4 : c) + 4 * a);
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
        auto rows = [&](int t, Tile &C, auto masked, auto reload) __attribute__((always_inline)) {
            Tile xa = logits(0, t, C, masked);
            fence();
            Tile xb = logits(1, t, C, masked);
            finish(0, t, xa, unshifted, std::false_type{});
            fence();
            xa = logits(2, t, C, masked);
            finish(1, t, xb, unshifted, std::false_type{});
            fence();
            xb = logits(3, t, C, masked);
            reload();
            finish(2, t, xa, unshifted, std::false_type{});
            fence();
            finish(3, t, xb, unshifted, std::false_type{});
            fence();
        };
        const f32x4 *tiles = TILES ? p.tiles + (int64_t)(h * NB + j) * NB * 256 : nullptr;
        auto load_tile = [&](int t) {
            Tile s;
            const char *from = reinterpret_cast<const char *>(tiles + min(t, NB - 1) * 256); // uniform; the lane's part in 32 bits
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s.x[i >> 1][i & 1] = *reinterpret_cast<const f32x4 *>(from + (16u * (uint32_t)lv + 1024u * i));
            }
            return s;
        };
        const int full = S >> 5;
        if constexpr (TILES) {
            Tile C0 = load_tile(0), C1 = load_tile(1);
            auto run = [&](int from, int to, auto masked) __attribute__((always_inline)) {
                int t = from;
                for (; t + 1 < to; t += 2) {
                    rows(t, C0, masked, [&] { C0 = load_tile(t + 2); });
                    rows(t + 1, C1, masked, [&] { C1 = load_tile(t + 3); });
                }
                if (t < to) {
                    rows(t, C0, masked, [&] { C0 = load_tile(t + 2); });
                    const Tile swap = C0;
                    C0 = C1, C1 = swap;
                }
            };
            const int plain = min(masked_from, NB);
            run(0, plain, std::false_type{});
            run(plain, NB, std::true_type{});
        } else {
            // Tiles without a mask, tiles with one, and the ragged last one, each in a loop of its own: with their choice inside one loop
            // a tile cost 76 vector instructions and 16 moves of register pairs more than the 160 that it needs (the whole operator, us: 1024
            // rows of 301 237 -> 221, 1000 of 420 432 -> 381).
            const int plain = min(masked_from, full);
            Raw raw = {zero_u4(), zero_u4()};
            if (S >= 8) {
                raw = load_nb(0);
            }
            auto run = [&](int from, int to, auto masked) __attribute__((always_inline)) {
                for (int t = from; t < to; ++t) {
                    Tile C = seeds(raw, std::false_type{}, std::false_type{});
                    raw = load_nb(t + 1);
                    rows(t, C, masked, [] {});
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
                Tile C = seeds(raw, std::true_type{}, std::false_type{});
                rows(full, C, std::true_type{}, [] {});
            }
        }
        // the two query halves side by side: lane l then has values 4 (l / 16 % 2) .. + 3 of query 16 (l / 32) + l % 16
        int le = lane;
        asm volatile("" : "+v"(le));
        const int pos = 32 * j + 16 * (le >> 5) + (le & 15);
        const uint32_t d0 = 4 * ((le >> 4) & 1), gate_at = (uint32_t)min(pos, S - 1) * (uint32_t)p.g_ss + d0, avg_at = (uint32_t)pos * (uint32_t)p.a_ss + d0;
        bf16x4 gates[ROWS]; // of all rows at once, one round trip (2000 rows of 384 627 -> 622 us, of 170 200 -> 195)
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            gates[i] = PROJECTS ? __builtin_bit_cast(bf16x4, stash[(i * NB + j) * 128 + 64 + le])
                                : *reinterpret_cast<const bf16x4 *>(p.gate + (int64_t)row_of(i) * S * p.g_ss + h * D + gate_at);
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
                auto again = [&](int t) {
                    if constexpr (TILES) {
                        return logits(i, t, load_tile(t), std::true_type{});
                    } else {
                        return logits(i, t, t < full ? seeds(load_nb(t), std::false_type{}, std::true_type{}) : seeds(load_tail(), std::true_type{}, std::true_type{}),
                                      std::true_type{});
                    }
                };
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

template <bool HAS_NB, bool PROJECTS, bool TILES = false>
int launch(SmallHeadParams p, hipStream_t stream)
{
    static size_t configured[KUTACC_DEVICE_SLOTS] = {};
    const size_t lds = lds_bytes(p.NB);
    if (const hipError_t e = kutacc_opt_in_lds(reinterpret_cast<const void *>(&small_head_attention_kernel<HAS_NB, PROJECTS, TILES>), lds, configured)) {
        return kutacc_hip_status(e);
    }
    // Four waves while three workgroups' keys fit a CU (the registers' limit of 12 waves), else eight.  A number that is no
    // multiple of four leaves SIMDs without their share: 1024 rows of 301 took 288 us at five waves, 240 at eight, 200 at four.
    const int waves = std::min(p.NB, 3 * lds <= (size_t)CU_LDS_BYTES ? 4 : 8);
    // a set's queries are dealt to several workgroups, each staging the keys again, only while the chip has room for them
    const int turns = (p.NB + waves - 1) / waves, room = 2 * kutacc_cu_count() / std::max(1, p.sets * p.H);
    p.splits = std::max(1, std::min(turns, room));
    const int64_t blocks = (int64_t)(p.sets + 7) / 8 * 8 * p.H * p.splits;
    if constexpr (TILES) {
        kutacc_prof::KernelTimer t("seed_tiles_kernel", 0.0, stream);
        seed_tiles_kernel<<<dim3((unsigned)((p.H * p.NB * p.NB + 3) / 4)), 256, 0, stream>>>(p);
    }
    const double C = (double)p.H * D, M = (double)p.B * p.S;
    kutacc_prof::KernelTimer t("small_head_attention_kernel", (PROJECTS ? 8.0 * M * C * C : 0.0) + 4.0 * M * (double)p.S * C, stream);
    small_head_attention_kernel<HAS_NB, PROJECTS, TILES><<<dim3((unsigned)blocks), 64 * waves, lds, stream>>>(p);
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

namespace {
// sets (of one head) whose queries and gates one scratch tensor of the call holds
int64_t stash_capacity(const kutacc_hip_attention_args_t &a)
{
    return std::min<int64_t>(INT32_MAX, a.batch * a.seq_len * a.nheads * D * 2 / (ROWS * ((a.seq_len + 31) / 32) * 1024));
}
} // namespace

// The projections inside: no pass that writes and reads four activations (1024 rows of 301 215 -> 181-191 us, of 107 3576 rows 199 -> 175, 5120 of
// 128 353 -> 281, 64 of 60 20.4 -> 12.8, whole operator), where the inputs are what projections_kernel takes, the scratch tensors are dense and hold
// the queries and gates (not where padding makes three times as much of the rows), and no workgroup writes what another one reads:
// neither the average nor the queries and gates, which lie in the scratch tensors in an order of their own, over the operands of the
// projections or over each other.  The kernel that reads q, k, v and gate takes those: it reads a position's queries and gates before it
// writes the position's average.  KUTACC_HIP_PATH_TILED asks for q, k, v and gate as the reference leaves them.
bool small_head_attention_projects(const kutacc_hip_attention_args_t &a)
{
    const int64_t C = a.nheads * D, M = a.batch * a.seq_len;
    if (a.path == KUTACC_HIP_PATH_TILED || C != PROJECTED || a.q_stride_s != C || a.k_stride_s != C || a.gate_stride_s != C ||
        3 * stash_capacity(a) < (a.batch + ROWS - 1) / ROWS * a.nheads || !small_head_attention_supports(a) || a.input_ld % 8 != 0 || a.input_ld >= (1 << 30) ||
        a.seq_len * a.input_ld >= (1 << 30) || !kutacc_hip_aligned16(a.input) || !kutacc_hip_aligned16(a.query_w) || !kutacc_hip_aligned16(a.key_w) ||
        !kutacc_hip_aligned16(a.value_w) || !kutacc_hip_aligned16(a.gating_w)) {
        return false;
    }
    struct Range {
        const void *from;
        int64_t bytes;
    };
    const auto apart = [](const Range &x, const Range &y) {
        const uintptr_t at = reinterpret_cast<uintptr_t>(x.from), other = reinterpret_cast<uintptr_t>(y.from);
        return at + (uintptr_t)x.bytes <= other || other + (uintptr_t)y.bytes <= at;
    };
    const Range avg = {a.avg, ((M - 1) * a.avg_stride_s + C) * 2}, stash[3] = {{a.q, M * C * 2}, {a.k, M * C * 2}, {a.gate, M * C * 2}};
    const Range read[] = {{a.input, ((M - 1) * a.input_ld + C) * 2}, {a.query_w, 2 * C * C}, {a.key_w, 2 * C * C}, {a.value_w, 2 * C * C},
                          {a.gating_w, 2 * C * C}, {a.gating_b, 4 * C}};
    for (const Range &operand : read) {
        if (!apart(operand, avg) || !apart(operand, stash[0]) || !apart(operand, stash[1]) || !apart(operand, stash[2])) {
            return false;
        }
    }
    return apart(avg, stash[0]) && apart(avg, stash[1]) && apart(avg, stash[2]);
}

int small_head_attention(const kutacc_hip_attention_args_t &a, bool projects, hipStream_t stream)
{
    SmallHeadParams p;
    p.q = (const bf16_t *)a.q, p.k = (const bf16_t *)a.k, p.v = (const bf16_t *)a.v, p.gate = (const bf16_t *)a.gate;
    p.bias = (const bf16_t *)a.bias, p.nb = (const bf16_t *)a.nonbatched_bias, p.avg = (bf16_t *)a.avg;
    p.q_ss = a.q_stride_s, p.k_ss = a.k_stride_s, p.g_ss = a.gate_stride_s, p.a_ss = a.avg_stride_s;
    p.v_se = a.v_stride_e, p.bias_sb = a.bias_stride_b, p.nb_sh = a.nb_stride_h, p.nb_sq = a.nb_stride_q;
    p.B = (int)a.batch, p.S = (int)a.seq_len, p.H = (int)a.nheads, p.NB = (p.S + 31) / 32, p.sets = (p.B + ROWS - 1) / ROWS, p.splits = 1;
    // (float)(1 / sqrt(head_size)) as the reference forms it (gating_attention.cpp:68)
    p.scale2 = (float)(1.0 / sqrt((double)D)) * LOG2E;
    if (!projects) {
        return p.nb ? launch<true, false>(p, stream) : launch<false, false>(p, stream);
    }
    p.x = (const bf16_t *)a.input, p.x_ss = a.input_ld;
    p.wq = (const bf16_t *)a.query_w, p.wk = (const bf16_t *)a.key_w, p.wv = (const bf16_t *)a.value_w, p.wg = (const bf16_t *)a.gating_w;
    p.bg = a.gating_b;
    p.stash[0] = (uint2 *)a.q, p.stash[1] = (uint2 *)a.k, p.stash[2] = (uint2 *)a.gate, p.stash_each = (int)stash_capacity(a);
    // The seeds as a pass of their own, behind the last stash where there is room for them: where the bias's rows start on any address, as they do
    // at seven lengths of eight -- the kernel's loads of them then cross lines --, and where sets and tiles pay for the pass: tiles of all
    // sets per CU, whose loads it makes cheaper, against its launch and its own tiles.  Operator, us, bias read in the kernel against this (256 CUs): 1024
    // rows of 301 171.5 164, of 253 122 118, of 381 240 235, 5120 of 127 274 254, 2000 of 199 196 186.5, of 319 438 330, 600 of 251 79.8 79.3, 300 of 301, on
    // the line, 70.3 69.9; below it 256 of 317 57.6 59.0, 400 of 219 58.1 58.4, 1024 of 94 43.2 45.5.  Rows on 16 bytes gain nothing: 2000 of 320 327 329, 600
    // of 256 75.6 79.
    const int64_t units = (int64_t)p.sets * p.H, last = std::max<int64_t>(0, units - 2 * (int64_t)p.stash_each), unit_bytes = (int64_t)ROWS * p.NB * 1024;
    char *const gate = (char *)a.gate, *const seeds = (char *)(((uintptr_t)gate + (uintptr_t)(last * unit_bytes) + 15) / 16 * 16);
    const int64_t seed_bytes = (int64_t)p.H * p.NB * p.NB * 4096, room = gate + a.batch * a.seq_len * a.nheads * D * 2 - seeds;
    const bool any_address = !kutacc_hip_aligned16(p.nb) || p.nb_sh % 8 != 0 || p.nb_sq % 8 != 0;
    if (p.nb && any_address && (int64_t)p.sets * p.NB * p.NB * 256 >= 7500 * (int64_t)kutacc_cu_count() && seed_bytes <= room) {
        p.tiles = (f32x4 *)seeds;
        return launch<true, true, true>(p, stream);
    }
    return p.nb ? launch<true, true>(p, stream) : launch<false, true>(p, stream);
}

} // namespace kutacc_launch
