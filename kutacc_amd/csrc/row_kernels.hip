// Row-wise HBM-bound kernels that sit in front of the attention operator: LayerNorm over the last
// axis, and the fused pair-bias producer LN(z) -> [H, c_z] projection -> [H, S, S] layout.
// Arithmetic follows reference src/normalization/layernorm_kernel.h:21-53 (shift by the first
// element, fp32 sum and sum of squares, clamped variance, rstd, then (x*rstd - rstd*mean)*gamma+beta)
// and reference src/linear/linear.cpp:21-42 (bf16 operands, result rounded to the storage type).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "device_util.h"
#include "launch_internal.h"
#include "mfma_tiles.h"
#include "profiler.h"

using namespace kutacc_dev;

namespace {

constexpr int ROW_WAVES = 4; // rows per workgroup, one wavefront each

// Per-row statistics exactly as the reference forms them; every lane returns the same values.
template <typename T>
__device__ __forceinline__ void row_stats(const T *__restrict__ row, int64_t size, int lane, float eps, float &rstd,
                                          float &shift)
{
    const float delta = to_f32(row[0]);
    float s1 = 0.f, s2 = 0.f;
    for (int64_t i = lane; i < size; i += 64) {
        const float v = to_f32(row[i]) - delta;
        s1 += v;
        s2 = fmaf(v, v, s2);
    }
    s1 = wave_sum(s1);
    s2 = wave_sum(s2);
    norm_from_sums<true>(s1, s2, delta, (float)size, eps, rstd, shift);
}

template <typename T>
__global__ __launch_bounds__(64 * ROW_WAVES) void layernorm_rows_kernel(const T *__restrict__ x, int64_t ld_x,
                                                                       const float *__restrict__ gamma,
                                                                       const float *__restrict__ beta,
                                                                       T *__restrict__ out, int64_t ld_out,
                                                                       int64_t rows, int64_t size, float eps, int64_t swap_j)
{
    const int lane = threadIdx.x % 64;
    const int64_t r = (int64_t)blockIdx.x * ROW_WAVES + threadIdx.x / 64;
    if (r >= rows) {
        return;
    }
    // swap_j != 0: rows are pairs (i, j) of an [rows / swap_j, swap_j] grid and output row (i, j) is computed from
    // input row (j, i) of the transposed grid
    const T *row = x + (swap_j ? (r % swap_j) * (rows / swap_j) + r / swap_j : r) * ld_x;
    float rstd, shift;
    row_stats(row, size, lane, eps, rstd, shift);
    T *orow = out + r * ld_out;
    for (int64_t i = lane; i < size; i += 64) {
        const float v = fmaf(to_f32(row[i]), rstd, shift);
        orow[i] = from_f32<T>(fmaf(v, gamma[i], beta[i]));
    }
}

// One wavefront per (i, j) row of z.  The normalised row is rounded to the storage type first (that
// is what a caller of the reference would hand to kutacc_af2_linear), then dotted with each of the
// H weight rows; nb[h, i, j] is written in place of the caller-side [S, S, H] -> [H, S, S] permute.
template <typename T>
__global__ __launch_bounds__(64 * ROW_WAVES) void pair_bias_kernel(const T *__restrict__ z,
                                                                  const float *__restrict__ gamma,
                                                                  const float *__restrict__ beta,
                                                                  const T *__restrict__ w, T *__restrict__ nb,
                                                                  T *__restrict__ z_norm, int64_t rows_i,
                                                                  int64_t rows_j, int64_t c_z, int64_t nheads, float eps,
                                                                  int transposed)
{
    const int lane = threadIdx.x % 64;
    const int64_t r = (int64_t)blockIdx.x * ROW_WAVES + threadIdx.x / 64;
    const int64_t rows = rows_i * rows_j;
    if (r >= rows) {
        return;
    }
    // transposed: output row (i, j) is computed from row (j, i) of z, stored [rows_j, rows_i, c_z]
    const T *row = z + (transposed ? (r % rows_j) * rows_i + r / rows_j : r) * c_z;
    float rstd, shift;
    row_stats(row, c_z, lane, eps, rstd, shift);
    for (int64_t h0 = 0; h0 < nheads; h0 += 8) {
        float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        for (int64_t c = lane; c < c_z; c += 64) {
            const float v = fmaf(to_f32(row[c]), rstd, shift);
            const T vn = from_f32<T>(fmaf(v, gamma[c], beta[c]));
            if (z_norm != nullptr && h0 == 0) {
                z_norm[r * c_z + c] = vn;
            }
            const float vf = to_f32(vn);
#pragma unroll
            for (int hh = 0; hh < 8; ++hh) {
                if (h0 + hh < nheads) {
                    acc[hh] = fmaf(vf, to_f32(w[(h0 + hh) * c_z + c]), acc[hh]);
                }
            }
        }
#pragma unroll
        for (int hh = 0; hh < 8; ++hh) {
            if (h0 + hh < nheads) {
                const float tot = wave_sum(acc[hh]);
                if (lane == 0) {
                    nb[(h0 + hh) * rows + r] = from_f32<T>(tot);
                }
            }
        }
    }
}


// ---------------------------------------------------------------------------------------------
// bf16 fast paths (row length a multiple of 8 with row_len/8 in {8, 16, 32, 64} lanes per row, rows
// and tensors 16-byte aligned).  A row is spread over LPR = row_len/8 lanes, 16 bytes each, so every
// load and store instruction moves whole cache lines and 64/LPR rows; sums run over the LPR lanes
// with DPP adds (no LDS traffic) up to 16 lanes and lane shuffles above.  Same arithmetic as the
// generic kernels: shift by the row's first element, fp32 sums, clamped variance.
// ---------------------------------------------------------------------------------------------
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

union Pack16 {
    uint4 u;
    bf16x8 b;
    bf16x2 p[4];
};

// NEAR: fewer than 2^24 rows, row pitches below 2^23 elements and less than 2^31 bytes from the first row to the end of
// the last (the launcher checks): rows are counted in 32 bits and addressed by 32-bit byte offsets from the tensors'
// first elements -- a 24-bit multiply per row where 64-bit pointer arithmetic spends three quarter-rate ones.
template <int LPR, bool NEAR>
__global__ __launch_bounds__(256) void layernorm_rows_bf16_kernel(const bf16_t *__restrict__ x, int64_t ld_x,
                                                                  const float *__restrict__ gamma,
                                                                  const float *__restrict__ beta, bf16_t *__restrict__ out,
                                                                  int64_t ld_out, int64_t rows, float eps, int64_t swap_j)
{
    constexpr int RPS = 64 / LPR; // rows per step of a wave
    constexpr int U = 4;          // steps in flight
    const int lane = threadIdx.x & 63;
    const int sub = lane % LPR, grp = lane / LPR;
    const int wave_in_block = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); // uniform
    float gm[8], bt[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        gm[e] = gamma[sub * 8 + e];
        bt[e] = beta[sub * 8 + e];
    }
    using index_t = std::conditional_t<NEAR, uint32_t, int64_t>;
    const index_t nrows = (index_t)rows, swap = (index_t)swap_j;
    const index_t r0 = ((index_t)blockIdx.x * 4 + wave_in_block) * (RPS * U);
    auto row_ptr = [&](auto *base, int64_t ld, index_t r) {
        if constexpr (NEAR) {
            using byte_t = std::conditional_t<std::is_const_v<std::remove_pointer_t<decltype(base)>>, const char, char>;
            return reinterpret_cast<decltype(base)>(reinterpret_cast<byte_t *>(base) +
                                                    (__umul24(r, 2u * (uint32_t)ld) + 16u * (uint32_t)sub));
        } else {
            return base + r * ld + sub * 8;
        }
    };
    Pack16 in[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        index_t r = r0 + u * RPS + grp;
        r = r < nrows ? r : nrows - 1;
        r = swap ? (r % swap) * (nrows / swap) + r / swap : r; // input row (j, i) for output row (i, j)
        in[u].u = *reinterpret_cast<const uint4 *>(row_ptr(x, ld_x, r));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const index_t r = r0 + u * RPS + grp;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            v[e] = (float)in[u].b[e];
        }
        const float x0 = __shfl(v[0], grp * LPR, 64);
        float rstd, shift;
        group_stats<LPR>(v, x0, (float)(LPR * 8), eps, rstd, shift);
        Pack16 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            o.b[e] = (bf16_t)fmaf(fmaf(v[e], rstd, shift), gm[e], bt[e]);
        }
        if (r < nrows) {
            *reinterpret_cast<uint4 *>(row_ptr(out, ld_out, r)) = o.u;
        }
    }
}

// Pair-bias producer, bf16, c_z = 128 (16 lanes per row), H <= 8.  A wave owns 32 consecutive rows of
// z; its four 16-lane groups walk 8 rows each (all loads of a lane are issued up front: 8 KB in
// flight per wave, and the small LDS tile leaves room for five workgroups per CU).  The normalised row is rounded to bf16, as a caller of the reference would hand it
// to kutacc_af2_linear, written out (if wanted) and parked in a wave-private LDS tile; when the rows
// are done, the [H, c_z] projection of all of them is 8 MFMAs (heads as MFMA rows, z rows as columns,
// fp32 accumulation), whose result has one z row per lane: every head's 32 values leave as one 64-byte store.
// The vector ALU, which bounds this kernel, is left with the LayerNorm alone.
constexpr int PAIR_BIAS_ROWS_PER_WAVE = 32; // a multiple of 32; LDS per workgroup = 1 KB per row
constexpr int64_t PAIR_BIAS_MAX_ROWS = (int64_t)1 << 23; // rows and byte offsets are counted in 32 bits: 2 GiB of z

// SHARED: the four waves of a workgroup normalise eight of the 32 rows each and the first one goes on alone, so that fewer units than the
// chip has SIMDs are not one wave's work each.
template <int H, bool SHARED>
__global__ __launch_bounds__(256) void pair_bias_bf16_kernel(const bf16_t *__restrict__ z, const float *__restrict__ gamma,
                                                             const float *__restrict__ beta, const bf16_t *__restrict__ w,
                                                             bf16_t *__restrict__ nb, bf16_t *__restrict__ z_norm,
                                                             int64_t rows, float eps, int64_t rows_i, int64_t rows_j,
                                                             int transposed, uint4 *__restrict__ nbf, int frag_nb,
                                                             int frag_nt, int frag_tiles)
{
    constexpr int LPR = 16, CZ = 128, STEPS = PAIR_BIAS_ROWS_PER_WAVE / (SHARED ? 16 : 4), RB = PAIR_BIAS_ROWS_PER_WAVE / 32;
    __shared__ uint4 tiles[SHARED ? 1 : 4][RB * 2 * 256]; // per wave (or of all four): its rows x 128 channels as 32 x 64 panels
    const int lane = threadIdx.x & 63;
    const int sub = lane & 15, grp = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); // uniform: the wave's first row stays in scalar registers
    // Rows are counted in 32 bits and addressed by 32-bit byte offsets from the tensors' first elements (the launcher
    // sends at most 2^23 rows here: 2 GiB of z), not by 64-bit products per lane and row.
    const uint32_t nrows = (uint32_t)rows, ncol = (uint32_t)rows_j, nrow_i = (uint32_t)rows_i;
    // A wave's rows: row0 and the `count` - 1 behind it.  Without the attention's copy they are 32 rows as they come.  With it they are
    // key tile t of query q, on a grid of whole blocks of queries and whole tiles of keys: the last tile of a query has fewer
    // rows (PAST_THE_END_F16 or LOWEST_BIAS takes the place of the others in the copy), and queries past the last repeat that one, in the copy only.  A workgroup's
    // waves take four queries that follow each other: their pieces of 16 bytes in the copy are neighbours, and so are their rows of z for the
    // ending node.  (Four tiles of one query, now: triangle attention of 160 residues 33.0 and 32.5 us, of 200 42.1 and 41.6, of 256 46.9 and 46.5, of 128 no
    // difference, of 112 20.0 and 20.6; MSA rows 256 x 256 100.6 and 99.2; 508 x 259 with eight heads, this kernel, 12.8 and 10.6.)
    uint32_t row0 = (SHARED ? (uint32_t)blockIdx.x : (uint32_t)blockIdx.x * 4 + wave) * PAIR_BIAS_ROWS_PER_WAVE, count = 0;
    const int first_row = (SHARED ? 8 * wave : 0) + grp * STEPS; // of this lane's group
    int q = 0, t = 0;
    if (nbf == nullptr) {
        if (row0 >= nrows) {
            return;
        }
        count = min(32u, nrows - row0);
    } else {
        q = SHARED ? (int)(blockIdx.x / (uint32_t)frag_nb) : (int)(blockIdx.x / (uint32_t)frag_nb * 4) + wave, t = (int)(blockIdx.x % (uint32_t)frag_nb);
        if (q >= 32 * frag_nb) {
            return;
        }
        row0 = min((uint32_t)q, nrow_i - 1) * ncol + 32u * t;
        count = min(32u, ncol - 32u * t);
    }
    const bool stores = q < (int)nrow_i; // (nrow_i = ncol where there is a copy)
    const char *zbytes = reinterpret_cast<const char *>(z);
    uint4 *tile = tiles[SHARED ? 0 : wave];
    Pack16 in[STEPS];
    {
        // transposed: output row (i, j) is computed from row (j, i) of z, stored [rows_j, rows_i, c_z]; the walk
        // over consecutive output rows then steps through z with stride rows_i rows
        uint32_t r = row0 + first_row;
        uint32_t i = transposed ? r / ncol : 0, j = transposed ? r % ncol : 0;
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            uint32_t src = transposed ? j * nrow_i + i : r;
            src = first_row + s < (int)count ? src : 0;
            in[s].u = *reinterpret_cast<const uint4 *>(zbytes + (src * (2u * CZ) + 16u * sub));
            ++r;
            if (++j == ncol) {
                j = 0, ++i;
            }
        }
    }
    float gm[8], bt[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        gm[e] = gamma[sub * 8 + e];
        bt[e] = beta[sub * 8 + e];
    }
    // weight fragments, heads as MFMA rows (rows >= H are zero): lane (head, g) holds w[head][16 ks + 8 g .. + 8]
    kutacc_dev::bf16x8 wf[8];
    if (!SHARED || wave == 0) {
        const int head = lane & 31, g = lane >> 5;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            uint4 v = make_uint4(0u, 0u, 0u, 0u);
            if (head < H) {
                v = *reinterpret_cast<const uint4 *>(w + head * CZ + ks * 16 + g * 8);
            }
            wf[ks] = kutacc_dev::as_bf16x8(v);
        }
    }
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
        const int row_local = first_row + s;
        const uint32_t r = row0 + row_local;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            v[e] = (float)in[s].b[e];
        }
        const float x0 = __shfl(v[0], grp * 16, 64);
        float rstd, shift;
        group_stats<LPR>(v, x0, (float)CZ, eps, rstd, shift);
        Pack16 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            o.b[e] = (bf16_t)fmaf(fmaf(v[e], rstd, shift), gm[e], bt[e]);
        }
        if (z_norm != nullptr && stores && row_local < (int)count) {
            *reinterpret_cast<uint4 *>(reinterpret_cast<char *>(z_norm) + (r * (2u * CZ) + 16u * sub)) = o.u;
        }
        tile[((row_local >> 5) * 2 + (sub >> 3)) * 256 + kutacc_dev::panel_slot(row_local & 31, sub & 7)] = o.u;
    }
    if constexpr (SHARED) {
        __syncthreads();
        if (wave != 0) {
            return;
        }
    }
    // otherwise the tile is private to the wave and LDS operations of a wave complete in order: no barrier
    const int col = lane & 31, g = lane >> 5;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        kutacc_dev::f32x16 acc = kutacc_dev::zero16();
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            const uint4 zf = tile[(rb * 2 + (ks >> 2)) * 256 + kutacc_dev::panel_slot(col, 2 * (ks & 3) + g)];
            acc = kutacc_dev::mfma(wf[ks], kutacc_dev::as_bf16x8(zf), acc);
        }
        // accumulator v < 4 of lane (col, g) is head 4 g + v of z row row0 + col
        static_assert(RB == 1, "a wave is one key tile");
        const uint32_t r = row0 + col;
        const bool real = col < (int)count;
        if (real && stores) {
            char *nbytes = reinterpret_cast<char *>(nb);
            const uint32_t first = 2u * (__umul24(4u * g, nrows) + r); // head 4 g of row r, in bytes; H * rows * 2 < 2^28
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if (4 * g + v < H) {
                    *reinterpret_cast<bf16_t *>(nbytes + (first + 2u * v * nrows)) = (bf16_t)acc[v];
                }
            }
        }
        if (nbf != nullptr && frag_tiles) {
            // The copy the two-row attention kernel reads: fp32 tiles in the order of its logits accumulators, in log2 units,
            // [head][query block][key tile][4][64 lanes] x 16 bytes -- lane (pi^-1(q mod 32), g') holds keys 16 g' .. + 15 of
            // the tile for query q, four per piece.  Through the wave's tile: [head][32 keys] fp32, of which a lane takes
            // the four keys of one piece.
            static_assert(RB == 1 && H <= 8, "one lane per piece: 8 pieces per head");
            float *t32 = reinterpret_cast<float *>(tile);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if (4 * g + v < H) {
                    const float x = real ? (float)(bf16_t)acc[v] * kutacc_dev::LOG2E : kutacc_dev::LOWEST_BIAS;
                    t32[(4 * g + v) * 32 + col] = x < kutacc_dev::LOWEST_BIAS ? kutacc_dev::LOWEST_BIAS : x; // finite, -inf too
                }
            }
            __builtin_amdgcn_wave_barrier(); // other lanes' stores: keep the loads below behind them
            if (lane < 8 * H) {
                const int h = lane >> 3, c = lane & 7; // piece c: keys 4 c .. 4 c + 3 = half g' = c >> 2, piece a = c & 3
                const uint4 val = *reinterpret_cast<const uint4 *>(t32 + h * 32 + c * 4);
                const int qr = q & 31;
                const int qlane = (qr & 3) | (((qr >> 4) & 1) << 2) | (((qr >> 2) & 3) << 3);
                uint4 *dst = nbf + ((((int64_t)h * frag_nb + (q >> 5)) * frag_nt + t) * 4 + (c & 3)) * 64 + qlane + 32 * (c >> 2);
                *dst = val;
                if (t + 1 == frag_nb && frag_nt > frag_nb) { // the phantom tile that pads the key tiles to a pair
                    const uint32_t out = __float_as_uint(kutacc_dev::LOWEST_BIAS);
                    dst[256] = make_uint4(out, out, out, out);
                }
            }
        } else if (nbf != nullptr) {
            // The copy the attention kernels read: for head h, query block j, key tile t, 16-key half g' and 8-key half e the 16 bytes of lane
            // (pi^-1(q mod 32), g'), pi being the row order of the attention's accumulators; values in log2 units as
            // fp16 (the bf16 pair bias times log2(e), eleven significant bits kept).  Through the wave's tile, which nobody
            // reads any more: [head][32 keys].
            static_assert(RB == 1, "the transposing buffer lies on the first row block of the tile");
            uint16_t *t16 = reinterpret_cast<uint16_t *>(tile);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if (4 * g + v < H) {
                    t16[(4 * g + v) * 32 + col] = real ? kutacc_dev::pair_bias_log2_f16((float)(bf16_t)acc[v]) : (uint16_t)kutacc_dev::PAST_THE_END_F16;
                }
            }
            __builtin_amdgcn_wave_barrier(); // other lanes' stores: keep the loads below behind them
            if (lane < 4 * H) {
                const int h = lane >> 2, c = lane & 3;
                const uint4 val = *reinterpret_cast<const uint4 *>(t16 + h * 32 + c * 8);
                const int qr = q & 31;
                const int qlane = (qr & 3) | (((qr >> 4) & 1) << 2) | (((qr >> 2) & 3) << 3);
                uint4 *dst = nbf + ((((int64_t)h * frag_nb + (q >> 5)) * frag_nt + t) * 2 + (c & 1)) * 64 + qlane + 32 * (c >> 1);
                *dst = val;
                if (t + 1 == frag_nb && frag_nt > frag_nb) { // the phantom tile that pads the key tiles to a pair
                    const uint32_t out = kutacc_dev::PAST_THE_END_F16 * 0x10001u;
                    dst[128] = make_uint4(out, out, out, out);
                }
            }
        }
    }
}

// kutacc_af2_linear in bf16 for input rows of K = 64, 128 or 256 features and at most 256 outputs (reference
// src/linear/linear.cpp:21-42): result = beta * result + act . W^T + bias.  HBM-bound (a pair-bias projection reads 256 bytes per
// row and writes 16), so the weights stay in the LDS as MFMA fragments, padded with zeros to whole blocks of 32 outputs, and every
// wave streams 32 rows at a time: whole cache lines in through its panel, the next rows requested before the current ones are
// multiplied, 64 outputs at a time out through the same panel.  A lane ends up with one row and four consecutive outputs per
// accumulator group.  The addition of beta * result is a kernel of its own (its sixteen guarded loads per block of outputs are sixteen
// branches, taken or not), groups of eight outputs past n are skipped, and with 128 registers four workgroups share a CU up to 128
// features.  The call on new rows, us: 147 456 x 128 -> 8 11.1 without these, 9.1 here (4.4 TB/s; the kernel alone 8.1 on average), 54.5 on
// the scalar kernel; over and over on the same rows, 100 000 x 128 -> 128 19.1 -> 15.7; 300 000 x 256 -> 256 105.5 -> 98.2.
template <int K, bool BETA>
__global__ __launch_bounds__(256, K == 256 ? 2 : 4) void linear_rows_kernel(const bf16_t *__restrict__ act, int64_t ld_act, const bf16_t *__restrict__ w,
                                                          int64_t ld_w, const float *__restrict__ bias, bf16_t *__restrict__ out, int64_t m,
                                                          int ld_out, int slice, float beta, int piece)
{
    using kutacc_dev::PanelRegs;
    constexpr int KS = K / 16, CP = K / 64;
    extern __shared__ uint4 lds[]; // [blocks of 32 outputs][KS][64 lanes], a panel per wave, the bias
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, g = lane >> 5;
    // this workgroup's outputs: slice blockIdx.y
    const int n = ld_out - (int)blockIdx.y * slice < slice ? ld_out - (int)blockIdx.y * slice : slice;
    w += (int64_t)blockIdx.y * slice * ld_w, out += blockIdx.y * slice, bias += bias != nullptr ? blockIdx.y * slice : 0;
    const int blocks = (n + 31) / 32;
    uint4 *panel = lds + blocks * KS * 64 + wave * 256;
    float *bias_s = reinterpret_cast<float *>(lds + blocks * KS * 64 + 4 * 256);
    const int64_t steps = (m + 31) / 32, stride = (int64_t)gridDim.x * 4;
    int64_t step = (int64_t)blockIdx.x * 4 + wave;
    auto load = [&](int64_t s, int cp) {
        const int64_t row0 = s * 32;
        return kutacc_dev::panel_load(act + row0 * ld_act, ld_act, 0, (int)(m - row0 < 32 ? m - row0 : 32) - 1, cp * 64, lane);
    };
    PanelRegs t[CP];
    if (step < steps) {
#pragma unroll
        for (int cp = 0; cp < CP; ++cp) {
            t[cp] = load(step, cp);
        }
    }
    for (int base = tid; base < blocks * KS * 64; base += 1024) { // four loads in flight per thread
        uint4 v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = base + 256 * i, ln = idx & 63, ks = (idx >> 6) % KS, row = (idx >> 6) / KS * 32 + (ln & 31);
            v[i] = make_uint4(0u, 0u, 0u, 0u);
            if (row < n) {
                v[i] = *reinterpret_cast<const uint4 *>(w + row * ld_w + ks * 16 + (ln >> 5) * 8);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (base + 256 * i < blocks * KS * 64) {
                lds[base + 256 * i] = v[i];
            }
        }
    }
    if (tid < blocks * 32) {
        bias_s[tid] = bias != nullptr && tid < n ? bias[tid] : 0.f;
    }
    __syncthreads();
    for (; step < steps; step += stride) {
        kutacc_dev::bf16x8 af[KS];
#pragma unroll
        for (int cp = 0; cp < CP; ++cp) {
            kutacc_dev::panel_store(panel, lane, t[cp]);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                af[4 * cp + k] = kutacc_dev::as_bf16x8(panel[kutacc_dev::panel_slot(r, 2 * k + g)]);
            }
        }
        if (step + stride < steps) {
#pragma unroll
            for (int cp = 0; cp < CP; ++cp) {
                t[cp] = load(step + stride, cp);
            }
        }
        const int64_t row0 = step * 32;
        const int rows = (int)(m - row0 < 32 ? m - row0 : 32);
        bf16_t *dst = out + row0 * ld_out;
        for (int f0 = 0; f0 < n; f0 += 64) {
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int fb = f0 + 32 * half; // a block of 32 outputs
                if (fb >= n) {
                    break;
                }
                kutacc_dev::f32x16 acc = kutacc_dev::zero16();
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    acc = kutacc_dev::mfma(kutacc_dev::as_bf16x8(lds[(fb / 32 * KS + ks) * 64 + lane]), af[ks], acc);
                }
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    if (fb + 8 * a >= n) {
                        break;
                    }
                    const int f = fb + 8 * a + 4 * g;
                    const kutacc_dev::f32x4 bv = *reinterpret_cast<const kutacc_dev::f32x4 *>(bias_s + f);
                    kutacc_dev::bf16x4 ov;
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        float v = acc[4 * a + c] + bv[c];
                        if constexpr (BETA) {
                            v += f + c < n && r < rows ? beta * to_f32(dst[r * ld_out + f + c]) : 0.f;
                        }
                        ov[c] = (bf16_t)v;
                    }
                    *(reinterpret_cast<kutacc_dev::bf16x4 *>(panel + kutacc_dev::panel_slot(r, half * 4 + a)) + g) = ov;
                }
            }
            // out as runs of `piece` outputs (8, 4 or 1: what n and the result's alignment allow)
            const int width = n - f0 < 64 ? n - f0 : 64, pieces = width / piece, shift = 31 - __clz(pieces);
            const bool pow2 = (1 << shift) == pieces;
            auto copy = [&](auto *to, auto *from) { *to = *from; };
            for (int i = lane; i < rows * pieces; i += 64) {
                const int row = pow2 ? i >> shift : i / pieces, col = (i - row * pieces) * piece;
                bf16_t *to = dst + row * ld_out + f0 + col;
                const bf16_t *from = reinterpret_cast<const bf16_t *>(panel + kutacc_dev::panel_slot(row, col >> 3)) + (col & 7);
                if (piece == 8) {
                    copy(reinterpret_cast<uint4 *>(to), reinterpret_cast<const uint4 *>(from));
                } else if (piece == 4) {
                    copy(reinterpret_cast<uint2 *>(to), reinterpret_cast<const uint2 *>(from));
                } else {
                    copy(to, from);
                }
            }
        }
    }
}

template <typename T>
int launch_layernorm(const void *x, int64_t ld_x, const float *gamma, const float *beta, void *out, int64_t ld_out,
                     int64_t rows, int64_t size, float eps, int64_t swap_j, hipStream_t stream)
{
    if (sizeof(T) == 2 && (size == 64 || size == 128 || size == 256 || size == 512) && ld_x % 8 == 0 && ld_out % 8 == 0 &&
        (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) % 16 == 0) {
        const int lpr = (int)(size / 8);
        const int64_t rows_per_block = 4 * 4 * (64 / lpr);
        const int64_t nblk = (rows + rows_per_block - 1) / rows_per_block;
        if (nblk > INT32_MAX) {
            return KUTACC_HIP_EUNSUPPORTED;
        }
        const bf16_t *xi = (const bf16_t *)x;
        bf16_t *oi = (bf16_t *)out;
        const int64_t pitch = ld_x > ld_out ? ld_x : ld_out;
        const bool near = rows < (1 << 24) && pitch < (1 << 23) && rows * pitch * 2 < ((int64_t)1 << 31);
        auto launch = [&](auto kernel) { kernel<<<(unsigned)nblk, 256, 0, stream>>>(xi, ld_x, gamma, beta, oi, ld_out, rows, eps, swap_j); };
        switch (lpr) {
            case 8: near ? launch(layernorm_rows_bf16_kernel<8, true>) : launch(layernorm_rows_bf16_kernel<8, false>); break;
            case 16: near ? launch(layernorm_rows_bf16_kernel<16, true>) : launch(layernorm_rows_bf16_kernel<16, false>); break;
            case 32: near ? launch(layernorm_rows_bf16_kernel<32, true>) : launch(layernorm_rows_bf16_kernel<32, false>); break;
            default: near ? launch(layernorm_rows_bf16_kernel<64, true>) : launch(layernorm_rows_bf16_kernel<64, false>); break;
        }
        return kutacc_hip_status(hipGetLastError());
    }
    const int64_t blocks = (rows + ROW_WAVES - 1) / ROW_WAVES;
    if (blocks > INT32_MAX) {
        return KUTACC_HIP_EUNSUPPORTED;
    }
    layernorm_rows_kernel<T><<<(unsigned)blocks, 64 * ROW_WAVES, 0, stream>>>((const T *)x, ld_x, gamma, beta, (T *)out,
                                                                               ld_out, rows, size, eps, swap_j);
    return kutacc_hip_status(hipGetLastError());
}

template <typename T>
int launch_pair_bias(const void *z, const float *gamma, const float *beta, const void *w, void *nb, void *z_norm,
                     int64_t rows_i, int64_t rows_j, int64_t c_z, int64_t nheads, float eps, int transposed,
                     hipStream_t stream, void *fragments, int frag_nb, int frag_nt, int frag_tiles)
{
    const int64_t rows = rows_i * rows_j;
    if (fragments != nullptr &&
        (!kutacc_launch::pair_bias_writes_fragments(z, w, z_norm, rows_i, rows_j, c_z, nheads,
                                                    sizeof(T) == 2 ? KUTACC_DTYPE_BF16 : KUTACC_DTYPE_FP32) ||
         frag_nb != (rows_j + 31) / 32 || frag_nt != ((frag_nb + 1) & ~1))) {
        return KUTACC_HIP_EINVAL;
    }
    if (sizeof(T) == 2 && c_z == 128 && (nheads == 4 || nheads == 8) && rows <= PAIR_BIAS_MAX_ROWS &&
        (reinterpret_cast<uintptr_t>(z) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(z_norm)) % 16 == 0) {
        const int64_t wave_tiles = fragments != nullptr ? (int64_t)32 * frag_nb * frag_nb : (rows + PAIR_BIAS_ROWS_PER_WAVE - 1) / PAIR_BIAS_ROWS_PER_WAVE;
        // Up to one unit a SIMD.  Triangle attention, whole block, a wave a unit against four (us): 48 residues 14.9 and 13.7, 77 17.8 and 16.8, 96
        // 19.2 and 17.5, 128 21.2 and 20.0, 160 (800 units) 32.6 and 30.6; beyond, 200 41.7 and 41.5, 256 45.5 and 45.4; MSA rows 32 x 64 20.1 and 18.9.
        const bool shared = wave_tiles <= 4 * (int64_t)kutacc_cu_count();
        const int64_t nblk = shared ? wave_tiles : (wave_tiles + 3) / 4;
        if (nblk > INT32_MAX) {
            return KUTACC_HIP_EUNSUPPORTED;
        }
        const auto launch = [&](auto kernel) {
            kernel<<<(unsigned)nblk, 256, 0, stream>>>((const bf16_t *)z, gamma, beta, (const bf16_t *)w, (bf16_t *)nb, (bf16_t *)z_norm, rows, eps, rows_i,
                                                       rows_j, transposed, (uint4 *)fragments, frag_nb, frag_nt, frag_tiles);
        };
        if (nheads == 4) {
            shared ? launch(pair_bias_bf16_kernel<4, true>) : launch(pair_bias_bf16_kernel<4, false>);
        } else {
            shared ? launch(pair_bias_bf16_kernel<8, true>) : launch(pair_bias_bf16_kernel<8, false>);
        }
        return kutacc_hip_status(hipGetLastError());
    }
    const int64_t blocks = (rows + ROW_WAVES - 1) / ROW_WAVES;
    if (blocks > INT32_MAX) {
        return KUTACC_HIP_EUNSUPPORTED;
    }
    pair_bias_kernel<T><<<(unsigned)blocks, 64 * ROW_WAVES, 0, stream>>>(
        (const T *)z, gamma, beta, (const T *)w, (T *)nb, (T *)z_norm, rows_i, rows_j, c_z, nheads, eps, transposed);
    return kutacc_hip_status(hipGetLastError());
}

} // namespace

namespace kutacc_launch {

int layernorm_rows(const void *x, int64_t ld_x, const float *gamma, const float *beta, void *out, int64_t ld_out,
                   int64_t rows, int64_t size, float eps, int32_t dtype, hipStream_t stream, int64_t swap_j)
{
    if (!x || !gamma || !beta || !out || rows <= 0 || size <= 0 || ld_x < size || ld_out < size || swap_j < 0 ||
        (swap_j > 0 && rows % swap_j != 0)) {
        return KUTACC_HIP_EINVAL;
    }
    if (dtype == KUTACC_DTYPE_BF16) {
        return launch_layernorm<bf16_t>(x, ld_x, gamma, beta, out, ld_out, rows, size, eps, swap_j, stream);
    }
    if (dtype == KUTACC_DTYPE_FP32) {
        return launch_layernorm<float>(x, ld_x, gamma, beta, out, ld_out, rows, size, eps, swap_j, stream);
    }
    return KUTACC_HIP_EINVAL;
}

// bf16 rows of 64, 128 or 256 features on the kernel above; other bf16 shapes on the MFMA tiles of pair_gemm where those
// take them (beta = 0, extents and pitches in multiples of 8); the rest, and fp32, on the shape-agnostic kernel
int linear(int32_t dtype, const void *act, int64_t ld_act, const void *w, int64_t ld_w, const float *bias, void *result, int64_t m,
           int64_t n, int64_t k, float beta, hipStream_t stream)
{
    if (dtype == KUTACC_DTYPE_BF16 && m > 0 && n > 0 && k > 0 && kutacc_hip_aligned16(act) && kutacc_hip_aligned16(w) && ld_act % 8 == 0 &&
        ld_w % 8 == 0) {
        if ((k == 64 || k == 128 || k == 256) && n <= 256 && m <= INT64_MAX / 4096) {
            // Slices of outputs whose weights fill at most 32 KB: four workgroups a CU, and few rows still make many workgroups
            // (all 256 outputs of 256 features at once, 62 899 rows: 39 us against 31 in slices; 3 313 rows x 128: 15 against 9).
            const int slice = (int)(n < 16384 / k ? n : 16384 / k), slices = (int)((n + slice - 1) / slice);
            const size_t lds_bytes = (size_t)((slice + 31) / 32 * (k / 16) * 64 + 4 * 256) * 16 + 256 * sizeof(float);
            const int cus = kutacc_cu_count();
            // as many workgroups as are resident at once, at most eight per CU; each stages the weights once
            const int64_t resident = (int64_t)(160 * 1024) / (int64_t)lds_bytes;
            const int64_t cap = (cus * (resident > 8 ? 8 : resident) + slices - 1) / slices, blocks = (m + 127) / 128;
            const uintptr_t to = reinterpret_cast<uintptr_t>(result);
            const int piece = n % 8 == 0 && to % 16 == 0 ? 8 : (n % 4 == 0 && to % 8 == 0 ? 4 : 1);
            auto launch = [&](auto kernel, size_t *configured) {
                if (const hipError_t e = kutacc_opt_in_lds(reinterpret_cast<const void *>(kernel), lds_bytes, configured)) {
                    return kutacc_hip_status(e);
                }
                kutacc_prof::KernelTimer t("linear_rows_kernel", 2.0 * (double)m * (double)n * (double)k, stream);
                kernel<<<dim3((unsigned)(blocks < cap ? blocks : cap), (unsigned)slices), 256, lds_bytes, stream>>>(
                    (const bf16_t *)act, ld_act, (const bf16_t *)w, ld_w, bias, (bf16_t *)result, m, (int)n, slice, beta, piece);
                return kutacc_hip_status(hipGetLastError());
            };
            static size_t configured[6][KUTACC_DEVICE_SLOTS] = {};
            if (beta != 0.f) {
                return k == 64 ? launch(linear_rows_kernel<64, true>, configured[0])
                               : (k == 128 ? launch(linear_rows_kernel<128, true>, configured[1]) : launch(linear_rows_kernel<256, true>, configured[2]));
            }
            return k == 64 ? launch(linear_rows_kernel<64, false>, configured[3])
                           : (k == 128 ? launch(linear_rows_kernel<128, false>, configured[4]) : launch(linear_rows_kernel<256, false>, configured[5]));
        }
        if (beta == 0.f) {
            kutacc_hip_gemm_args_t g = {};
            g.m = m, g.n = n, g.k = k, g.batches = 1, g.dtype = dtype, g.path = KUTACC_HIP_PATH_FUSED;
            g.a = act, g.a_stride_m = ld_act, g.a_stride_k = 1, g.b = w, g.b_stride_n = ld_w, g.b_stride_k = 1;
            g.c = result, g.c_stride_m = n, g.bias = bias, g.bias_axis = bias ? 1 : 0;
            const int rc = pair_gemm(g, stream);
            if (rc >= 0) {
                return rc;
            }
        }
    }
    return gemm_nt(dtype, act, ld_act, w, ld_w, bias, result, n, 1, m, n, k, beta, stream);
}

bool pair_bias_writes_fragments(const void *z, const void *w, const void *z_norm, int64_t rows_i, int64_t rows_j, int64_t c_z,
                                int64_t nheads, int32_t dtype)
{
    // The MFMA producer, on a square grid.  At lengths that are no multiple of 32 the whole tiles cost it some waves (77
    // residues 48 %, 500 5 %) and the block saves a launch: triangle attention at 77 residues 27.2 -> 24.9 us,
    // 301: 111.2 -> 107.7, 691: 543 -> 539; MSA rows 64 x 77: 42.3 -> 38.0, 508 x 259: 317.9 -> 312.6.
    return dtype == KUTACC_DTYPE_BF16 && c_z == 128 && (nheads == 4 || nheads == 8) && rows_i == rows_j &&
           rows_i * rows_j <= PAIR_BIAS_MAX_ROWS &&
           (reinterpret_cast<uintptr_t>(z) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(z_norm)) % 16 == 0;
}

int pair_bias(const void *z, const float *gamma, const float *beta, const void *w, void *nb, void *z_norm,
              int64_t rows_i, int64_t rows_j, int64_t c_z, int64_t nheads, float eps, int32_t dtype, int transposed,
              hipStream_t stream, void *fragments, int frag_nb, int frag_nt, int frag_tiles)
{
    if (!z || !gamma || !beta || !w || !nb || rows_i <= 0 || rows_j <= 0 || c_z <= 0 || nheads <= 0) {
        return KUTACC_HIP_EINVAL;
    }
    if (dtype == KUTACC_DTYPE_BF16) {
        return launch_pair_bias<bf16_t>(z, gamma, beta, w, nb, z_norm, rows_i, rows_j, c_z, nheads, eps, transposed, stream,
                                        fragments, frag_nb, frag_nt, frag_tiles);
    }
    if (dtype == KUTACC_DTYPE_FP32) {
        return launch_pair_bias<float>(z, gamma, beta, w, nb, z_norm, rows_i, rows_j, c_z, nheads, eps, transposed, stream,
                                       fragments, frag_nb, frag_nt, frag_tiles);
    }
    return KUTACC_HIP_EINVAL;
}

} // namespace kutacc_launch
