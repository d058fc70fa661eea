// Gated attention for fp32 storage on the fp32 matrix core (v_mfma_f32_16x16x4_f32), head_size 32, short sequences.
//
// The reference serves every call through its GEMM (src/linear/mm.cpp:77-86); the bf16 kernels of fused_attention.hip
// take bf16 storage only, and an fp32 tensor rounded to bf16 operands would miss the fp32 bar (1e-4 relative).  The
// fp32 MFMA multiplies fp32 operands exactly and accumulates in fp32, at a sixteenth of the bf16 rate -- enough for the
// small fp32 problems (the MSA-row benchmark shape is 0.74 GFLOP), which are bound by latency, not by arithmetic.
//
//   fp32_head_kernel     one workgroup of eight waves per (batch row b, head h) and share of its queries: the four
//       projections of the head (a wave holds 16 features of one matrix in registers; the positions are staged
//       through the LDS, 32 at a time), then flash-style attention with a running maximum, 16 queries per wave at a time, the
//       sigmoid gate, and the gated average stored where the reference leaves it
//       (src/attention/gating_attention.cpp:47-66, 73-150).  q, k, v, gate, logits and probabilities never leave the chip.
//   fp32_rows_gemm_kernel   out[m, n] = sum_k a[m, k] * w[n, k] + bias[n]: the output projection (reference :152-157).
//
// What bounds it: the fp32 matrix rate (64 multiply-adds per cycle and SIMD: 16 positions x 32 features x 256 channels
// take 4096 cycles) once loads are out of the way.  The smaller 16x16x4 form has the rate of 32x32x2 and twice the
// pieces to deal out: two waves per SIMD cover each other's LDS reads, and 64 queries occupy four SIMDs instead of two.
// A wave's whole weight block is in flight before the first position arrives.  In front of the first product stand the loads:
// whole lines (load_rows below) brought 16 rows x 64 positions x 256 channels from 21.8 to 19.1 us and 64 x 200 x 256 from 151 to 131,
// of which the output projection's are 30 and 17.4: its floor, the matrix cores', is 10.7.  (With four waves of 32x32x2 and weights
// loaded as they were used they were 40.9 and 235.)  Two tiles of positions in the LDS, in turn or both at once, gave the first
// projections under 1 % or cost 4 %.
//
// Operand and accumulator layouts of the 16x16x4 MFMA: A is 16 x 4, lane l holds A[l % 16][l / 16]; B is 4 x 16, lane l
// holds B[l / 16][l % 16]; D[4 g + v][j] sits in lane j + 16 g, register v.  A lane reads four consecutive k with one
// 16-byte load and uses them in four successive products (the order of k is the same for both operands).  Products are
// formed so that an accumulator is the next product's B operand as it stands: register v of the transposed
// probabilities holds keys 4 g + v, and the value operand reads the same four keys from a transposed V.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <type_traits>

#include "device_util.h"
#include "launch_internal.h"
#include "profiler.h"

using namespace kutacc_dev;

namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef f32x4 f32x4_any __attribute__((aligned(4))); // global loads and stores of 16 bytes need 4-byte alignment only

constexpr int HEAD = 32;
constexpr int LDP = 36;            // row pitch of the [position][feature] arrays in LDS, in floats: 16 rows' 16-byte pieces in 16 bank groups
constexpr int MAX_SEQ = 224;       // what the LDS holds of K, V, Q and gate of one head in fp32
constexpr int64_t GEMM_WORKGROUPS_PER_CU = 3; // 64 x 200 x 256 positions' projection 17.4 us, with 2 or 4 a CU 18.8 and 20.3, with one tile each 20.3
constexpr int MAX_CHANNELS = 256;  // input rows are staged 32 positions x C channels at a time
constexpr float LOG2E_F = 1.44269504088896340736f;

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

__device__ __forceinline__ f32x4 load4(const float *ptr) { return *reinterpret_cast<const f32x4 *>(ptr); }

// A wave's 16 rows of 16 PIECES values, loaded in whole lines (eight rows of 32 values a load), put into operand order: the
// four values 16 i + 4 g of row r for lane r + 16 g, through 2 KB of the LDS that are the wave's own.  (Loaded in operand
// order, a 16-byte piece of another row in every lane, each load takes the address path some 50 cycles instead of 16.)
template <int PIECES>
__device__ __forceinline__ void load_rows(f32x4 (&w)[PIECES], const float *rows, int64_t ld, int lane)
{
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        w[i] = load4(rows + (int64_t)((lane >> 3) + 8 * (i & 1)) * ld + 32 * (i / 2) + 4 * (lane & 7));
    }
}
template <int PIECES>
__device__ __forceinline__ void to_operand_order(f32x4 (&w)[PIECES], float *own, int lane)
{
    const auto slot = [](int row, int piece) { return 4 * (8 * row + (piece ^ ((row >> 1) & 7))); }; // 16 rows' in 16 bank groups
#pragma unroll
    for (int i = 0; i < PIECES; i += 2) {
        *reinterpret_cast<f32x4 *>(own + slot(lane >> 3, lane & 7)) = w[i];
        *reinterpret_cast<f32x4 *>(own + slot(8 + (lane >> 3), lane & 7)) = w[i + 1];
        w[i] = load4(own + slot(lane & 15, lane >> 4));
        w[i + 1] = load4(own + slot(lane & 15, 4 + (lane >> 4)));
    }
}

// the four lanes that hold one query's keys: l, l ^ 16, l ^ 32, l ^ 48
__device__ __forceinline__ float quad_max(float x)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    const float y = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(y), __float_as_uint(y), false, false);
    return fmaxf(__uint_as_float(q[0]), __uint_as_float(q[1]));
}
__device__ __forceinline__ float quad_sum(float x)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    const float y = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(y), __float_as_uint(y), false, false);
    return __uint_as_float(q[0]) + __uint_as_float(q[1]);
}

struct Fp32Params {
    const float *x, *wq, *wk, *wv, *wg, *bg, *bias, *nb;
    float *avg;
    int64_t x_ld, bias_sb, nb_sh, nb_sq, avg_sb, avg_ss, avg_sh;
    int S, H;
    int parts; // workgroups that share a head's queries
    float scale;
};

// PIECES: C / 16, the 16-channel pieces of a row, of which a lane holds four channels each
template <int PIECES>
__global__ __launch_bounds__(512, 2) void fp32_head_kernel(Fp32Params p)
{
    extern __shared__ float lds_f[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 15, g = lane >> 4;
    constexpr int C = 16 * PIECES;
    const int S = p.S, NB = (S + 31) / 32, S32 = NB * 32;
    // neighbouring workgroups, dealt to different XCDs, take different heads: with eight each L2 holds one head's weights
    const int h = blockIdx.x % p.H, rest = blockIdx.x / p.H;
    const int part = rest % p.parts, b = rest / p.parts;
    const int t_lo = NB * part / p.parts, t_hi = NB * (part + 1) / p.parts; // query tiles of this workgroup
    const int XP = C + 4, VP = S32 + 4; // odd multiples of 16 bytes, as LDP

    float *xs = lds_f;             // [32][XP]
    float *ks = xs + 32 * XP;      // [S32][LDP]
    float *qs = ks + S32 * LDP;    // [S32][LDP], scaled by 1/sqrt(d)
    float *gs = qs + S32 * LDP;    // [S32][LDP], sigmoid applied
    float *vt = gs + S32 * LDP;    // [32][VP], transposed
    float *ms = vt + HEAD * VP;    // [S32] mask bias, -inf past S

    // ---- projections: waves w and w + 4 share a SIMD, so they take different matrices: where the queries are shared out,
    // every SIMD has one of k, v (all positions) and one of q, gate (this workgroup's) ----
    const int half = wave >> 2, mat = (wave + 2 * half) & 3; // 0 k, 1 v, 2 q, 3 gate
    const float *wmat = mat == 0 ? p.wk : mat == 1 ? p.wv : mat == 2 ? p.wq : p.wg;
    // the next 32 positions wait in registers while the staged ones are used
    const float *xb = p.x + (int64_t)b * S * p.x_ld;
    constexpr int c4 = C / 4, pieces = 32 * c4, LOADS = (pieces + 511) / 512;
    f32x4 xr[LOADS];
    int xrow_i[LOADS], xcol[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int idx = tid + 512 * i < pieces ? tid + 512 * i : pieces - 1;
        xrow_i[i] = idx / c4;
        xcol[i] = 4 * (idx % c4);
    }
    const auto fetch = [&](int t) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int pos = t * 32 + xrow_i[i] < S ? t * 32 + xrow_i[i] : S - 1;
            xr[i] = load4(xb + (int64_t)pos * p.x_ld + xcol[i]);
        }
    };
    fetch(0);
    f32x4 w[PIECES];
    load_rows<PIECES>(w, wmat + (int64_t)(h * HEAD + 16 * half) * C, C, lane);
    f32x4 start = {0.f, 0.f, 0.f, 0.f};
    if (mat == 3) {
        start = *reinterpret_cast<const f32x4_any *>(p.bg + h * HEAD + 16 * half + 4 * g);
    }
    const float mask = tid < S ? p.bias[(int64_t)b * p.bias_sb + tid] : -INFINITY;
    // four keys' pair bias of query q0 + r; a step's is requested one step ahead, the first one's before the projections
    const auto pair_bias = [&](int q0, int key0) {
        f32x4 nv = {0.f, 0.f, 0.f, 0.f};
        if (p.nb != nullptr) {
            const float *nbrow = p.nb + (int64_t)h * p.nb_sh + (int64_t)(q0 + r < S ? q0 + r : S - 1) * p.nb_sq;
            if (key0 + 4 <= S) {
                nv = *reinterpret_cast<const f32x4_any *>(nbrow + key0);
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    nv[c] = key0 + c < S ? nbrow[key0 + c] : 0.f;
                }
            }
        }
        return nv;
    };
    const int q_first = 32 * t_lo + 16 * wave, q_end = 32 * t_hi < S ? 32 * t_hi : S;
    f32x4 next0 = pair_bias(q_first, 4 * g), next1 = pair_bias(q_first, 16 + 4 * g);
    to_operand_order<PIECES>(w, lds_f + 512 * wave, lane); // on the arrays, which are empty still
    if (tid < S32) {
        ms[tid] = mask;
    }
    for (int t = 0; t < NB; ++t) {
        __syncthreads(); // the weights' places, or the previous tile, have been read
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            if (tid + 512 * i < pieces) {
                *reinterpret_cast<f32x4 *>(xs + xrow_i[i] * XP + xcol[i]) = xr[i];
            }
        }
        __syncthreads();
        if (t + 1 < NB) {
            fetch(t + 1);
        }
        if (mat >= 2 && (t < t_lo || t >= t_hi)) {
            continue;
        }
        f32x4 acc[2] = {start, start}; // positions 0-15 and 16-31 of the tile
        const float *xrow = xs + r * XP + 4 * g;
        const auto project = [&](auto transposed, auto units) { // D[position][feature] for v, D[feature][position] for the others
#pragma unroll
            for (int i = 0; i < PIECES; ++i) {
                f32x4 xa[2];
#pragma unroll
                for (int u = 0; u < units; ++u) {
                    xa[u] = load4(xrow + 16 * u * XP + 16 * i);
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
#pragma unroll
                    for (int u = 0; u < units; ++u) {
                        acc[u] = transposed ? mfma_f32(xa[u][j], w[i][j], acc[u]) : mfma_f32(w[i][j], xa[u][j], acc[u]);
                    }
                }
            }
        };
        using One = std::integral_constant<int, 1>;
        using Two = std::integral_constant<int, 2>;
        const bool full = t * 32 + 16 < S; // else the second half's keys and values are zero, and their mask -inf
        if (mat == 1) {
            full ? project(std::true_type{}, Two{}) : project(std::true_type{}, One{});
        } else {
            full ? project(std::false_type{}, Two{}) : project(std::false_type{}, One{});
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int pos0 = t * 32 + 16 * u;
            if (mat == 1) {
                *reinterpret_cast<f32x4 *>(vt + (16 * half + r) * VP + pos0 + 4 * g) = acc[u];
                continue;
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                acc[u][v] = mat == 2   ? acc[u][v] * p.scale
                            : mat == 3 ? 1.0f / (1.0f + __builtin_amdgcn_exp2f(-acc[u][v] * LOG2E_F))
                                       : acc[u][v];
            }
            *reinterpret_cast<f32x4 *>((mat == 0 ? ks : mat == 2 ? qs : gs) + (pos0 + r) * LDP + 16 * half + 4 * g) = acc[u];
        }
    }
    __syncthreads();

    // ---- attention: 16 queries per wave at a time, 32 keys per step ----
    for (int q0 = q_first; q0 < q_end; q0 += 128) {
        const int qpos = q0 + r;
        const f32x4 qop0 = load4(qs + qpos * LDP + 4 * g), qop1 = load4(qs + qpos * LDP + 16 + 4 * g);
        float m_run = -INFINITY, lsum = 0.f;
        f32x4 o0 = {0.f, 0.f, 0.f, 0.f}, o1 = o0;
        for (int kt = 0; kt < NB; ++kt) {
            const f32x4 nv0 = next0, nv1 = next1;
            if (kt + 1 < NB) {
                next0 = pair_bias(q0, 32 * kt + 32 + 4 * g);
                next1 = pair_bias(q0, 32 * kt + 48 + 4 * g);
            } else if (q0 + 128 < q_end) {
                next0 = pair_bias(q0 + 128, 4 * g);
                next1 = pair_bias(q0 + 128, 16 + 4 * g);
            }
            // logits^T: rows = keys, columns = queries
            const float *krow = ks + (32 * kt + r) * LDP + 4 * g;
            const f32x4 k00 = load4(krow), k01 = load4(krow + 16), k10 = load4(krow + 16 * LDP), k11 = load4(krow + 16 * LDP + 16);
            f32x4 x0 = {0.f, 0.f, 0.f, 0.f}, x1 = x0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                x0 = mfma_f32(k00[j], qop0[j], x0);
                x1 = mfma_f32(k10[j], qop0[j], x1);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                x0 = mfma_f32(k01[j], qop1[j], x0);
                x1 = mfma_f32(k11[j], qop1[j], x1);
            }
            // (logit * scale + bias[b, k]) + nb[h, q, k], in that order (reference :109-118)
            const f32x4 mv0 = load4(ms + 32 * kt + 4 * g), mv1 = load4(ms + 32 * kt + 16 + 4 * g);
            float mx = -INFINITY;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                x0[c] = (x0[c] + mv0[c]) + nv0[c];
                x1[c] = (x1[c] + mv1[c]) + nv1[c];
                mx = fmaxf(mx, fmaxf(x0[c], x1[c]));
            }
            mx = quad_max(mx);
            const float m_new = fmaxf(m_run, mx); // finite: every tile has a key below S, whose bias is finite
            const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * LOG2E_F);
            m_run = m_new;
            float psum = 0.f;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                x0[c] = __builtin_amdgcn_exp2f((x0[c] - m_new) * LOG2E_F);
                x1[c] = __builtin_amdgcn_exp2f((x1[c] - m_new) * LOG2E_F);
                psum += x0[c] + x1[c];
                o0[c] *= alpha;
                o1[c] *= alpha;
            }
            lsum = lsum * alpha + psum;
            // O^T += V^T . P^T: k-step j takes the keys 4 g + j that register j holds
            const float *vrow = vt + r * VP + 32 * kt + 4 * g;
            const f32x4 v00 = load4(vrow), v01 = load4(vrow + 16), v10 = load4(vrow + 16 * VP), v11 = load4(vrow + 16 * VP + 16);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                o0 = mfma_f32(v00[j], x0[j], o0);
                o1 = mfma_f32(v10[j], x0[j], o1);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                o0 = mfma_f32(v01[j], x1[j], o0);
                o1 = mfma_f32(v11[j], x1[j], o1);
            }
        }
        const float inv = 1.0f / quad_sum(lsum);
        if (qpos < S) { // register c of o0 is head dim 4 g + c, of o1 16 + 4 g + c
            float *out = p.avg + (int64_t)b * p.avg_sb + (int64_t)qpos * p.avg_ss + (int64_t)h * p.avg_sh + 4 * g;
            const f32x4 g0 = load4(gs + qpos * LDP + 4 * g), g1 = load4(gs + qpos * LDP + 16 + 4 * g);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                o0[c] = o0[c] * inv * g0[c];
                o1[c] = o1[c] * inv * g1[c];
            }
            *reinterpret_cast<f32x4 *>(out) = o0;
            *reinterpret_cast<f32x4 *>(out + 16) = o1;
        }
    }
}

// out[m, n] = sum_k a[m, k] * w[n, k] + bias[n] over 16 PIECES k.  A workgroup keeps 64 rows of w, 16 a wave, in registers and walks
// tiles of 16 rows of a, which lie in the LDS for its four waves; the next tile's wait in registers meanwhile.  Rows of a and
// w are 16-byte aligned.
template <int PIECES>
__global__ __launch_bounds__(256, 2) void fp32_rows_gemm_kernel(const float *__restrict__ a, int64_t a_ld, const float *__restrict__ w,
                                                                const float *__restrict__ bias, float *__restrict__ out,
                                                                int64_t out_ld, int64_t M, int N)
{
    constexpr int K = 16 * PIECES, AP = K + 4, LOADS = (4 * K + 255) / 256;
    __shared__ __attribute__((aligned(16))) float rows[16 * AP], own[4][512];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int n0 = (blockIdx.y * 4 + wave) * 16;
    const bool live = n0 < N; // N is a multiple of 32
    f32x4 av[LOADS], wv[PIECES];
    const auto fetch = [&](int64_t m0) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int idx = tid + 256 * i < 4 * K ? tid + 256 * i : 4 * K - 1;
            const int64_t row = m0 + idx / (K / 4) < M ? m0 + idx / (K / 4) : M - 1;
            av[i] = load4(a + row * a_ld + 4 * (idx % (K / 4)));
        }
    };
    fetch((int64_t)blockIdx.x * 16);
    f32x4 bv = {0.f, 0.f, 0.f, 0.f};
    if (live) {
        load_rows<PIECES>(wv, w + (int64_t)n0 * K, K, lane);
        if (bias != nullptr) {
            bv = *reinterpret_cast<const f32x4_any *>(bias + n0 + 4 * g);
        }
        to_operand_order<PIECES>(wv, own[wave], lane);
    }
    for (int64_t m0 = (int64_t)blockIdx.x * 16; m0 < M; m0 += (int64_t)gridDim.x * 16) {
        if (m0 != (int64_t)blockIdx.x * 16) {
            __syncthreads(); // the previous tile has been read
        }
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int idx = tid + 256 * i;
            if (idx < 4 * K) {
                *reinterpret_cast<f32x4 *>(rows + idx / (K / 4) * AP + 4 * (idx % (K / 4))) = av[i];
            }
        }
        __syncthreads();
        if (m0 + (int64_t)gridDim.x * 16 < M) {
            fetch(m0 + (int64_t)gridDim.x * 16);
        }
        if (live) {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f}; // D[output feature][row]
#pragma unroll
            for (int i = 0; i < PIECES; ++i) {
                const f32x4 x = load4(rows + r * AP + 16 * i + 4 * g);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    acc = mfma_f32(wv[i][e], x[e], acc);
                }
            }
            if (m0 + r < M) {
                *reinterpret_cast<f32x4_any *>(out + (m0 + r) * out_ld + n0 + 4 * g) = acc + bv;
            }
        }
    }
}

inline bool aligned16(const void *ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0; }

size_t head_kernel_lds(int S, int C)
{
    const int S32 = (S + 31) / 32 * 32;
    return (size_t)(32 * (C + 4) + 3 * S32 * LDP + HEAD * (S32 + 4) + S32) * sizeof(float);
}

template <int PIECES>
int launch(const kutacc_hip_attention_args_t &a, const Fp32Params &p, hipStream_t stream)
{
    constexpr int C = 16 * PIECES;
    const size_t lds_bytes = head_kernel_lds(p.S, C);
    static size_t configured[KUTACC_DEVICE_SLOTS] = {};
    const hipError_t e = kutacc_opt_in_lds(reinterpret_cast<const void *>(fp32_head_kernel<PIECES>), lds_bytes, configured);
    if (e != hipSuccess) {
        return (int)e;
    }
    const double BS = (double)a.batch * (double)a.seq_len;
    {
        kutacc_prof::KernelTimer t("fp32_head_kernel", 8.0 * BS * C * C + 4.0 * BS * (double)a.seq_len * C, stream);
        fp32_head_kernel<PIECES><<<dim3((unsigned)(a.batch * a.nheads * p.parts)), 512, lds_bytes, stream>>>(p);
        const int rc = kutacc_hip_status(hipGetLastError());
        if (rc != 0) {
            return rc;
        }
    }
    const int64_t M = a.batch * a.seq_len;
    kutacc_prof::KernelTimer t("fp32_rows_gemm_kernel", 2.0 * BS * C * C, stream);
    const int64_t columns = (C + 63) / 64, cap = GEMM_WORKGROUPS_PER_CU * (int64_t)kutacc_cu_count() / columns;
    const dim3 grid((unsigned)std::min<int64_t>((M + 15) / 16, std::max<int64_t>(cap, 1)), (unsigned)columns);
    fp32_rows_gemm_kernel<PIECES><<<grid, 256, 0, stream>>>((const float *)a.avg, a.avg_stride_s, (const float *)a.output_w,
                                                            a.output_b, (float *)a.out, a.out_ld, M, C);
    return kutacc_hip_status(hipGetLastError());
}

} // namespace

namespace kutacc_launch {

bool fp32_attention_supports(const kutacc_hip_attention_args_t &a)
{
    if (a.dtype != KUTACC_DTYPE_FP32 || a.head_size != HEAD || a.batch <= 0 || a.seq_len <= 0 || a.seq_len > MAX_SEQ) {
        return false;
    }
    const int64_t C = a.nheads * a.head_size;
    if (C > MAX_CHANNELS || a.batch * a.nheads > INT32_MAX || a.batch * a.seq_len > INT32_MAX) {
        return false;
    }
    // 16-byte loads of input and weight rows, 16-byte stores of the gated average
    if (a.input_ld % 4 != 0 || a.avg_stride_b % 4 != 0 || a.avg_stride_s % 4 != 0 || a.avg_stride_h % 4 != 0 || !aligned16(a.input) ||
        !aligned16(a.query_w) || !aligned16(a.key_w) || !aligned16(a.value_w) || !aligned16(a.gating_w) || !aligned16(a.output_w) ||
        !aligned16(a.avg)) {
        return false;
    }
    // the output projection reads the gated average as [batch * seq_len] rows of C values
    return a.avg_stride_h == HEAD && a.avg_stride_b == a.seq_len * a.avg_stride_s && a.avg_stride_s >= C;
}

int gating_attention_fp32(const kutacc_hip_attention_args_t &a, hipStream_t stream)
{
    if (!fp32_attention_supports(a)) {
        return KUTACC_HIP_EUNSUPPORTED;
    }
    Fp32Params p;
    p.x = (const float *)a.input, p.wq = (const float *)a.query_w, p.wk = (const float *)a.key_w, p.wv = (const float *)a.value_w;
    p.wg = (const float *)a.gating_w, p.bg = a.gating_b, p.bias = (const float *)a.bias, p.nb = (const float *)a.nonbatched_bias;
    p.avg = (float *)a.avg;
    p.x_ld = a.input_ld, p.bias_sb = a.bias_stride_b, p.nb_sh = a.nb_stride_h, p.nb_sq = a.nb_stride_q;
    p.avg_sb = a.avg_stride_b, p.avg_ss = a.avg_stride_s, p.avg_sh = a.avg_stride_h;
    p.S = (int)a.seq_len, p.H = (int)a.nheads;
    // With fewer heads than CUs a head's queries go to several workgroups, each of which forms all keys and values: the
    // projections of a workgroup shrink towards half, on CUs that were idle (16 rows x 64
    // positions x 8 heads 24.0 us unshared, 22.3 shared; 4 x 64 x 4 heads 15.6 and 14.5).
    const int64_t heads = a.batch * a.nheads, tiles = (a.seq_len + 31) / 32;
    p.parts = (int)std::max<int64_t>(1, std::min<int64_t>(tiles, kutacc_cu_count() / heads));
    p.scale = (float)(1.0 / sqrt((double)a.head_size)); // reference gating_attention.cpp:68
    switch (a.nheads) {
    case 1: return launch<2>(a, p, stream);
    case 2: return launch<4>(a, p, stream);
    case 3: return launch<6>(a, p, stream);
    case 4: return launch<8>(a, p, stream);
    case 5: return launch<10>(a, p, stream);
    case 6: return launch<12>(a, p, stream);
    case 7: return launch<14>(a, p, stream);
    default: return launch<16>(a, p, stream);
    }
}

} // namespace kutacc_launch
