// Small device-side helpers shared by the HIP translation units: storage-type loads/stores with
// the library's rounding rule (fp32 -> bf16 is round-to-nearest-even, bf16 -> fp32 is exact, as in
// reference src/wrapper/svcvt.h:23-37), wavefront reductions for 64-wide waves, error mapping.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kutacc_hip.h"

namespace kutacc_dev {

typedef __bf16 bf16_t;

__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ float to_f32(bf16_t v) { return (float)v; }

template <typename T>
__device__ __forceinline__ T from_f32(float v);
template <>
__device__ __forceinline__ float from_f32<float>(float v)
{
    return v;
}
template <>
__device__ __forceinline__ bf16_t from_f32<bf16_t>(float v)
{
    return (bf16_t)v; // v_cvt_pk_bf16_f32: round to nearest even
}

__device__ __forceinline__ float wave_max(float v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        v = fmaxf(v, __shfl_xor(v, off, 64));
    }
    return v;
}

__device__ __forceinline__ float wave_sum(float v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        v += __shfl_xor(v, off, 64);
    }
    return v;
}

// lane-group sums without LDS: a row spread over LPR consecutive lanes (LPR = 8, 16, 32 or 64)
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v)
{
    const int moved = __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false);
    return v + __int_as_float(moved);
}

// sum over the LPR lanes that hold one row; every lane of the group gets the total
template <int LPR>
__device__ __forceinline__ float group_sum(float v)
{
    v = dpp_add<0xB1>(v);  // quad_perm [1,0,3,2]: lane ^ 1
    v = dpp_add<0x4E>(v);  // quad_perm [2,3,0,1]: lane ^ 2
    v = dpp_add<0x141>(v); // row_half_mirror: pairs the two quads of 8 lanes
    if (LPR >= 16) {
        v = dpp_add<0x140>(v); // row_mirror: pairs the two halves of 16 lanes
    }
    if (LPR >= 32) {
        v += __shfl_xor(v, 16, 64);
    }
    if (LPR >= 64) {
        v += __shfl_xor(v, 32, 64);
    }
    return v;
}

// LayerNorm's scale and shift from a row's sum and sum of squares, both of x - x0 with x0 the row's first element: y = x * rstd + shift,
// then gamma and beta (reference src/normalization/layernorm_kernel.h:21-53).  ROUNDED: correctly rounded square root and quotient;
// otherwise the hardware's reciprocal square root (1 ulp), for rows of which every lane forms it: the two rounded operations
// expand to some 25 instructions per lane and row.
template <bool ROUNDED>
__device__ __forceinline__ void norm_from_sums(float s1, float s2, float x0, float n, float eps, float &rstd, float &shift)
{
    const float mean = s1 / n + x0;
    const float var = fmaxf((s2 - s1 * s1 / n) / n, 0.f);
    rstd = ROUNDED ? 1.0f / sqrtf(var + eps) : __builtin_amdgcn_rsqf(var + eps);
    shift = -rstd * mean;
}

// the same of one row held as 8 values per lane of LPR consecutive lanes; x0 = first element of the row
template <int LPR>
__device__ __forceinline__ void group_stats(const float (&x)[8], float x0, float n, float eps, float &rstd, float &shift)
{
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float v = x[e] - x0;
        s1 += v;
        s2 = fmaf(v, v, s2);
    }
    norm_from_sums<false>(group_sum<LPR>(s1), group_sum<LPR>(s2), x0, n, eps, rstd, shift);
}

__device__ __forceinline__ float sigmoid_f32(float x) { return 1.0f / (1.0f + __expf(-x)); }

// 1 / d rounded to nearest where it is a normal number: one Newton step on the hardware's reciprocal, which is within a unit of it
// (P. W. Markstein, Computation of elementary functions on the IBM RISC System/6000 processor, 1990).  The bits of 1.0f / d for
// every significand, in 3 instructions instead of some 10.
__device__ __forceinline__ float reciprocal(float d)
{
    const float r = __builtin_amdgcn_rcpf(d);
    return fmaf(fmaf(-d, r, 1.0f), r, r);
}

// sigmoid_f32 of N values, bit for bit
template <int N>
__device__ __forceinline__ void sigmoids_f32(float (&x)[N])
{
    float most = 0.f;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        x[i] = 1.0f + __expf(-x[i]);
        most = fmaxf(most, x[i]);
    }
    if (__any(most >= 0x1p126f)) { // below -87: the quotient is no normal number
#pragma unroll
        for (int i = 0; i < N; ++i) {
            x[i] = 1.0f / x[i];
        }
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            x[i] = reciprocal(x[i]);
        }
    }
}

} // namespace kutacc_dev
