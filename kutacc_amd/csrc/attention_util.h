// Pieces of the attention loops (log2 units, head size 32).
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "mfma_tiles.h"

namespace kutacc_dev {

// A operand of the row-sum MFMA (16x16x32: lane -> row lane&15, k-chunk lane>>4).  The B operand is a
// probability fragment of the 32x32x16 layout (lane -> query lane&31, 8 keys of half lane>>5), which the
// 16x16x32 shape reads as column lane&15, k-chunk lane>>4: chunks 0 and 2 belong to query n, chunks 1 and
// 3 to query n+16.  Row 0 of A therefore sums chunks 0 and 2, row 1 chunks 1 and 3; the sums of
// queries n and n+16 end up in lane n, accumulator registers 0 and 1.
__device__ __forceinline__ bf16x8 rowsum_selector(int lane)
{
    const int i = lane & 15, c = lane >> 4;
    const float v = ((i == 0 && (c & 1) == 0) || (i == 1 && (c & 1) == 1)) ? 1.0f : 0.0f;
    bf16x8 a;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        a[e] = (bf16_t)v;
    }
    return a;
}

__device__ __forceinline__ float rowsum_fetch(const f32x4 &lacc, int lane)
{
    const int q = lane & 31;
    const int src = (q & 15) * 4;
    const float a0 = __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(lacc[0])));
    const float a1 = __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(lacc[1])));
    return (q >> 4) ? a1 : a0;
}

// The mask bias of a key as two bf16, v = hi + lo to 2^-17 of |v|: the k-slots 0 and 1 of the A operand of the MFMA that adds a
// row's masks to its logits.  -inf: hi = -inf, lo = 0.
__device__ __forceinline__ uint32_t mask_word(float mv)
{
    const bf16_t hi = (bf16_t)mv;
    const float hf = to_f32(hi);
    const float rest = (hf == mv || !(fabsf(hf) < INFINITY)) ? 0.f : mv - hf; // a NaN stays one through hi
    bf16x2 pair;
    pair[0] = hi, pair[1] = (bf16_t)rest;
    return __builtin_bit_cast(uint32_t, pair);
}

__device__ __forceinline__ float mask_word_value(uint32_t w)
{
    return __uint_as_float(w << 16) + __uint_as_float(w & 0xffff0000u);
}

// avg[b, q, h, :] = O / l * gate for the 32 queries of one block; gate values in accumulator order
__device__ __forceinline__ void store_gated(bf16_t *dst, const f32x16 &o, float inv, const f32x16 &gate)
{
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        bf16x4 ov;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            ov[c] = (bf16_t)(o[4 * a + c] * inv * gate[4 * a + c]);
        }
        *reinterpret_cast<bf16x4 *>(dst + 8 * a) = ov;
    }
}

} // namespace kutacc_dev
