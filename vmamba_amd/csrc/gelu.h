// Exact (erf) GELU for 16-bit activations, shared by the kernels that fuse it.
//   * bf16: the argument is a bf16 value, so gelu(x) = 0.5 x + |x| E(|x|), E(x) = 0.5 erf(x / sqrt 2), with E read from
//     a 2176-entry fp32 table (copied into LDS by the kernel) indexed by the bf16 bit pattern clamped to [2^-14, 8)
//     (below, |x| E is under 1e-4 of 0.5 |x|; above, E is 0.5 to fp32 precision).  The table is generated in double
//     precision at build time (gen_gelu_table.py);
//   * fp16: x Phi(x) with 1 - Phi(|x|) = exp(-x^2 / 2) (1/2 - |x| t S(t)), t = 1 / (1 + 0.34 |x|), a least-squares fit of degree 6 in S: a relative
//     error of 6e-7, so that large negative x keeps its digits, and nothing but roundings near 0.  Of all fp16 arguments in (-8, -4], (-4, -3], (-3, -2],
//     (-1, 1] 0, 0, 0 and 2 results are another neighbour than the exact value's; with 0.5 x (1 + erff) 275, 50, 2 and 0, with Abramowitz-Stegun 7.1.26
//     (absolute error 1.5e-7, an instruction or two less) 285, 155, 12 and 5.  The two are one argument, 0.0013, whose exact GELU lies 4.2e-8 of itself from
//     the middle of two neighbours.  normal_cdf leaves none there, and made 384 -> 1536 at 25 088 positions 79 us where this and 7.1.26 take 69.
#pragma once

#include "ss2d_common.h"

namespace ss2d {

#include "gelu_table.inc"

constexpr int kGeluEntries = kGeluHiBits - kGeluLoBits;

__device__ __forceinline__ float gelu_half(float x) {
    const float t = __builtin_amdgcn_rcpf(fmaf(0.34f, fabsf(x), 1.0f));
    float q = 0.015613869f;
    q = fmaf(q, t, -0.054586105f);
    q = fmaf(q, t, 0.03962224f);
    q = fmaf(q, t, 0.024110418f);
    q = fmaf(q, t, 0.08061656f);
    q = fmaf(q, t, 0.12354839f);
    q = fmaf(q, t, 0.17001599f);
    q = fmaf(-fabsf(x), q * t, 0.5f);
    const float tail = __builtin_amdgcn_exp2f(x * x * -0.72134752044448170f) * q;
    return x * (x < 0.0f ? tail : 1.0f - tail);
}

// GELU of two packed 16-bit values, result packed and rounded again; tbl: the table in LDS (bf16 only)
__device__ __forceinline__ uint32_t gelu_pair(bf16_t, uint32_t w, const float *tbl) {
    const uint32_t a0 = w & 0x7fffu, a1 = (w >> 16) & 0x7fffu;
    const uint32_t m0 = min(max(a0, (uint32_t)kGeluLoBits), (uint32_t)kGeluHiBits - 1u) - kGeluLoBits;
    const uint32_t m1 = min(max(a1, (uint32_t)kGeluLoBits), (uint32_t)kGeluHiBits - 1u) - kGeluLoBits;
    const float e0 = tbl[m0], e1 = tbl[m1];
    const float x0 = bits_to_f32(w << 16), x1 = bits_to_f32(w & 0xffff0000u);
    return pack2_from_f32<bf16_t>(fmaf(fabsf(x0), e0, 0.5f * x0), fmaf(fabsf(x1), e1, 0.5f * x1));
}
__device__ __forceinline__ uint32_t gelu_pair(f16_t, uint32_t w, const float *) {
    return pack2_from_f32<f16_t>(gelu_half(unpack_lo<f16_t>(w)), gelu_half(unpack_hi<f16_t>(w)));
}

}  // namespace ss2d
