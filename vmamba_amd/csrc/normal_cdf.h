// The normal distribution function in single precision, which exact GELU is made of: GELU(x) = x Phi(x), GELU'(x) = Phi(x) + x phi(x).
#pragma once

#include "ss2d_common.h"

namespace ss2d {

// Phi(x), and exp(-x^2 / 2) in `e`.  Two least-squares fits with weights driven to an even relative error, their coefficients rounded to fp32 from
// the leading one on, each time with the others fitted again:
//   |x| < 1.1   0.5 + x P(x^2), degree 5 (4e-9 of the smaller of Phi and 1 - Phi): near 0 nothing but the last rounding is lost;
//   beyond      1 - Phi(|x|) = exp(-x^2 / 2) Q(1 / (1 + 0.38 |x|)), degree 7 (3e-8, up to |x| = 14; from 13.2 on the exponential is 0).
// One fit of degree 9 for all x has 1.4 times the error of 0.5 (1 + erff(x / sqrt 2)) over a normal x, three times near 0.  Against float64, rms, this /
// the erff form with erff rounded correctly: GELU over a normal x 2.2e-8 / 2.4e-8, GELU' 2.5e-8 / 2.6e-8, within 0.01 1.1e-10 / 1.1e-10 and 2.2e-8 / 2.2e-8,
// in (-4, -3) 3.6e-10 / 3.0e-8 and 1.1e-9 / 8.6e-9; no range in steps of a half is worse.
__device__ __forceinline__ float normal_cdf(float x, float &e) {
    const float xx = x * x, t = __builtin_amdgcn_rcpf(fmaf(0.38f, fabsf(x), 1.0f));
    e = __builtin_amdgcn_exp2f(xx * -0.72134752044448170f);
    float q = 0.06340273f;
    q = fmaf(q, t, -0.20329623f);
    q = fmaf(q, t, 0.16641408f);
    q = fmaf(q, t, 0.027755821f);
    q = fmaf(q, t, 0.14480415f);
    q = fmaf(q, t, 0.14923643f);
    q = fmaf(q, t, 0.15180245f);
    q = fmaf(q, t, -7.5026933e-06f);
    float p = -6.80655e-06f;
    p = fmaf(p, xx, 0.00011091021f);
    p = fmaf(p, xx, -0.0011834479f);
    p = fmaf(p, xx, 0.00997189f);
    p = fmaf(p, xx, -0.06649006f);
    p = fmaf(p, xx, 0.39894226f);
    const float tail = e * q;
    return fabsf(x) < 1.1f ? fmaf(x, p, 0.5f) : x < 0.0f ? tail : 1.0f - tail;
}

}  // namespace ss2d
