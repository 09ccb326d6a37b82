// The denoisers' short forms of vpt_expf, vpt_logf and of divisions: fewer
// instructions for the arguments that arise there, the same results.  Host
// and device, so that tests/native compares this code with the full forms
// (compile with -ffp-contract=off; fmaf is one rounding on both sides).
#pragma once

#include <math.h>
#include <stdint.h>

#include "vpt/vpt_numerics.h"

namespace vpt {

// vpt_expf for -32 <= x <= 0: the same polynomial; kf has at most seven bits
// (for x down to -88) and LN2_HI eight, so their product is exact and the
// subtraction one fma; the scaling by 2^k, k >= -46, is exact in one step.
VPT_HD float expf_32(float x)
{
    const float LOG2E = 1.44269502162933349609375f;
    const float LN2_HI = 0.693145751953125f;
    const float LN2_LO = 1.428606765330187045e-06f;
    const float kf = floorf(x * LOG2E + 0.5f);
    float r = __builtin_fmaf(-kf, LN2_HI, x);
    r = r - kf * LN2_LO;
    float p = 0.0013829420786350965f;
    p = p * r + 0.008374771103262901f;
    p = p * r + 0.0416683591902256f;
    p = p * r + 0.1666642129421234f;
    p = p * r + 0.49999991059303284f;
    p = p * r + 1.0f;
    p = p * r + 1.0f;
    return __builtin_ldexpf(p, (int)kf);
}

// vpt_expf for x <= 0, where it is 0 below -87.34; above, p 2^k is rounded at
// most once, in either form of the scaling.
VPT_HD float expf_down(float x)
{
    const float e = expf_32(fmaxf(x, -88.0f));
    return x < -87.33654022216796875f ? 0.0f : e;
}

// a / b given y = 1 / b (the correctly rounded reciprocal), for quotients
// that are zero or normal with an exactly representable remainder, which is
// the case for every weighted mean and weight ratio of the denoisers: q0 = a
// y lies within an ulp of a / b, the remainder a - b q0 is exact in an fma,
// and q0 + (a - b q0) y rounded once is the correctly rounded quotient
// (Markstein, IBM J. Res. Dev. 34(1), 1990).  A zero q0 is returned as is,
// keeping the sign that the correction's addition would drop.  Three VALU
// operations and a select per quotient, against about ten for a division,
// where several quotients share a divisor.
VPT_HD float div_rcp(float a, float b, float y)
{
    const float q0 = a * y;
    const float q = __builtin_fmaf(__builtin_fmaf(-b, q0, a), y, q0);
    return q0 == 0.0f ? q0 : q;
}

// x / 3 for 0 <= x <= 2: q0 = x fl(1/3), then one correction with the exact
// remainder x - 3 q0 (an fma).  Equal to the IEEE division for every float
// in [0, 2], subnormals included (tests/test_exact_division_cpu.py checks
// all of them); three VALU operations in place of the division's ten.
VPT_HD float div3_unit(float x)
{
    const float y = 1.0f / 3.0f;
    const float q0 = x * y;
    return __builtin_fmaf(__builtin_fmaf(-3.0f, q0, x), y, q0);
}

// vpt_logf for x in (1/2, 1): the same operations without the cases that
// cannot arise there.  x = m 2^e with m up to sqrt(2) (e = -1) or m = x (e =
// 0); the caller divides s = (m - 1) / (m + 1).
struct UnitLog {
    float m, e;
};

VPT_HD UnitLog log_unit_reduce(float x)
{
    const bool low = x + x <= 1.41421353816986083984375f;
    return UnitLog{low ? x + x : x, low ? -1.0f : 0.0f};
}

VPT_HD float log_unit_sum(float s, float e)
{
    const float LN2_HI = 0.693145751953125f;
    const float LN2_LO = 1.428606765330187045e-06f;
    float s2 = s * s;
    float p = 0.111111111111f;
    p = p * s2 + 0.142857142857f;
    p = p * s2 + 0.2f;
    p = p * s2 + 0.333333333333f;
    float lm = (s + s) + (s + s) * (s2 * p);
    return e * LN2_HI + (e * LN2_LO + lm);
}

}  // namespace vpt
