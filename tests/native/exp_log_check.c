/* The denoisers' short forms of vpt_expf, vpt_logf and x / 5 against the full
 * ones, as vpt_svgf.hip computes them (expf_32, expf_down, logf_unit, div_rcp):
 *   - exp for x in [-32, 0], and with the clamp at -88 and the cut at -87.34
 *     for every x <= 0: one fma for x - k LN2_HI (the product is exact) and
 *     one ldexp for the scaling.  Every 11th float.
 *   - log for every x in (0.5, 1).  The device's quotient (m - 1) / (m + 1)
 *     is compared with the division on the device.
 *   - x / 5 for every mantissa, at exponents -60, 0 and 60.
 * Prints the number of mismatches and exits non-zero if there is one. */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include "vpt/vpt_numerics.h"

static float exp_32(float x)
{
    const float kf = floorf(x * 1.44269502162933349609375f + 0.5f);
    float r = fmaf(-kf, 0.693145751953125f, x);
    float p = 0.0013829420786350965f;
    r = r - kf * 1.428606765330187045e-06f;
    p = p * r + 0.008374771103262901f;
    p = p * r + 0.0416683591902256f;
    p = p * r + 0.1666642129421234f;
    p = p * r + 0.49999991059303284f;
    p = p * r + 1.0f;
    p = p * r + 1.0f;
    return ldexpf(p, (int)kf);
}

static float exp_down(float x) { return x < -87.33654022216796875f ? 0.0f : exp_32(fmaxf(x, -88.0f)); }

static float log_unit(float x)
{
    const int low = x + x <= 1.41421353816986083984375f;
    const float m = low ? x + x : x, fe = low ? -1.0f : 0.0f;
    const float s = (m - 1.0f) / (m + 1.0f), s2 = s * s;
    float p = 0.111111111111f, lm;
    p = p * s2 + 0.142857142857f;
    p = p * s2 + 0.2f;
    p = p * s2 + 0.333333333333f;
    lm = (s + s) + (s + s) * (s2 * p);
    return fe * 0.693145751953125f + (fe * 1.428606765330187045e-06f + lm);
}

static float div_5(float a)
{
    const float y = 1.0f / 5.0f, q0 = a * y, q = fmaf(fmaf(-5.0f, q0, a), y, q0);
    return q0 == 0.0f ? q0 : q;
}

static long bad;

static void same(const char* what, float x, float fast, float full)
{
    uint32_t a, b;
    memcpy(&a, &fast, 4);
    memcpy(&b, &full, 4);
    if (a != b && bad++ < 5) printf("%s x=%a fast=%a full=%a\n", what, x, fast, full);
}

int main(void)
{
    uint32_t u;
    float x;
    int e;
    for (u = 0x80000000u; u <= 0xff800000u; u += 11u) {   /* -0 down to -inf */
        memcpy(&x, &u, 4);
        same("exp_down", x, exp_down(x), vpt_expf(x));
        if (x >= -32.0f) same("exp_32", x, exp_32(x), vpt_expf(x));
    }
    for (u = 0x3f000001u; u < 0x3f800000u; u++) {
        memcpy(&x, &u, 4);
        same("log_unit", x, log_unit(x), vpt_logf(x));
    }
    for (e = -60; e <= 60; e += 60)
        for (u = 0; u < 0x800000u; u++) {
            const uint32_t v = ((uint32_t)(127 + e) << 23) | u;
            memcpy(&x, &v, 4);
            same("div_5", x, div_5(x), x / 5.0f);
        }
    printf("%ld mismatches\n", bad);
    return bad != 0;
}
