// The denoisers' short forms (vpt_short_math.h, the code that vpt_svgf.hip
// compiles) against the full ones:
//   - exp for x in [-32, -0], and with the clamp at -88 and the cut at -87.34
//     for x <= 0, whose results lie in [0, 1]: every float of magnitude 2^-26
//     to 128 and every 101st of the others (where exp is 1 or 0);
//   - log for every x in (0.5, 1), with the IEEE division for the quotient
//     (the device's is compared with the division on the device);
//   - x / 5 for every mantissa, at exponents -60, 0 and 60.
// Prints the number of mismatches and exits non-zero if there is one.
#include <atomic>
#include <cstdio>
#include <cstring>
#include <thread>
#include <vector>

#include "vpt_short_math.h"

static std::atomic<long> bad{0};

static void same(const char* what, float x, float fast, float full)
{
    if (vpt_f2u(fast) != vpt_f2u(full) && bad++ < 5) printf("%s x=%a fast=%a full=%a\n", what, x, fast, full);
}

int main()
{
    const uint32_t first = 0x80000000u, end = 0xff800001u;   // -0 down to -inf
    const uint32_t parts = 8;
    std::vector<std::thread> pool;
    for (uint32_t k = 0; k < parts; k++)
        pool.emplace_back([=] {
            for (uint32_t u = first + k; u < end; u += parts) {
                const uint32_t e = (u >> 23) & 0xffu;   // 101 and 134: 2^-26 and 128
                if ((e < 101u || e > 133u) && u % 101u) continue;
                const float x = vpt_u2f(u), full = vpt_expf(x);
                same("expf_down", x, vpt::expf_down(x), full);
                if (x >= -32.0f) same("expf_32", x, vpt::expf_32(x), full);
                if (!(full >= 0.0f && full <= 1.0f)) same("range", x, full, 0.0f);
            }
        });
    for (std::thread& t : pool) t.join();
    for (uint32_t u = 0x3f000001u; u < 0x3f800000u; u++) {
        const float x = vpt_u2f(u);
        const vpt::UnitLog r = vpt::log_unit_reduce(x);
        same("log_unit", x, vpt::log_unit_sum((r.m - 1.0f) / (r.m + 1.0f), r.e), vpt_logf(x));
    }
    for (int e = -60; e <= 60; e += 60)
        for (uint32_t u = 0; u < 0x800000u; u++) {
            const float x = vpt_u2f(((uint32_t)(127 + e) << 23) | u);
            same("div_rcp 5", x, vpt::div_rcp(x, 5.0f, 1.0f / 5.0f), x / 5.0f);
        }
    printf("%ld mismatches\n", bad.load());
    return bad != 0;
}
