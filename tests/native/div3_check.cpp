// The shadow filter's x / 3 through the reciprocal (div3_unit of
// vpt_short_math.h) compared with the IEEE division for every float x in
// [+0, 2] (subnormals included).  Prints the number of mismatches and exits
// non-zero if there is one.
#include <cstdio>

#include "vpt_short_math.h"

int main()
{
    long bad = 0;
    for (uint32_t u = 0; u <= 0x40000000u; u++) {
        const float x = vpt_u2f(u), q = vpt::div3_unit(x), e = x / 3.0f;
        if (vpt_f2u(q) != vpt_f2u(e) && bad++ < 5) printf("x=%a fast=%a ieee=%a\n", x, q, e);
    }
    printf("%ld mismatches\n", bad);
    return bad != 0;
}
