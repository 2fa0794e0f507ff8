/* The reciprocals of the thermal strips (rcp_core, rcp_back in
 * geoflac_amd/csrc/gf_therm.h) against IEEE division on random operands.
 * rcp_core: two Newton steps and a remainder step from an estimate of 1/d, here 1/d with
 * a relative error of up to 2^-20 (the hardware's estimate is closer).  rcp_back:
 * a = RN(1/d), then 1/a by one Newton step from d.  Both for an operand (d, a) whose
 * significand is not all ones, which the kernel sends to the division.  Exponents stay in +-400.  Prints the mismatches of each. */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static uint64_t s = 88172645463325252ull;
static uint64_t rnd(void)
{
    s ^= s << 13;
    s ^= s >> 7;
    s ^= s << 17;
    return s;
}
static double rd(int k)
{
    uint64_t m = rnd() & 0xfffffffffffffull;
    if (k % 16 == 0) m = 0xfffffffffffffull - rnd() % 4; /* significands of (nearly) all ones */
    if (k % 16 == 1) m = rnd() % 4;
    uint64_t u = ((uint64_t)(1023 + (int)(rnd() % 800) - 400) << 52) | m | (rnd() << 63);
    double d;
    memcpy(&d, &u, 8);
    return d;
}
int main(int argc, char **argv)
{
    long n = argc > 1 ? atol(argv[1]) : 1000000, bad0 = 0, bad1 = 0;
    for (long k = 0; k < n; k++) {
        const double d = rd((int)(k & 15)), q = 1.0 / d;
        const double e = ((double)(rnd() >> 11) / 9007199254740992.0 - 0.5) * 0x1p-19;
        double y = q * (1.0 + e);
        y = fma(fma(-d, y, 1.0), y, y);
        y = fma(fma(-d, y, 1.0), y, y);
        y = fma(fma(-d, y, 1.0), y, y);
        uint64_t u;
        memcpy(&u, &d, 8);
        if ((u & 0xfffffffffffffull) != 0xfffffffffffffull) bad0 += y != q;
        memcpy(&u, &q, 8);
        if ((u & 0xfffffffffffffull) != 0xfffffffffffffull) {
            const double b = fma(fma(-q, d, 1.0), d, d);
            bad1 += b != 1.0 / q;
        }
    }
    printf("%ld %ld\n", bad0, bad1);
    return 0;
}
