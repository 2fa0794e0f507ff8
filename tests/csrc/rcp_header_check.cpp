// The reciprocals of gf_rcp.h, compiled for the host, against IEEE division.  Prints: operands
// that rcp_safe accepts and rcp_refine (from an estimate off by up to 2^-20) does not round
// correctly; the same of rcp_back; operands that rcp_safe ought to refuse and accepts, or the
// other way round.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <initializer_list>

#include "gf_rcp.h"

static uint64_t s = 88172645463325252ull;
static uint64_t rnd()
{
    s ^= s << 13;
    s ^= s >> 7;
    s ^= s << 17;
    return s;
}
static double make(int exponent, uint64_t significand)
{
    const uint64_t u = ((uint64_t)(1023 + exponent) << 52) | significand | (rnd() << 63);
    double d;
    memcpy(&d, &u, 8);
    return d;
}
int main(int argc, char **argv)
{
    const uint64_t ones = 0xfffffffffffffull;
    const long n = argc > 1 ? atol(argv[1]) : 1000000;
    long bad_refine = 0, bad_back = 0, bad_safe = 0;
    for (long k = 0; k < n; k++) {
        uint64_t m = rnd() & ones;
        if (k % 16 == 0) m = ones - rnd() % 4;  // significands of (nearly) all ones, and of zeros
        if (k % 16 == 1) m = rnd() % 4;
        const int e = k % 8 == 0 ? (rnd() & 1 ? 1 : -1) * (398 + (int)(rnd() % 5)) : (int)(rnd() % 801) - 400;
        const double d = make(e, m), q = 1.0 / d;
        bad_safe += rcp_safe(d) != (e >= -400 && e <= 400 && m != ones);
        if (!rcp_safe(d)) continue;
        const double off = ((double)(rnd() >> 11) / 9007199254740992.0 - 0.5) * 0x1p-19;
        bad_refine += rcp_refine(d, q * (1.0 + off)) != q;
        if (rcp_safe(q)) bad_back += rcp_back(q, d) != 1.0 / q;
    }
    for (double d : {0.0, -0.0, 5e-324, 0x1p-1022, (double)INFINITY, -(double)INFINITY, (double)NAN}) bad_safe += rcp_safe(d);
    printf("%ld %ld %ld\n", bad_refine, bad_back, bad_safe);
    return 0;
}
