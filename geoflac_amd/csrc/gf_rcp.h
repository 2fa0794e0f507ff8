// gf_rcp.h -- correctly rounded reciprocals without the scaling of a full IEEE division.
// Also built for the host, by the test of their rounding.
#pragma once
#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define RCP_DEV static __host__ __device__ __forceinline__
#else
#define RCP_DEV static inline
#endif

// 1 / d from an estimate y of it (2^-20 or closer), correctly rounded for an operand that
// rcp_safe accepts: two Newton steps and a last step from the exact remainder (the steps of
// an IEEE division without the scaling that keeps extreme exponents in range)
RCP_DEV double rcp_refine(double d, double y)
{
    y = __builtin_fma(__builtin_fma(-d, y, 1.0), y, y);
    y = __builtin_fma(__builtin_fma(-d, y, 1.0), y, y);
    return __builtin_fma(__builtin_fma(-d, y, 1.0), y, y);
}
// |d| in [2^-400, 2^401), and a significand that is not all ones (the operands for which
// the last step need not round correctly: Markstein's exception)
RCP_DEV bool rcp_safe(double d)
{
    unsigned long long u;
    __builtin_memcpy(&u, &d, 8);
    const unsigned h = (unsigned)(u >> 32), e = (h >> 20) & 0x7ffu;
    return e - (1023u - 400u) <= 800u && ((h | 0xfff00000u) & (unsigned)u) != 0xffffffffu;
}
// 1 / a where a = RN(1 / d), correctly rounded where rcp_safe(a): the remainder 1 - a d is
// exact and d is within one ulp of 1 / a, so one step from d does
RCP_DEV double rcp_back(double a, double d) { return __builtin_fma(__builtin_fma(-a, d, 1.0), d, d); }

#ifdef __HIPCC__
// ... from the hardware's estimate
static __device__ __forceinline__ double rcp_core(double d) { return rcp_refine(d, __builtin_amdgcn_rcp(d)); }
#endif
