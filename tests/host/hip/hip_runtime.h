// What trips_math.h takes from HIP, for a host compiler: its scalar functions can then be run over whole ranges of floats.
#pragma once
#include <cmath>
#include <cstdint>
#include <cstring>
#include <algorithm>

#define __device__
#define __host__
#define __forceinline__ inline
#define asm(...)  // (scalar_const only names a kind of register)

using std::fabs;
using std::fma;
using std::max;
using std::min;
using std::rint;

struct float4
{
    float x, y, z, w;
};
struct double2
{
    double x, y;
};
inline double2 make_double2(double x, double y) { return {x, y}; }
inline uint32_t __float_as_uint(float f)
{
    uint32_t u;
    std::memcpy(&u, &f, 4);
    return u;
}
inline float __uint_as_float(uint32_t u)
{
    float f;
    std::memcpy(&f, &u, 4);
    return f;
}
inline int __float_as_int(float f) { return (int)__float_as_uint(f); }
inline double __builtin_amdgcn_ldexp(double v, int n)
{
    const int half = n / 2;  // (exact but for a result below the normal doubles, which no argument here has)
    auto power     = [](int e) { const uint64_t u = (uint64_t)(1023 + e) << 52; double d; std::memcpy(&d, &u, 8); return d; };
    return v * power(half) * power(n - half);
}
// The hardware's reciprocal is within one unit of the last place: the host's, moved by the units that a test asks for.
inline thread_local int t_rcp_units = 0;
inline float __builtin_amdgcn_rcpf(float b) { return __uint_as_float(__float_as_uint(1.f / b) + (uint32_t)t_rcp_units); }
