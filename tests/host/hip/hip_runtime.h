/* Stand-ins that let rmhd_device.hpp be compiled by a host compiler, for the tests of its point
 * functions. The hardware approximations of 1/x and 1/sqrt(x) are cut to 26 bits, about what
 * the instructions give; the lane exchanges (used by one lane's worth of code only in
 * branches that these tests do not call) return the caller's own value. */
#pragma once

#include <cmath>
#include <cstdint>
#include <cstring>

#define __device__
#define __host__
#define __forceinline__ inline

static const struct { unsigned x; } threadIdx = { 0 };

inline double cut26(double y)
{
  std::uint64_t b;
  std::memcpy(&b, &y, 8);
  b &= ~((std::uint64_t(1) << 26) - 1);
  std::memcpy(&y, &b, 8);
  return y;
}
inline double __builtin_amdgcn_rcp(double x) { return cut26(1.0 / x); }
inline double __builtin_amdgcn_rsq(double x) { return cut26(1.0 / std::sqrt(x)); }
inline float __builtin_amdgcn_rcpf(float x) { return 1.0f / x; }
inline float __builtin_amdgcn_sqrtf(float x) { return std::sqrt(x); }
inline double __builtin_amdgcn_div_fixup(double r, double d, double)
{
  return d == 0.0 || std::isinf(d) || std::isnan(d) ? 1.0 / d : r;
}
inline int __builtin_amdgcn_update_dpp(int, int v, int, int, int, bool) { return v; }
inline unsigned long long __ballot(bool b) { return b; }
inline int __shfl(int v, int, int = 64) { return v; }
inline int __ffs(int v) { return __builtin_ffs(v); }
inline long long __double_as_longlong(double d) { long long r; std::memcpy(&r, &d, 8); return r; }
inline double __longlong_as_double(long long d) { double r; std::memcpy(&r, &d, 8); return r; }
inline int __float_as_int(float d) { int r; std::memcpy(&r, &d, 4); return r; }
inline float __int_as_float(int d) { float r; std::memcpy(&r, &d, 4); return r; }
