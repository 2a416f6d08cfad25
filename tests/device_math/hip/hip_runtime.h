// What csrc/mcf_device.h and mcf_prec.h take from the HIP headers and the
// compiler, for a host compiler: the device's arithmetic is IEEE double and
// float, so the point routines give the same values here.
#pragma once
#include <cmath>
#include <cstring>

#define __device__
#define __forceinline__ inline

using std::copysign;
using std::fabs;
using std::signbit;
using std::sqrt;

inline int __double2hiint(double a) {
  long long b;
  std::memcpy(&b, &a, 8);
  return (int)(b >> 32);
}
inline float __builtin_amdgcn_rcpf(float a) { return 1.0f / a; }
inline float __builtin_amdgcn_sqrtf(float a) { return sqrtf(a); }
inline float __builtin_amdgcn_fmed3f(float a, float b, float c) { // no NaN operand
  return fmaxf(fminf(a, b), fminf(fmaxf(a, b), c));
}
// V_DIV_FIXUP_F64 as the instruction set's manual describes it: q kept, with
// the quotient's sign, unless an operand is zero, infinite or NaN
inline double __builtin_amdgcn_div_fixup(double q, double d, double n) {
  const double s = signbit(d) != signbit(n) ? -1.0 : 1.0;
  if (n != n || d != d) return n != n ? n : d;
  if ((d == 0.0 && n == 0.0) || (std::isinf(d) && std::isinf(n))) return NAN;
  if (d == 0.0 || std::isinf(n)) return s * INFINITY;
  if (std::isinf(d) || n == 0.0) return s * 0.0;
  return copysign(q, s);
}
