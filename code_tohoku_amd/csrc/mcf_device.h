// mcf_device.h -- FP64 point routines of the MCF3DSG* step for gfx950.
//
// Each routine restates the reference routine named beside it
// (M3 = 3DMHD-CfCA/MCF3DSGincfca3.f90) with the reference's evaluation
// order; the translation unit is built with -ffp-contract=off so no
// multiply-add is fused and IEEE division / square root are used, which
// keeps every cell bit-identical to the reference wherever no
// transcendental function is involved.
#pragma once
#include <hip/hip_runtime.h>

namespace mcf {

constexpr double KB = 8.63359;      // M3:11
constexpr double KCOND = 1.6384e-2; // M3:11
constexpr double EPSL = 1.0e-10;    // VLIMIT eps (M3:1697)

// dmax1 / dmin1 as flang lowers them (compare + select)
__device__ __forceinline__ double dmax(double a, double b) { return a > b ? a : b; }
__device__ __forceinline__ double dmin(double a, double b) { return a < b ? a : b; }

// (0.5-sign(0.5,-Q))*Q + (0.5+sign(0.5,-Q))*U : positivity fallback (M3:1389).
// One of the two weights is 1 and the other 0: Q where Q's sign bit is clear
// and U elsewhere, plus 0 times the other one, which keeps a NaN or an
// infinity of a blown-up reconstruction in the state.
__device__ __forceinline__ double posfix(double Q, double U) {
  const bool neg = signbit(Q);
  return __builtin_fma(0.0, neg ? Q : U, neg ? U : Q);
}

// n / d for several n over one d, each correctly rounded: the reciprocal y of
// d once (an IEEE division), then per quotient q = n*y corrected by its exact
// remainder, q + (n - q*d)*y (Markstein's correction step), and the hardware's
// fix-up of zero, infinite and NaN operands.  A quotient costs 4 instructions
// instead of the 11 of a division.  Correct while y and n - q*d are normal
// numbers: |d| in [2^-1022, 2^1022], |n| above 2^-968 (below it about one
// quotient in 400 is off by one unit in the last place).  A quotient that
// overflows comes out NaN where the division gives an infinity; telling them
// apart would cost an instruction a quotient, and both mark a blown-up state.
// tests/test_device_math.py holds these bounds.
struct Quot {
  double d, y;
  __device__ __forceinline__ explicit Quot(double d_) : d(d_), y(1.0 / d_) {}
  __device__ __forceinline__ double operator()(double n) const {
    double q = n * y;
    q = __builtin_fma(__builtin_fma(-q, d, n), y, q);
    return __builtin_amdgcn_div_fixup(q, d, n);
  }
};

// The limiter switch of VLIMIT (M3:1721): whether T = 1.27*U5/(kb*rho),
// rounded, is at least 3.  That is a/b > 3 - 2^-52 for a = 1.27*U5 and
// b = kb*rho (the lower end of 3's rounding interval, which no quotient of two
// doubles meets), which the exact a - 3b decides without the division; the
// strict comparison also holds for zero and infinite a or b.
__device__ __forceinline__ bool t_at_least_3(double u5, double rho) {
  const double a = 1.27 * u5, b = KB * rho;
  const double s = __builtin_fma(-3.0, b, a), t = -0x1p-52 * b;
  return signbit(b) ? s < t : s > t;
}

// RIEMAN (M3:1474-1551): four unrolled two-shock iterations with the
// tangential magnetic pressure added to P.
__device__ __forceinline__ void rieman(double D1, double V1, double P1, double B1sq, double D2, double V2,
                                       double P2, double B2sq, double gam, double &Pa, double &Va) {
  double gammi1 = gam - 1.0, gammi2 = gam - 2.0, gammi3 = gam - 3.0, gampl1 = gam + 1.0, gampl3 = gam + 3.0;
  double B1 = 0.5 * B1sq, B2 = 0.5 * B2sq;
  P1 = P1 + B1;
  P2 = P2 + B2;
  double GP1 = gammi1 * P1, GP2 = gammi1 * P2;
  double GP1B1 = gammi3 * P1 - gammi2 * B1 * 2.0;
  double GP2B2 = gammi3 * P2 - gammi2 * B2 * 2.0;
  double pa = (P1 + P2) * 0.5, q1 = 0.0, q2 = 0.0;
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    double pp1 = gampl3 * pa + GP1B1;
    double s1 = pp1 + sqrt(pp1 * pp1 - 8.0 * (pa - P1) * (gampl1 * pa + GP1));
    q1 = sqrt(s1 * D1) * 0.5;
    double pp2 = gampl3 * pa + GP2B2;
    double s2 = pp2 + sqrt(pp2 * pp2 - 8.0 * (pa - P2) * (gampl1 * pa + GP2));
    q2 = sqrt(s2 * D2) * 0.5;
    double old = pa;
    pa = q2 * P1 + q1 * P2 + q2 * q1 * (V1 - V2);
    if (it < 3) {
      pa = pa / (q2 + q1);
    } else {
      const Quot over(q2 + q1);
      pa = over(pa);
      Va = over(q1 * V1 + q2 * V2 + P1 - P2);
    }
    if (pa <= 0.0) pa = 0.1 * old;
  }
  Pa = pa;
}

// CHAREQ (M3:2101-2111)
__device__ __forceinline__ void chareq(double vyp, double Byp, double rl, double vym, double Bym, double rr,
                                       double &Bay, double &Vay) {
  double sp = sqrt(rl), sm = sqrt(rr);
  const Quot over(sp + sm);
  Vay = over(sp * vyp + sm * vym + Bym - Byp);
  Bay = over(sp * sm * (vym - vyp) + sp * Bym + sm * Byp);
}

// Koyama-Inutsuka net cooling (1DMHDKIcool/1DMHDwCC3KIcool.f90:1165-1171)
// with N = rho/1.27 (3DMHD-feedback/MCF3DSGincfca3-feedback.f90:3586).
__device__ __forceinline__ double fcool_ki(double rho, double T) {
  const Quot o127(1.27); // the reciprocal is a constant
  double N = o127(rho);
  double Laml = 1.0e7 * exp(-1.184e5 / (T * 1.0e3 + 1.0e3));
  Laml = dmin(Laml, 5.0e3);
  double Lamc = 1.4e-2 * sqrt(T * 1.0e3) * exp(-9.2e1 / (T * 1.0e3));
  return (N * N * (Laml + Lamc) - N) * 3.94656e1;
}

// IMC (M3:2898-2921): backward-Euler P + gammi1*Lambda(P)*dt = P_old by
// bisection in log10 P on [1e-10, 1e10], at most 30 steps.  The reference
// keeps the bracket in P and takes log10 of both ends and a power of ten per
// step; the bracket is kept in log10 P here.  Its upper end comes from
// 2 Pm/(2 + 1e-10) where the root lies below Pm: log10 Pm - IMC_DU.
constexpr double IMC_DU = 2.1714724094619722e-11; // log10(1 + 5e-11)
__device__ __forceinline__ double imc(double P, double n, double dt, double rho, double gammi1) {
  double lu = 10.0, ld = -10.0, lm = 1.0, Pm = 1.0e1, Pmold = -1.0;
  double nkbi = 1.0 / (KB * n);
  for (int it = 0; it < 30; ++it) {
    double T = Pm * nkbi;
    double CooL = fcool_ki(rho, T);
    double fev = Pm + CooL * dt * gammi1 - P;
    if (signbit(fev)) ld = dmax(lm, ld);
    else lu = dmin(lm - IMC_DU, lu);
    lm = 0.5 * (lu + ld);
    Pm = exp10(lm);
    if (fabs(Pm - Pmold) < 1.0e-5) break;
    Pmold = Pm;
  }
  return Pm;
}

} // namespace mcf
