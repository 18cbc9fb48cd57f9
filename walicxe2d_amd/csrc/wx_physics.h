// wx_physics.h -- per-cell / per-face FP64 physics for the gfx950 kernels.
//
// Every function keeps the reference's evaluation order term by term (the
// library is compiled with -ffp-contract=off), so results agree with the
// Fortran to the last few ulps; the only differences come from the device
// libm (exp/log/pow/sin) against glibc.
#pragma once
#include <hip/hip_runtime.h>
#include "wx_device.h"
#include "wx_libm.h"

namespace wx {

__device__ __forceinline__ double dmax(double a, double b) { return a > b ? a : b; }
__device__ __forceinline__ double dmin(double a, double b) { return a < b ? a : b; }

// Branches taken (almost) never: the register allocator places its spills
// there, not on the path every cell takes.
#define WX_RARE(c) __builtin_expect(!!(c), 0)

// ---------------------------------------------------------------------
// Division and square root in a known range.  The compiler's FP64 division
// is 11 instructions (two v_div_scale, v_rcp, four fma, mul, fma,
// v_div_fmas, v_div_fixup, plus the wait states of the vcc they share); the
// scaling and the fix-up act only on operands near the ends of the exponent
// range.  Between them the sequence is rdiv/quot below, so on operands where
// v_div_scale leaves both unscaled (the denominator's exponent within
// +-900, the numerator zero or at least 2^-900, their exponents less than
// 768 apart) the quotient is the same, bit for bit, in 8 instructions, and in
// 3 more for each further numerator over the same denominator.  A zero
// numerator keeps its sign for a positive denominator.  The same holds for
// the square root without its scaling (used on [2^-700, 2^700]).  Every use
// below is behind a test of the range, and the general form runs outside it.
struct Rcp {
  double b, y;
};
__device__ __forceinline__ Rcp rdiv(double b) {
  double y = __builtin_amdgcn_rcp(b);
  y = __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
  y = __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
  return Rcp{b, y};
}
__device__ __forceinline__ double quot(double a, const Rcp &r) {
  const double q = a * r.y;
  return __builtin_fma(-__builtin_fma(r.b, q, -a), r.y, q);
}
__device__ __forceinline__ double fdiv(double a, double b) { return quot(a, rdiv(b)); }
__device__ __forceinline__ double fsqrt(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}

// F: the short forms above, or (F false) the operators.
template <bool F>
__device__ __forceinline__ double div_(double a, double b) { return F ? fdiv(a, b) : a / b; }
template <bool F>
__device__ __forceinline__ double sqrt_(double x) { return F ? fsqrt(x) : sqrt(x); }
template <bool F>
__device__ __forceinline__ Rcp rdiv_(double b) { return F ? rdiv(b) : Rcp{b, 0.0}; }
template <bool F>
__device__ __forceinline__ double quot_(double a, const Rcp &r) { return F ? quot(a, r) : a / r.b; }

// The reciprocals of the constants every cell divides by.
struct RecipP {
  Rcp cv, Tempsc;
};
__device__ __forceinline__ double uniform(double x) {
  const uint64_t u = __double_as_longlong(x);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((int)u), hi = __builtin_amdgcn_readfirstlane((int)(u >> 32));
  return __longlong_as_double(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ RecipP recip_params(const wx_params *__restrict__ p) {
  return RecipP{Rcp{p->cv, uniform(rdiv(p->cv).y)}, Rcp{p->Tempsc, uniform(rdiv(p->Tempsc).y)}};
}
// x in [2^-k, 2^k), k = 64 (x from memory, uniform: scalar instructions)
__device__ __forceinline__ bool unit_range(double x) {
  return (uint32_t)(__double_as_longlong(x) >> 32) - 0x3bf00000u < 0x08000000u;
}
// The run's constants the short forms divide by, or scale by, are ordinary.
__device__ __forceinline__ bool mild_params(const wx_params *__restrict__ p, int level) {
  return unit_range(p->cv) & unit_range(p->Tempsc) & unit_range(p->gamma) & unit_range(p->dx[level - 1]) &
         unit_range(p->dy[level - 1]);
}

// "Mild" primitives: rho in [1e-15, 2^64], p in [2^-64, 2^64], every
// velocity and passive zero or in [tiny, 2^64] in magnitude.  Then every
// operand of the solvers' divisions is in the range above except where two
// speeds nearly agree or a star speed's numerator nearly vanishes, which the
// solvers test themselves.  tiny: with HLLC and minmod 2^-800 (a face value is
// a cell's plus half a difference of cells, zero or at least 2^-853, and
// enters the divisions once); with HLL, the hybrid, van Leer or the
// cylindrical sources, which divide products of up to three such values,
// 2^-220.  Around every expanding
// flow a few cells hold velocities below either bound, down to the last
// denormal; their blocks take the general form.
constexpr double kHuge = 0x1p64;
__device__ __forceinline__ double mild_tiny(const wx_params *__restrict__ p) {
  return p->solver == 0 && p->limiter == 1 && !p->cylindrical ? 0x1p-800 : 0x1p-220;
}

// src/uprim.f90:5-63 : conserved -> primitive, floors, T by cooling mode.
template <int NEQ>
__device__ __forceinline__ void uprim(const wx_params *__restrict__ p, double *q,
                                      const double *uu, double &T) {
  const double cv = p->cv;
  double r = dmax(uu[0], 1e-15);
  q[0] = r;
  q[1] = uu[1] / r;
  q[2] = uu[2] / r;
#pragma unroll
  for (int k = 4; k < NEQ; ++k) q[k] = uu[k];
  q[3] = (uu[3] - 0.5 * r * (q[1] * q[1] + q[2] * q[2])) / cv;
  q[3] = dmax(q[3], 1e-15);
  const int mode = p->cooling;
  if (mode == 0) {
    T = q[3] / r;
  } else if (mode == 1) {
    double dentot = (2.0 * r - (NEQ > 4 ? q[NEQ > 4 ? 4 : 0] : 0.0));
    dentot = dmax(dentot, 1e-15);
    T = dmax(1.0, (q[3] / dentot) * p->Tempsc);
    q[3] = dentot * T / p->Tempsc;
  } else {
    r = dmax(r, 1e-15);
    T = dmax(1.0, (q[3] / (r)) * p->Tempsc);
    q[3] = r * T / p->Tempsc;
  }
}

// uprim with the short divisions.  Returns whether q is uprim's bit for bit
// and mild (false: q is not to be used).  The floors make the small numerators
// harmless: a quotient below 1e-15 is replaced.  0.5 r (v^2) is taken as half
// of r (v^2) inside the fused subtraction, an exact scaling.  tiny 0: the
// velocities are only for sums that a value below 2^-300 leaves unchanged
// (kinetic energies, signal speeds), so small ones pass.
template <int NEQ>
__device__ __forceinline__ bool uprim_mild(const wx_params *__restrict__ p, const RecipP &rp, double tiny, double *q,
                                           const double *uu, double &T) {
  const double r = __builtin_fmax(uu[0], 1e-15);
  const Rcp rr = rdiv(r);
  q[0] = r;
  q[1] = quot(uu[1], rr);
  q[2] = quot(uu[2], rr);
  const double N = __builtin_fma(-0.5, r * (q[1] * q[1] + q[2] * q[2]), uu[3]);
  q[3] = __builtin_fmax(quot(N, rp.cv), 1e-15);
  // (no short circuits here: they would cost branches)
  bool ok = (fabs(N) <= 0x1p300) & ((fabs(q[1]) >= tiny) | (uu[1] == 0.0)) & ((fabs(q[2]) >= tiny) | (uu[2] == 0.0));
#pragma unroll
  for (int k = 4; k < NEQ; ++k) {
    q[k] = uu[k];
    ok &= (fabs(uu[k]) <= kHuge) & ((fabs(uu[k]) >= 0x1p-220) | (uu[k] == 0.0));
  }
  const int mode = p->cooling;
  if (mode == 0) {
    T = quot(q[3], rr);
  } else {
    double dentot = r;
    if (mode == 1) dentot = __builtin_fmax(__builtin_fma(2.0, r, -(NEQ > 4 ? q[NEQ > 4 ? 4 : 0] : 0.0)), 1e-15);
    T = __builtin_fmax(1.0, fdiv(q[3], dentot) * p->Tempsc);
    q[3] = quot(dentot * T, rp.Tempsc);
  }
  return ok & (__builtin_fmax(__builtin_fmax(r, q[3]), __builtin_fmax(fabs(q[1]), fabs(q[2]))) <= kHuge);
}

// Both: the short form, and uprim for the lanes it does not serve.  Returns
// whether q is mild.
template <int NEQ>
__device__ __forceinline__ bool uprim_any(const wx_params *__restrict__ p, const RecipP &rp, bool pok, double tiny,
                                          double *q, const double *uu, double &T) {
  const bool ok = uprim_mild<NEQ>(p, rp, tiny, q, uu, T) & pok;
  if (WX_RARE(!ok)) uprim<NEQ>(p, q, uu, T);
  return ok;
}

// src/primu.f90:4-19
template <int NEQ>
__device__ __forceinline__ void primu(double cv, const double *q, double *uu) {
  uu[0] = q[0];
  uu[1] = q[0] * q[1];
  uu[2] = q[0] * q[2];
  uu[3] = 0.5 * q[0] * (q[1] * q[1] + q[2] * q[2]) + cv * q[3];
#pragma unroll
  for (int k = 4; k < NEQ; ++k) uu[k] = q[k];
}

// src/primf.f90:5-23
template <int NEQ>
__device__ __forceinline__ void primf(double cv, const double *q, double *ff) {
  double etot = 0.5 * q[0] * (q[1] * q[1] + q[2] * q[2]) + cv * q[3];
  ff[0] = q[0] * q[1];
  ff[1] = q[0] * q[1] * q[1] + q[3];
  ff[2] = q[0] * q[1] * q[2];
  ff[3] = q[1] * (etot + q[3]);
#pragma unroll
  for (int k = 4; k < NEQ; ++k) ff[k] = q[k] * q[1];
}

// src/limiter.f90:26-87 `average`
__device__ __forceinline__ double average(int lim, double a, double b) {
  double s, c, d, r;
  switch (lim) {
    case -1: return 0.0;
    case 0: return 0.5 * (a + b);
    case 1:
      s = copysign(1.0, a);
      return s * dmax(0.0, dmin(fabs(a), s * b));
    case 2:
      if (a * b <= 0.0) return 0.0;
      return a * b * (a + b) / (a * a + b * b);
    case 3: {
      const double delta = 1.e-7;
      return (a * (b * b + delta) + b * (a * a + delta)) / (a * a + b * b + delta);
    }
    case 4:
      s = copysign(1.0, a);
      c = 0.25 * a + 0.75 * b;
      d = 0.75 * a + 0.25 * b;
      r = dmin(dmin(dmin(2.0 * fabs(a), 2.0 * s * b), s * c), s * d);
      return s * dmax(0.0, r);
    case 5:
      s = copysign(1.0, a);
      c = 0.5 * (a + b);
      r = dmin(dmin(2.0 * fabs(a), 2.0 * s * b), s * c);
      return s * dmax(0.0, r);
    case 6: {
      s = copysign(1.0, b);
      double av1 = dmin(2.0 * fabs(b), s * a);
      double av2 = dmin(fabs(b), 2.0 * s * a);
      return s * dmax(dmax(0.0, av1), av2);
    }
    default: return 0.0;
  }
}

// src/limiter.f90:7-24 (all variables, passives included)
template <int NEQ>
__device__ __forceinline__ void limiter(int lim, const double *pll, double *pl, double *pr,
                                        const double *prr) {
#pragma unroll
  for (int k = 0; k < NEQ; ++k) {
    double dl = pl[k] - pll[k];
    double dm = pr[k] - pl[k];
    double dr = prr[k] - pr[k];
    double al = average(lim, dl, dm);
    double ar = average(lim, dm, dr);
    pl[k] = pl[k] + al * 0.5;
    pr[k] = pr[k] - ar * 0.5;
  }
}

// HLLC star flux on one side: src/hllcfluxes.f90:131-166.
template <int NEQ>
__device__ __forceinline__ void hllc_star(const wx_params *__restrict__ p, const double *q,
                                          double s, double smu, double sst, bool right,
                                          double *ff) {
  const double cv = p->cv;
  double uu[NEQ], uuk[NEQ];
  double rhost = q[0] * (smu) / (s - sst);
  double ek = 0.5 * q[0] * (q[1] * q[1] + q[2] * q[2]) + cv * q[3];
  uuk[0] = rhost;
  uuk[1] = rhost * sst;
  uuk[2] = rhost * q[2];
  double den = (right && (p->compat & 1)) ? (q[3] * smu) : (q[0] * smu);
  uuk[3] = rhost * (ek / q[0] + (sst - q[1]) * (sst + q[3] / den));
#pragma unroll
  for (int k = 4; k < NEQ; ++k) uuk[k] = rhost * q[k] / q[0];
  primf<NEQ>(cv, q, ff);
  primu<NEQ>(cv, q, uu);
#pragma unroll
  for (int k = 0; k < NEQ; ++k) ff[k] = ff[k] + s * (uuk[k] - uu[k]);
}

// Riemann solvers: HLLC (src/hllcfluxes.f90:98-173), HLL
// (src/hllfluxes.f90:98-131), HLL/HLLC hybrid (src/hll_hllcfluxes.f90:95-209).
// Returns nonzero on the reference's `stop` path (NaN star speed).
// SOLVER >= 0 fixes the solver at compile time (the same arithmetic, with
// the other solvers' branches compiled out); -1 reads it from p.
template <int NEQ, int SOLVER = -1>
__device__ __forceinline__ int riemann(const wx_params *__restrict__ p, const double *pl,
                                       const double *pr, double *ff) {
  const double cv = p->cv, gam = p->gamma;
  const int solver = SOLVER >= 0 ? SOLVER : p->solver;
  double beta1 = 1.0, beta2 = 0.0;
  if (solver == 2) {
    double dq1 = pr[1] - pl[1], dq2 = pr[2] - pl[2];
    double mag = sqrt(dq1 * dq1 + dq2 * dq2);
    if (mag <= 1e-6) {
      beta1 = 1.0;
      beta2 = 0.0;
    } else {
      double alpha1 = fabs(dq1) / mag;
      beta1 = sqrt(alpha1);
      beta2 = 1.0 - beta1;
    }
  }
  double csl = sqrt(gam * pl[3] / pl[0]);
  double csr = sqrt(gam * pr[3] / pr[0]);
  double sr = dmax(pl[1] + csl, pr[1] + csr);
  double sl = dmin(pl[1] - csl, pr[1] - csr);
  // supersonic faces take the upwind state's flux; the side is selected
  // first so that a wave evaluates primf once whichever sides its lanes need
  if (sl > 0 || sr < 0) {
    const bool up = sl > 0;
    double qu[NEQ];
#pragma unroll
    for (int k = 0; k < NEQ; ++k) qu[k] = up ? pl[k] : pr[k];
    primf<NEQ>(cv, qu, ff);
    return 0;
  }
  if (solver == 1) {
    double fl[NEQ], fr[NEQ], ul[NEQ], ur[NEQ];
    primf<NEQ>(cv, pl, fl); primf<NEQ>(cv, pr, fr);
    primu<NEQ>(cv, pl, ul); primu<NEQ>(cv, pr, ur);
#pragma unroll
    for (int k = 0; k < NEQ; ++k)
      ff[k] = (sr * fl[k] - sl * fr[k] + sl * sr * (ur[k] - ul[k])) / (sr - sl);
    return 0;
  }
  double slmul = sl - pl[1];
  double srmur = sr - pr[1];
  double rholul = pl[0] * pl[1];
  double rhorur = pr[0] * pr[1];
  double sst = (srmur * rhorur - slmul * rholul - pr[3] + pl[3]) / (srmur * pr[0] - slmul * pl[0]);
  // star region of the side sst points away from (one evaluation per lane,
  // the side selected first); a NaN star speed is the reference's `stop`
  const bool left = sst >= 0.0;
  const int err = (left || sst <= 0.0) ? 0 : 1;
  {
    double qs[NEQ];
#pragma unroll
    for (int k = 0; k < NEQ; ++k) qs[k] = left ? pl[k] : pr[k];
    hllc_star<NEQ>(p, qs, left ? sl : sr, left ? slmul : srmur, sst, !left, ff);
  }
  if (err) {
#pragma unroll
    for (int k = 0; k < NEQ; ++k) ff[k] = 0.0;
  }
  if (solver == 2 && !err) {
    double fl[NEQ], fr[NEQ], ul[NEQ], ur[NEQ];
    primf<NEQ>(cv, pl, fl); primf<NEQ>(cv, pr, fr);
    primu<NEQ>(cv, pl, ul); primu<NEQ>(cv, pr, ur);
#pragma unroll
    for (int k = 0; k < NEQ; ++k)
      ff[k] = beta1 * (ff[k]) + beta2 * ((sr * fl[k] - sl * fr[k] + sl * sr * (ur[k] - ul[k])) / (sr - sl));
  }
  return err;
}

// ---------------------------------------------------------------------
// The same fluxes on mild states (mild_tiny), for HLLC, HLL and the hybrid
// and the minmod and van Leer limiters: the operations of the functions
// above in their order, with the short divisions and square roots, the
// hardware's max and min (no NaN reaches them), products with a power of two
// fused into the addition that follows (the product is exact), and one
// reciprocal of each density for the sound speed and the star state.

// average(lim, a, b) of the limiters 1 and 2
template <int LIM>
__device__ __forceinline__ double average_mild(double a, double b) {
  static_assert(LIM == 1 || LIM == 2, "minmod or van Leer");
  if constexpr (LIM == 1) {
    const double s = copysign(1.0, a);
    return s * __builtin_fmax(0.0, __builtin_fmin(fabs(a), s * b));
  } else {
    const double ab = a * b;
    const double v = fdiv(ab * (a + b), a * a + b * b);
    return ab <= 0.0 ? 0.0 : v;   // (where the denominator is zero, too)
  }
}

template <int NEQ, int LIM>
__device__ __forceinline__ void limiter_mild(const double *pll, double *pl, double *pr, const double *prr) {
#pragma unroll
  for (int k = 0; k < NEQ; ++k) {
    const double dl = pl[k] - pll[k];
    const double dm = pr[k] - pl[k];
    const double dr = prr[k] - pr[k];
    pl[k] = __builtin_fma(average_mild<LIM>(dl, dm), 0.5, pl[k]);
    pr[k] = __builtin_fma(average_mild<LIM>(dm, dr), -0.5, pr[k]);
  }
}

// primf and primu of one state (src/primf.f90:5-23, src/primu.f90:4-19)
template <int NEQ>
__device__ __forceinline__ void flux_state(double cv, const double *q, double *ff, double *uu) {
  const double e = __builtin_fma(0.5, q[0] * (q[1] * q[1] + q[2] * q[2]), cv * q[3]);
  uu[0] = q[0];
  uu[1] = q[0] * q[1];
  uu[2] = q[0] * q[2];
  uu[3] = e;
  ff[0] = uu[1];
  ff[1] = uu[1] * q[1] + q[3];
  ff[2] = uu[1] * q[2];
  ff[3] = q[1] * (e + q[3]);
#pragma unroll
  for (int k = 4; k < NEQ; ++k) {
    uu[k] = q[k];
    ff[k] = q[k] * q[1];
  }
}

// riemann<NEQ, SOLVER> on mild states whose sound speeds are given (and, with
// RECIP, the reciprocals of their densities).  Returns whether ff is valid;
// false (a face with two speeds that agree to 2^-250 or so, or without a star
// speed, or with a numerator below 2^-900) leaves ff to riemann.
template <int NEQ, int SOLVER, bool RECIP>
__device__ __forceinline__ bool riemann_mild(const wx_params *__restrict__ p, const double *pl, const double *pr,
                                             double csl, double csr, const Rcp &rl, const Rcp &rr, double *ff) {
  const double cv = p->cv;
  const double sr = __builtin_fmax(pl[1] + csl, pr[1] + csr);
  const double sl = __builtin_fmin(pl[1] - csl, pr[1] - csr);
  if (sl > 0 || sr < 0) {
    const bool up = sl > 0;
    double qu[NEQ], uu[NEQ];
#pragma unroll
    for (int k = 0; k < NEQ; ++k) qu[k] = up ? pl[k] : pr[k];
    flux_state<NEQ>(cv, qu, ff, uu);
    return true;
  }
  bool ok = true;
  if constexpr (SOLVER != 1) {
    const double slmul = sl - pl[1];
    const double srmur = sr - pr[1];
    const double num = srmur * (pr[0] * pr[1]) - slmul * (pl[0] * pl[1]) - pr[3] + pl[3];
    const double sst = fdiv(num, srmur * pr[0] - slmul * pl[0]);
    const bool left = sst >= 0.0;
    double qs[NEQ], uu[NEQ];
#pragma unroll
    for (int k = 0; k < NEQ; ++k) qs[k] = left ? pl[k] : pr[k];
    const double s = left ? sl : sr, smu = left ? slmul : srmur;
    const Rcp rq = RECIP ? Rcp{qs[0], left ? rl.y : rr.y} : rdiv(qs[0]);
    flux_state<NEQ>(cv, qs, ff, uu);
    const double rsmu = qs[0] * smu, ss = s - sst;
    const double den = (!left && (p->compat & 1)) ? (qs[3] * smu) : rsmu;
    // (false too where the star speed is a NaN)
    ok = (fabs(ss * den) >= 0x1p-250) & ((fabs(num) >= 0x1p-900) | (num == 0.0));
    const double rhost = fdiv(rsmu, ss);
    ff[0] = ff[0] + s * (rhost - uu[0]);
    ff[1] = ff[1] + s * (rhost * sst - uu[1]);
    ff[2] = ff[2] + s * (rhost * qs[2] - uu[2]);
    ff[3] = ff[3] + s * (rhost * (quot(uu[3], rq) + (sst - qs[1]) * (sst + fdiv(qs[3], den))) - uu[3]);
#pragma unroll
    for (int k = 4; k < NEQ; ++k) ff[k] = ff[k] + s * (quot(rhost * qs[k], rq) - uu[k]);
  }
  if constexpr (SOLVER != 0) {
    double fl[NEQ], fr[NEQ], ul[NEQ], ur[NEQ];
    flux_state<NEQ>(cv, pl, fl, ul);
    flux_state<NEQ>(cv, pr, fr, ur);
    const double ds = sr - sl, slsr = sl * sr;
    const Rcp rs = rdiv(ds);
    ok &= ds >= 0x1p-250;
    double beta1 = 0.0, beta2 = 1.0;
    if constexpr (SOLVER == 2) {
      const double dq1 = pr[1] - pl[1], dq2 = pr[2] - pl[2];
      const double mag = sqrt(dq1 * dq1 + dq2 * dq2);
      beta1 = 1.0;
      beta2 = 0.0;
      if (mag > 1e-6) {
        beta1 = sqrt(fdiv(fabs(dq1), mag));
        beta2 = 1.0 - beta1;
      }
    }
#pragma unroll
    for (int k = 0; k < NEQ; ++k) {
      const double h = quot(sr * fl[k] - sl * fr[k] + slsr * (ur[k] - ul[k]), rs);
      ff[k] = SOLVER == 1 ? h : beta1 * ff[k] + beta2 * h;
    }
  }
  return ok;
}

// ---------------------------------------------------------------------
// Cooling.  src/coolingh.f90:41-76 rates, :88-165 ALOSS, :171-259 atomic.
// Every operation is the routine's, in its order; exp and ** are the host C
// library's functions (wx_libm.h: equal to them bit for bit), log is
// correctly rounded.
__device__ __forceinline__ double rate_alpha(double T) { return 2.55e-13 * libm::wpow(1.e4 / T, 0.79); }
__device__ __forceinline__ double rate_colf(double T) { return 5.83e-11 * sqrt(T) * libm::wexp(-(157828. / T)); }
__device__ __forceinline__ double rate_betah(double T) {
  double a = 157890. / T;
  double lga;   // log(a), sharing pow's logarithm of a
  const double pw = libm::wlog_pow(a, -0.33333, &lga);
  return 1.133e-24 / sqrt(a) * (-0.0713 + 0.5 * lga + 0.640 * pw);
}

__device__ __forceinline__ double aloss(double x1, double den, double dh0, double te0) {
  const double XION = 2.179e-11, XO = 1.e-3;
  const double C0 = 0.5732, C1 = 1.8288e-5, C2 = -1.15822e-10, C3 = 9.4288e-16;
  const double D0 = 0.5856, D1 = 1.55083e-5, D2 = -9.669e-12, D3 = 5.716e-19;
  const double ENK = 118409., EN = 1.634E-11;
  double TE = dmax(te0, 1000.);
  double DH = den;
  double DHP = (1. - x1) * DH;
  double DE = DHP + 1.E-4 * DH;
  double DOI = XO * dh0;
  double DOII = XO * DHP;
  double OMEGA = 0.0;
  if (TE <= 55000.) OMEGA = C0 + TE * (C1 + TE * (C2 + TE * C3));
  if (TE >= 72000.) OMEGA = D0 + TE * (D1 + TE * (D2 + TE * D3));
  if (TE > 55000. && TE < 72000.) {
    double OMEGAL = C0 + TE * (C1 + TE * (C2 + TE * C3));
    double OMEGAH = D0 + TE * (D1 + TE * (D2 + TE * D3));
    double FRAC = (TE - 55000.) / 17000.;
    OMEGA = (1. - FRAC) * OMEGAL + FRAC * OMEGAH;
  }
  double QLA = 8.6287E-6 / (2. * sqrt(TE)) * OMEGA * libm::wexp(-(ENK / TE));
  double ECOLL = DE * dh0 * QLA * EN;
  ECOLL = dmax(ECOLL, 0.);
  double CION = 5.834E-11 * sqrt(TE) * libm::wexp(-(1.579E5 / TE));
  double EION = DE * dh0 * CION * XION;
  double FR = 0.0;
  if (TE <= 44770.) FR = 0.;
  if (TE >= 54770.) FR = 1.;
  if (TE > 44770. && TE < 54770.) {
    double EX2 = libm::wexp(-(2. * (TE - 49770.) / 500.));
    double TANH = (1. - EX2) / (1. + EX2);
    FR = 0.5 * (1. + TANH);
  }
  // The recombination + oxygen terms enter with weight 1 - FR and the
  // equilibrium curve with weight FR: each is evaluated only where its weight
  // is nonzero (both are finite, so a skipped term contributes the same +0
  // as the routine's product with a zero weight).
  double LOW = 0.0, HIGH = 0.0;
  if (TE < 54770.) {
    double EREC = DE * DHP * (rate_betah(TE));
    EREC = dmax(EREC, 0.);
    double TM = 1. / TE;
    double T2 = TM * TM;
    double EOI = DE * DOI * libm::wpow(10., 1381465 * T2 - 12328.69 * TM - 19.82621);
    double EOII = DE * DOII * libm::wpow(10., -(2061075. * T2) - 14596.24 * TM - 19.01402);
    EOI = dmax(EOI, 0.);
    EOII = dmax(EOII, 0.);
    LOW = EREC + 7.033 * (EOI + EOII);
  }
  if (TE > 44770.) {
    double BETAF = 1.3 * 1.42E-27 * libm::wpow(TE, 0.5);
    double HIICOOL = DE * DHP * BETAF;
    HIGH = (1.0455E-18 / libm::wpow(TE, 0.63)) * (1. - libm::wexp(-libm::wpow(TE * 1.E-5, 1.63))) * DE * den + HIICOOL;
  }
  return ECOLL + EION + LOW * (1. - FR) + HIGH * FR;
}

// src/coolingh.f90:171-259 atomic: H neutral fraction + radiative loss.
template <int NEQ>
__device__ __forceinline__ void atomic_h(const wx_params *__restrict__ p, double dt, double *uu) {
  if constexpr (NEQ >= 5) {
    const double xi = 1.e-4, boltzm = 1.3807e-16;
    double q[NEQ], T;
    uprim<NEQ>(p, q, uu, T);
    double col = rate_colf(T);
    double rec = rate_alpha(T);
    double y0 = uu[4] / uu[0];
    double dh = uu[0];
    double a = rec + col;
    double b = -((2. + xi) * rec + (1. + xi) * col);
    double c = (1. + xi) * rec;
    double d = sqrt(b * b - 4. * a * c);
    double g0 = (2. * a * y0 + b + d) / (2. * a * y0 + b - d);
    double e = libm::wexp(-(d * dh * dt));
    double y1 = (-b - d * (1. + g0 * e) / (1. - g0 * e)) / (2. * a);
    y1 = dmin(y1, 1.);
    y1 = dmax(y1, 0.0001);
    uu[4] = y1 * uu[0];
    double dh0 = uu[4];
    double al = aloss(y0, dh, dh0, T) / (dh * dh);
    double tprime = 10.;
    double ce = (2. * dh * al) / (3. * boltzm * T);
    double t1 = tprime + (T - tprime) * libm::wexp(-(ce * dt));
    t1 = dmax(t1, 0.1 * T);
    t1 = dmin(t1, 10. * T);
    t1 = dmax(t1, tprime);
    uu[3] = p->cv * (2. * uu[0] - uu[4]) * t1 / p->Tempsc + 0.5 * q[0] * (q[1] * q[1] + q[2] * q[2]);
  }
}

// atomic_h of a cell whose uprim_mild (q, T) held and whose density is not
// floored: the same operations in their order with the short divisions and
// square roots, the quotients over T and TE each sharing one reciprocal, and
// sqrt(T) taken once where TE is T.  Returns false, leaving uu as it was,
// where one of the two differences divided by vanishes (then atomic_h).
__device__ __forceinline__ double aloss_mild(double x1, double den, double dh0, double TE, double sqTE) {
  const double XION = 2.179e-11, XO = 1.e-3;
  const double C0 = 0.5732, C1 = 1.8288e-5, C2 = -1.15822e-10, C3 = 9.4288e-16;
  const double D0 = 0.5856, D1 = 1.55083e-5, D2 = -9.669e-12, D3 = 5.716e-19;
  const double ENK = 118409., EN = 1.634E-11;
  const Rcp rTE = rdiv(TE);
  double DH = den;
  double DHP = (1. - x1) * DH;
  double DE = DHP + 1.E-4 * DH;
  double DOI = XO * dh0;
  double DOII = XO * DHP;
  double OMEGA = 0.0;
  if (TE <= 55000.) OMEGA = C0 + TE * (C1 + TE * (C2 + TE * C3));
  if (TE >= 72000.) OMEGA = D0 + TE * (D1 + TE * (D2 + TE * D3));
  if (TE > 55000. && TE < 72000.) {
    double OMEGAL = C0 + TE * (C1 + TE * (C2 + TE * C3));
    double OMEGAH = D0 + TE * (D1 + TE * (D2 + TE * D3));
    double FRAC = (TE - 55000.) / 17000.;
    OMEGA = (1. - FRAC) * OMEGAL + FRAC * OMEGAH;
  }
  double QLA = fdiv(8.6287E-6, 2. * sqTE) * OMEGA * libm::wexp(-quot(ENK, rTE));
  double ECOLL = DE * dh0 * QLA * EN;
  ECOLL = __builtin_fmax(ECOLL, 0.);
  double CION = 5.834E-11 * sqTE * libm::wexp(-quot(1.579E5, rTE));
  double EION = DE * dh0 * CION * XION;
  double FR = 0.0;
  if (TE >= 54770.) FR = 1.;
  if (TE > 44770. && TE < 54770.) {
    double EX2 = libm::wexp(-(2. * (TE - 49770.) / 500.));
    double TANH = (1. - EX2) / (1. + EX2);
    FR = 0.5 * (1. + TANH);
  }
  double LOW = 0.0, HIGH = 0.0;
  if (TE < 54770.) {
    const double a = quot(157890., rTE);   // rate_betah
    double lga;
    const double pw = libm::wlog_pow(a, -0.33333, &lga);
    const double betah = fdiv(1.133e-24, fsqrt(a)) * (-0.0713 + 0.5 * lga + 0.640 * pw);
    double EREC = DE * DHP * betah;
    EREC = __builtin_fmax(EREC, 0.);
    double TM = quot(1., rTE);
    double T2 = TM * TM;
    double EOI = DE * DOI * libm::wpow(10., 1381465 * T2 - 12328.69 * TM - 19.82621);
    double EOII = DE * DOII * libm::wpow(10., -(2061075. * T2) - 14596.24 * TM - 19.01402);
    EOI = __builtin_fmax(EOI, 0.);
    EOII = __builtin_fmax(EOII, 0.);
    LOW = EREC + 7.033 * (EOI + EOII);
  }
  if (TE > 44770.) {
    double BETAF = 1.3 * 1.42E-27 * libm::wpow(TE, 0.5);
    double HIICOOL = DE * DHP * BETAF;
    HIGH = fdiv(1.0455E-18, libm::wpow(TE, 0.63)) * (1. - libm::wexp(-libm::wpow(TE * 1.E-5, 1.63))) * DE * den + HIICOOL;
  }
  return ECOLL + EION + LOW * (1. - FR) + HIGH * FR;
}

template <int NEQ>
__device__ __forceinline__ bool atomic_mild(const wx_params *__restrict__ p, const RecipP &rp, double dt,
                                            const double *q, double T, double *uu) {
  static_assert(NEQ >= 5, "n_HI is variable 5");
  const double xi = 1.e-4, boltzm = 1.3807e-16;
  const Rcp rT = rdiv(T);
  const double sqT = fsqrt(T);
  const double col = 5.83e-11 * sqT * libm::wexp(-quot(157828., rT));   // rate_colf
  const double rec = 2.55e-13 * libm::wpow(quot(1.e4, rT), 0.79);       // rate_alpha
  const double y0 = fdiv(uu[4], uu[0]);
  const double dh = uu[0];
  const double a = rec + col;
  const double b = -((2. + xi) * rec + (1. + xi) * col);
  const double c = (1. + xi) * rec;
  const double d = fsqrt(b * b - 4. * a * c);
  const double n2 = 2. * a * y0 + b - d;
  const double g0 = fdiv(2. * a * y0 + b + d, n2);
  const double e = libm::wexp(-(d * dh * dt));
  const double n3 = 1. - g0 * e;
  if (WX_RARE(!((fabs(n2) >= 0x1p-600) & (fabs(n3) >= 0x1p-300)))) return false;
  double y1 = fdiv(-b - fdiv(d * (1. + g0 * e), n3), 2. * a);
  y1 = __builtin_fmin(y1, 1.);
  y1 = __builtin_fmax(y1, 0.0001);
  uu[4] = y1 * uu[0];
  const double dh0 = uu[4];
  const double TE = __builtin_fmax(T, 1000.);
  const double al = fdiv(aloss_mild(y0, dh, dh0, TE, T >= 1000. ? sqT : fsqrt(TE)), dh * dh);
  const double tprime = 10.;
  const double ce = fdiv(2. * dh * al, 3. * boltzm * T);
  double t1 = tprime + (T - tprime) * libm::wexp(-(ce * dt));
  t1 = __builtin_fmax(t1, 0.1 * T);
  t1 = __builtin_fmin(t1, 10. * T);
  t1 = __builtin_fmax(t1, tprime);
  uu[3] = __builtin_fma(0.5, q[0] * (q[1] * q[1] + q[2] * q[2]),
                        quot(p->cv * __builtin_fma(2., uu[0], -uu[4]) * t1, rp.Tempsc));
  return true;
}

// src/dmc_module.f90:14-32 cooldmc (row 42 at T == 1e8 clamps to row 41)
__device__ __forceinline__ double cooldmc(const wx_params *__restrict__ p, double T) {
  if (T > 1e8) return 0.21e-26 * sqrt(T);
  int if1 = (int)(log10(T) * 10) - 39;
  int if2 = if1 + 1;
  if (if1 < 1) if1 = 1;
  if (if2 > 41) if2 = 41;
  double T0 = p->cooltab[2 * (if1 - 1)], c0 = p->cooltab[2 * (if1 - 1) + 1];
  double T1 = p->cooltab[2 * (if2 - 1)], c1 = p->cooltab[2 * (if2 - 1) + 1];
  if (T1 == T0) return c0;
  return (c1 - c0) * (T - T0) / (T1 - T0) + c0;
}

// src/coolingdmc.f90:19-50 on one cell's conserved state and its primitives
template <int NEQ>
__device__ __forceinline__ void cool_dmc(const wx_params *__restrict__ p, double dt, const double *q, double T,
                                         double *uu, double &pcool) {
  pcool = q[3];
  if (T > 1.e4) {
    double Eth0 = p->cv * q[3];
    double Aloss = cooldmc(p, T);
    double dens = q[0];
    double Ce = (Aloss * (dens * dens)) / (Eth0 * p->Psc);
    double pn = q[3] * libm::wexp(-(Ce * dt));
    uu[3] = uu[3] - Eth0 + p->cv * pn;
    pcool = pn;   // the primitive the reference keeps (src/coolingdmc.f90:38)
  }
}

// Jet source (JET/jet.f90:41-77, through src/user_mod.f90:73-84).
struct JetState {
  double vjet;
};

__device__ __forceinline__ bool in_jet(const wx_params *__restrict__ p, int level, int icx,
                                       int icy, int i, int j) {
  double x = ((double)(i + icx) - 0.5) * p->dx[level - 1];
  double y = ((double)(j + icy) - 0.5) * p->dy[level - 1];
  return (fabs(x - p->jet[2]) <= p->jet[1]) && (fabs(y - p->jet[3]) <= p->jet[0]);
}

template <int NEQ>
__device__ __forceinline__ void jet_state(const wx_params *__restrict__ p, double vjet, double *uu) {
  const double den = p->jet[4];
  uu[0] = den;
  uu[1] = den * vjet;
  uu[2] = 0.;
  uu[3] = 0.5 * den * (vjet * vjet) + p->cv * den * p->jet[10] * p->jet[5];
  if constexpr (NEQ >= 5) uu[4] = den * p->jet[9];
  if constexpr (NEQ >= 6) uu[5] = den;
}

__device__ __forceinline__ double jet_velocity(const wx_params *__restrict__ p, double time) {
  const double pi = 3.141592653589793;  // acos(-1.)
  return p->jet[6] + p->jet[7] * libm::wsin(2. * pi * time / p->jet[8]);
}

// The source speed at `time`: the value the dt reduction stored for that
// time (the same function of the same time), else computed here.
__device__ __forceinline__ double jet_velocity_at(const wx_params *__restrict__ p, const DevScalars *S,
                                                  double time) {
  if (S->vjet_ok && S->vjet_time == time) return S->vjet;
  return jet_velocity(p, time);
}

}  // namespace wx
