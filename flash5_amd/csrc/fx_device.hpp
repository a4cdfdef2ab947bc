// fx_device.hpp -- device-side math of the unsplit hydro block update.
//
// Reference semantics (paths relative to
// source/physics/Hydro/HydroMain/unsplit):
//   primitive eigen system      hy_eigenParameters.F90:42-89,
//                               hy_eigenValue.F90:33-50,
//                               OnlyHydro/hy_eigenVector.F90:46-151
//   slope limiters              hy_slopeLimiters.F90:38-60
//   TVD slopes                  hy_TVDslope.F90:54-265
//   transverse flux sigma       hy_upwindTransverseFlux.F90:43-211
//   PPM + characteristic trace  hy_DataReconstructNormalDir_PPM.F90:73-958
//   HLLC                        hy_HLLC.F90:53-324, hy_prim2con.F90,
//                               hy_prim2flx.F90
//
// The eigenvectors are sparse (each left/right vector has at most three
// non-zero entries); the products below keep only those entries, in the
// reference's summation order, so that every non-zero result rounds the
// same way as the dense 5x5 form.
//
// Primitive vectors are double[8]: dens, velx, vely, velz, pres, gamc, game,
// eint.  Waves: 0 fast-left, 1 slow-left, 2 entropy, 3 slow-right,
// 4 fast-right.
#pragma once
#include <hip/hip_runtime.h>

#include "fx_hydro.h"

namespace fx {

enum { P_DENS = 0, P_VELX = 1, P_VELY = 2, P_VELZ = 3, P_PRES = 4, P_GAMC = 5,
       P_GAME = 6, P_EINT = 7 };

// Pointers read from device memory (a tile's U, flux and pavg arrays) are
// generic, and accesses through generic pointers compile to flat
// instructions, which also count against the LDS wait counter.  The arrays
// are device memory, so the kernels hold them as global-address-space
// pointers (gdouble*) from the point they are read; loads and stores through
// them are global instructions, which also take a scalar base address.
typedef __attribute__((address_space(1))) double gdouble;
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T* as_global(T* p) {
  return (__attribute__((address_space(1))) T*)p;
}

struct DevParams {
  int ndim, nxb, nyb, nzb, ng, nunk;
  int nx, ny, nz;            // guard-inclusive extents
  long ncell;                // cells per tile
  long voff[FX_NVAR_USED];   // var slot * ncell
  int lo[3], hi[3];          // interior limits, 0-based inclusive
  double gamma;
  int limiter;
  double beta;
  int charLim, flat, steep, ctu3d, aux, riemann, precision, learned;
  int velSlot[3];            // var slots of velx, vely, velz
  double fP, smlrho, smallE, eintSwitch, tiny;
  double gammam1, gam1inv, ggprodinv, abar;
  int exactMaxIter;
  double exactTol;
  long shokOff;              // SHOK_VAR slot * ncell, or -1 without shock detection
  int bext[3][3];            // [dir][axis] extent of the dir-band of state cells
  long bcells[3];            // cells per dir-band
  long boff[3];              // offset of each band in a tile's state scratch
  long scellsPerTile;        // sum of band cells
  int fext[3][3];            // [dir][axis] flux-array extents
  long nface[3];
  long icells;               // interior cells per tile
};

// Every routine below is templated on the real type R of the reconstruction:
// double in the FP64 modes, float in the mixed mode.  Literal constants are
// written R(c) so that the double instantiation performs exactly the FP64
// operations of the reference order.
template <typename R> struct EigT {
  R un, cf, ahinv, lfp, a2inv, rp, rho;
};
using Eig = EigT<double>;

// ---- FP64 quotients and roots without the range handling ----
// The compiler's FP64 division spends three of its eleven instructions, and
// its root eight of some twenty, on operands near the ends of the exponent
// range, and reciprocals of one divisor are not shared.  The forms below give
// the same bits between: a reciprocal from the hardware's (good to about 2^-24)
// by one cubic step, (1 + e + e^2) r0 with e = 1 - y r0, then Markstein's
// residual correction q + (x - y q) r in two FMAs.  They hold while the
// divisor, the quotient and the residual x - y q are normal: |x| at least
// 2^-960 (below, the quotient may differ in its last place), |x| and |y| below
// 2^1000 and y normal (else: NaN), and a zero quotient is +0.  The eigen
// systems and the exact solver check their operands (window_pos,
// exact_window) and divide plainly outside, HLLC its divisor; the van Leer
// limiter and the flattening check nothing, and drop the result where the
// divisor is zero.  So what differs from plain division is the last place of
// slopes of differences, or of star-state momenta, below about 2^-480 and
// 2^-960.  For a divisor of all-ones significand the hardware's estimate has
// to lie above 1/y, and gfx950's does.  tests/test_gpu_fast_division.py runs
// these functions against IEEE division and root,
// tests/cdiv/fast_div_check.c their steps from other starts.  The march and the
// 2-D/3-D steps are bound by instruction issue: 4096 x 16^3 FP64 HLLC step 6.02 ->
// 5.72 ms, 1024^2 in 64^2 blocks 492 -> 475 us a step, 1024 x 16^3 exact 3.15 ->
// 2.96 ms, the same bits.
__device__ __forceinline__ double recip_fast(double y) {
  const double r0 = __builtin_amdgcn_rcp(y);
  const double e = fma(-y, r0, 1.0);
  return fma(r0, fma(e, e, e), r0);
}
// the correctly rounded reciprocal, for quotients that share it
__device__ __forceinline__ double recip_rn(double y) {
  const double r = recip_fast(y);
  return fma(fma(-y, r, 1.0), r, r);
}
__device__ __forceinline__ double quot_r(double x, double y, double r) {
  const double q = x * r;
  return fma(fma(-y, q, x), r, q);
}
__device__ __forceinline__ double quot(double x, double y) { return quot_r(x, y, recip_fast(y)); }
// sqrt(x) by a coupled Newton step on x r and r / 2, then two residual
// corrections (Markstein)
__device__ __forceinline__ double sqrt_fast(double x) {
  const double r = __builtin_amdgcn_rsq(x);
  double g = x * r, h = 0.5 * r;
  const double d = fma(-h, g, 0.5);
  g = fma(g, d, g);
  h = fma(h, d, h);
  g = fma(fma(-g, g, x), h, g);
  return fma(fma(-g, g, x), h, g);
}
// 2^-400 <= x < 2^400 (x > 0), as an unsigned distance of the high word that
// is at least kWindow outside
constexpr unsigned kWindow = 800u << 20;
__device__ __forceinline__ unsigned window_pos(double x) {
  return (unsigned)(__builtin_bit_cast(unsigned long long, x) >> 32) - ((1023u - 400u) << 20);
}

// x / y as the compiler divides in FP32 at the accuracy the FP32 code is
// built for (LLVM's AMDGPU lowering of fdiv with 2.5 ulp allowed: a reciprocal
// and a product, y scaled down by 2^-32 above 2^96, where the reciprocal would
// be flushed), spelled out: where code merges two branches' divisions
// into one, the compiler drops that accuracy setting and emits the correctly
// rounded sequence, with other bits.
__device__ __forceinline__ float quot(float x, float y) {
  const float s = fabsf(y) > 0x1p+96f ? 0x1p-32f : 1.f;
  return s * (x * __builtin_amdgcn_rcpf(y * s));
}

// False on an imaginary (or undefined) sound speed; e is then NaN or
// infinite.  The parts are formed either way: no branch separates them from
// the caller's arithmetic.
template <int DIR, typename R>
__device__ __forceinline__ bool eig_make(const R* V, EigT<R>& e) {
  e.rho = V[P_DENS];
  e.un = V[P_VELX + DIR];
  const R gp = V[P_GAMC] * V[P_PRES];
  R a2;
  if constexpr (sizeof(R) == sizeof(double)) {
    // the window holds every wave's states but degenerate ones
    const unsigned wd = window_pos(V[P_DENS]), wp = window_pos(gp);
    if (__builtin_expect(__any((wd > wp ? wd : wp) >= kWindow) == 0, 1)) {
      const double dinv = recip_rn(V[P_DENS]);
      a2 = quot_r(gp, V[P_DENS], dinv);
      e.cf = sqrt_fast(a2);
      const double a2e = e.cf * e.cf;
      e.a2inv = recip_rn(a2e);
      e.ahinv = quot(0.5, e.cf);
      e.lfp = dinv * (0.5 * e.a2inv);
      e.rp = V[P_DENS] * a2e;
      return a2 > 0.0;
    }
  }
  a2 = gp / V[P_DENS];
  e.cf = sqrt(a2);
  const R dinv = R(1.0) / V[P_DENS];
  const R a2e = e.cf * e.cf;
  e.a2inv = R(1.0) / a2e;
  e.ahinv = R(0.5) / e.cf;
  const R Na = R(0.5) * e.a2inv;
  e.lfp = dinv * Na;
  e.rp = V[P_DENS] * a2e;
  return a2 > R(0.0);
}

template <typename R>
__device__ __forceinline__ void eig_lambda(const EigT<R>& e, R lam[5]) {
  lam[0] = e.un - e.cf;
  lam[1] = e.un;
  lam[2] = e.un;
  lam[3] = e.un;
  lam[4] = e.un + e.cf;
}

// velocity slots normal / first / second transverse to DIR
template <int DIR> struct Vel {
  static constexpr int v1 = 1 + DIR, v2 = 1 + (DIR + 1) % 3, v3 = 1 + (DIR + 2) % 3;
};

// L_n . d over the five primitive slots
template <int DIR, int N, typename R>
__device__ __forceinline__ R eig_left1(const EigT<R>& e, const R* d) {
  constexpr int v1 = Vel<DIR>::v1, v2 = Vel<DIR>::v2, v3 = Vel<DIR>::v3;
  if constexpr (N == 0) return (-e.ahinv) * d[v1] + e.lfp * d[P_PRES];
  else if constexpr (N == 1) return d[v2];
  else if constexpr (N == 2) return d[P_DENS] + (-e.a2inv) * d[P_PRES];
  else if constexpr (N == 3) return d[v3];
  else return e.ahinv * d[v1] + e.lfp * d[P_PRES];
}

template <int DIR, typename R>
__device__ __forceinline__ void eig_left(const EigT<R>& e, const R* d, R w[5]) {
  w[0] = eig_left1<DIR, 0>(e, d);
  w[1] = eig_left1<DIR, 1>(e, d);
  w[2] = eig_left1<DIR, 2>(e, d);
  w[3] = eig_left1<DIR, 3>(e, d);
  w[4] = eig_left1<DIR, 4>(e, d);
}

// out[0..4] = sum_n R_n * w[n]
template <int DIR, typename R>
__device__ __forceinline__ void eig_right(const EigT<R>& e, const R w[5], R* out) {
  constexpr int v1 = Vel<DIR>::v1, v2 = Vel<DIR>::v2, v3 = Vel<DIR>::v3;
  out[P_DENS] = e.rho * w[0] + w[2] + e.rho * w[4];
  out[v1] = (-e.cf) * w[0] + e.cf * w[4];
  out[v2] = w[1];
  out[v3] = w[3];
  out[P_PRES] = e.rp * w[0] + e.rp * w[4];
}

template <typename R> __device__ __forceinline__ R sgn1(R a) { return copysign(R(1.0), a); }

// Limited value of two one-sided differences (hy_slopeLimiters.F90:38-60).
// Straight-line code: van Leer divides in every lane and selects after.
template <int KIND, typename R>
__device__ __forceinline__ R limit(R a, R b, R beta) {
  if constexpr (KIND == FX_MINMOD) {
    return R(.5) * (sgn1(a) + sgn1(b)) * fmin(fabs(a), fabs(b));
  } else if constexpr (KIND == FX_VANLEER) {
    const R q = quot(R(2.) * a * b, a + b);
    return (a * b <= R(0.)) ? R(0.) : q;
  } else if constexpr (KIND == FX_LIMITED) {
    const R hi = fmax(fmax(R(0.), fmin(beta * a, b)), fmin(a, beta * b));
    const R lo = fmin(fmin(R(0.), fmax(beta * a, b)), fmax(a, beta * b));
    return b > R(0.) ? hi : lo;
  } else {  // FX_MC
    return (sgn1(a) + sgn1(b)) * fmin(fmin(fabs(a), R(.25) * fabs(a + b)), fabs(b));
  }
}

// Limited slope of the cell whose eigen system is e (hy_TVDslope), projected
// back to primitive slopes when characteristic limiting is on
// (PPM.F90:523-570): out[dens, velocities, pres, eint] (the gamma slots stay
// unset; a face state takes its cell's gammas).  KIND limits the entropy
// wave and the scalars, KW the other waves (they differ for FX_HYBRID only).
// The kinds are told apart once per cell, outside the arithmetic: told apart
// within each wave's limiter, the choice cut a cell's slope into some sixty
// basic blocks, each with its own division chain to wait for (and the
// operands of every minimum and maximum re-quieted, since a value that
// crosses blocks is not known to be quiet).  With straight-line limiters,
// monotone limits and eigen systems the FP64 march of 4096 x 16^3 has 364
// basic blocks instead of 1,499 and takes 6.0 instead of 7.0 ms.
template <int DIR, int KIND, int KW, typename R>
__device__ __forceinline__ void tvd_slope_kind(const DevParams& P, const R* VL, const R* V0,
                                               const R* VR, const EigT<R>& e, R out[8]) {
  const R beta = R(P.beta);
  R dL[8], dR[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    if (k == P_GAMC || k == P_GAME) continue;
    dL[k] = V0[k] - VL[k];
    dR[k] = VR[k] - V0[k];
  }
  out[P_EINT] = limit<KIND>(dL[P_EINT], dR[P_EINT], beta);
  if (P.charLim) {
    R a[5], b[5], w[5];
    eig_left<DIR>(e, dL, a);
    eig_left<DIR>(e, dR, b);
#pragma unroll
    for (int n = 0; n < 5; ++n)
      w[n] = n == 2 ? limit<KIND>(a[n], b[n], beta) : limit<KW>(a[n], b[n], beta);
    eig_right<DIR>(e, w, out);
  } else {
    out[P_DENS] = limit<KIND>(dL[P_DENS], dR[P_DENS], beta);
#pragma unroll
    for (int k = P_VELX; k <= P_PRES; ++k) out[k] = limit<KW>(dL[k], dR[k], beta);
    if (KIND != KW) out[P_EINT] = R(0.);
  }
}

template <int DIR, typename R>
__device__ __forceinline__ void tvd_slope(const DevParams& P, const R* VL, const R* V0,
                                          const R* VR, const EigT<R>& e, R out[8]) {
  switch (P.limiter) {
    case FX_VANLEER: tvd_slope_kind<DIR, FX_VANLEER, FX_VANLEER>(P, VL, V0, VR, e, out); break;
    case FX_MINMOD: tvd_slope_kind<DIR, FX_MINMOD, FX_MINMOD>(P, VL, V0, VR, e, out); break;
    case FX_LIMITED: tvd_slope_kind<DIR, FX_LIMITED, FX_LIMITED>(P, VL, V0, VR, e, out); break;
    case FX_HYBRID: tvd_slope_kind<DIR, FX_MC, FX_MINMOD>(P, VL, V0, VR, e, out); break;
    default: tvd_slope_kind<DIR, FX_MC, FX_MC>(P, VL, V0, VR, e, out); break;
  }
}

// Transverse flux sigma of one cell (hy_upwindTransverseFlux, order 1).
template <int DIR, typename R>
__device__ __forceinline__ void trans_sigma(const DevParams& P, const R* vm1, const R* vc0,
                                            const R* vp1, const EigT<R>& e, R sig[8]) {
  R lam[5];
  eig_lambda(e, lam);
  constexpr int v1 = Vel<DIR>::v1, v2 = Vel<DIR>::v2, v3 = Vel<DIR>::v3;
#pragma unroll
  for (int v = 0; v < 8; ++v) sig[v] = R(0.);
  R dm[5], dp[5];
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    dm[v] = vc0[v] - vm1[v];
    dp[v] = vp1[v] - vc0[v];
  }
  // upwinded characteristic amplitude of wave N
#define FX_TS_DB(N) (lam[N] > R(0.) ? eig_left1<DIR, N>(e, dm) : eig_left1<DIR, N>(e, dp))
  {
    const R db = FX_TS_DB(0);
    sig[P_DENS] = sig[P_DENS] + lam[0] * e.rho * db;
    sig[v1] = sig[v1] + lam[0] * (-e.cf) * db;
    sig[P_PRES] = sig[P_PRES] + lam[0] * e.rp * db;
  }
  { const R db = FX_TS_DB(1); sig[v2] = sig[v2] + lam[1] * db; }
  { const R db = FX_TS_DB(2); sig[P_DENS] = sig[P_DENS] + lam[2] * db; }
  { const R db = FX_TS_DB(3); sig[v3] = sig[v3] + lam[3] * db; }
  {
    const R db = FX_TS_DB(4);
    sig[P_DENS] = sig[P_DENS] + lam[4] * e.rho * db;
    sig[v1] = sig[v1] + lam[4] * e.cf * db;
    sig[P_PRES] = sig[P_PRES] + lam[4] * e.rp * db;
  }
#undef FX_TS_DB
  if (P.aux) {
    const R d = (lam[2] > R(0.)) ? vc0[P_EINT] - vm1[P_EINT] : vp1[P_EINT] - vc0[P_EINT];
    sig[P_EINT] = lam[2] * d;
  }
}

// x / C for C = 3, 6, 12 with the IEEE quotient's bits, in four FP64
// instructions instead of the division sequence (a quarter-rate reciprocal
// and about ten instructions).  q = x RN(1/C) is faithful, so rho = x - q C
// is exact in one FMA; q + rho RN(1/C), rounded once by a second FMA, lies
// within 2^-52 ulp of x/C.  As C = 3 * 2^k, a normal quotient x/C sits 0,
// 1/3 or 2/3 of an ulp past a double, never within 1/6 ulp of a rounding
// midpoint, so both round alike; copysign keeps the sign of a zero.  This
// holds for every finite x whose quotient is normal or zero (checked against
// IEEE division by tests/cdiv/const_div_check.c); for C = 6 and 12 a
// quotient below 2^-1022 may differ in its last place, and an infinite x
// gives NaN (fma(-inf, C, inf)) where IEEE division gives inf.  Those are the
// limits of the bitwise-parity claim: states whose PPM differences are
// subnormal or infinite.  FP32 divides.
template <int C>
__device__ __forceinline__ double div_const(double x) {
  static_assert(C == 3 || C == 6 || C == 12, "constants of the form 3 * 2^k");
  constexpr double r = 1.0 / C;
  const double q = x * r;
  const double rho = fma(-q, double(C), x);
  return copysign(fma(rho, r, q), x);
}
template <int C>
__device__ __forceinline__ float div_const(float x) {
  return x / float(C);
}

// PPM interface values, limiting and characteristic tracing from the three
// projected slopes of cells i-1, i, i+1 (PPM.F90:578-842).  Vm/Vc/Vp are the
// primitive vectors of i-1, i, i+1; densMM/densPP the densities of i-2, i+2
// (contact steepening only).
template <int DIR, typename R>
__device__ __forceinline__ void ppm_trace(const DevParams& P, R dtn, R delta, const R* Vm,
                                          const R* Vc, const R* Vp, R densMM, R densPP,
                                          const R* dbN, const R* db0, const R* dbP, R flatC,
                                          const EigT<R>& e0, R Wp[8], R Wm[8]) {
  R Vmm[1] = {densMM}, Vpp[1] = {densPP};
  // every traced variable: dens, velocities, pres, eint (eint is carried along
  // when the aux equation is off, where nothing reads it)
  constexpr auto traced = [](int v) { return v <= P_PRES || v == P_EINT; };
  R vL[8], vR[8];
#pragma unroll
  for (int v = 0; v < 8; ++v) {
    if (!traced(v)) continue;
    vL[v] = R(0.5) * (Vc[v] + Vm[v]) - div_const<6>(db0[v] - dbN[v]);
    vR[v] = R(0.5) * (Vc[v] + Vp[v]) - div_const<6>(dbP[v] - db0[v]);
  }
  if (P.steep) {
    const R temp1 = Vp[P_DENS] - Vm[P_DENS];
    if (fabs(temp1) > R(P.tiny)) {
      const R d2R = (Vpp[0] - R(2.) * Vp[P_DENS] + Vc[P_DENS]) / (R(6.) * delta * delta);
      const R d2L = (Vc[P_DENS] - R(2.) * Vm[P_DENS] + Vmm[0]) / (R(6.) * delta * delta);
      R eta = (d2L - d2R) * (delta * delta) / temp1;
      if (d2R * d2L >= R(0.)) eta = R(0.);
      if (R(0.01) * fmin(Vp[P_DENS], Vm[P_DENS]) - fabs(Vp[P_DENS] - Vm[P_DENS]) >= R(0.)) eta = R(0.);
      eta = fmax(R(0.), fmin(R(1.), R(20.0) * (eta - R(0.05))));
      const R t2 = fabs(Vp[P_PRES] - Vm[P_PRES]) / fmin(Vp[P_PRES], Vm[P_PRES]);
      const R t3 = fabs(Vp[P_DENS] - Vm[P_DENS]) / fmin(Vp[P_DENS], Vm[P_DENS]);
      if (Vc[P_GAME] * R(0.1) * t3 - t2 < R(0.0)) eta = R(0.);
      vL[P_DENS] = vL[P_DENS] * (R(1.) - eta) + (Vm[P_DENS] + R(0.5) * dbN[P_DENS]) * eta;
      vR[P_DENS] = vR[P_DENS] * (R(1.) - eta) + (Vp[P_DENS] - R(0.5) * dbP[P_DENS]) * eta;
    }
  }
  // one branch for the flattening of all variables; the monotone limits are
  // selects, so the variables' chains interleave
  if (P.flat) {
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      if (!traced(n)) continue;
      vL[n] = flatC * Vc[n] + (R(1.0) - flatC) * vL[n];
      vR[n] = flatC * Vc[n] + (R(1.0) - flatC) * vR[n];
    }
  }
  R dW[8], W6[8];
#pragma unroll
  for (int n = 0; n < 8; ++n) {
    if (!traced(n)) continue;
    const bool ext = (vR[n] - Vc[n]) * (Vc[n] - vL[n]) <= R(0.);
    vL[n] = ext ? Vc[n] : vL[n];
    vR[n] = ext ? Vc[n] : vR[n];
    R dd = vR[n] - vL[n];
    const R l3 = R(3.) * Vc[n] - R(2.) * vR[n];
    vL[n] = (R(6.) * (vR[n] - vL[n]) * (Vc[n] - R(0.5) * (vL[n] + vR[n])) > dd * dd) ? l3 : vL[n];
    dd = vR[n] - vL[n];
    const R r3 = R(3.) * Vc[n] - R(2.) * vL[n];
    vR[n] = (R(6.) * (vR[n] - vL[n]) * (Vc[n] - R(0.5) * (vL[n] + vR[n])) < -(dd * dd)) ? r3 : vR[n];
    dW[n] = vR[n] - vL[n];
    W6[n] = R(6.) * (Vc[n] - R(0.5) * (vR[n] + vL[n]));
  }
  R lam[5];
  eig_lambda(e0, lam);
  const R hdtn = R(0.5) * dtn;
  const R four3 = R(4.) / R(3.);
  {
    // eint, upwinded with the entropy wave
    constexpr int v = P_EINT;
    const R a = fmax(lam[2], R(0.)), b = -fmin(lam[2], R(0.));
    Wp[v] = vR[v] - a * hdtn * (dW[v] - (R(1.0) - div_const<3>(a * hdtn * R(4.))) * W6[v]);
    Wm[v] = vL[v] + b * hdtn * (dW[v] + (R(1.0) - div_const<3>(b * hdtn * R(4.))) * W6[v]);
  }
  Wp[P_GAMC] = Vc[P_GAMC];
  Wp[P_GAME] = Vc[P_GAME];
  Wm[P_GAMC] = Vc[P_GAMC];
  Wm[P_GAME] = Vc[P_GAME];
  // characteristic tracing (PPM.F90:751-800): the branch of every solver but
  // Roe's, which fx_hydro_init refuses
  R sL[5] = {R(0.), R(0.), R(0.), R(0.), R(0.)}, sR[5] = {R(0.), R(0.), R(0.), R(0.), R(0.)};
  R mW6[5];
#pragma unroll
  for (int v = 0; v < 5; ++v) mW6[v] = -W6[v];
  constexpr int v1 = Vel<DIR>::v1, v2 = Vel<DIR>::v2, v3 = Vel<DIR>::v3;
  R cA[5], cB[5];
  eig_left<DIR>(e0, dW, cA);
  eig_left<DIR>(e0, mW6, cB);
  // contribution of wave N through its right-eigenvector entry RV at slot V
#define FX_TRACE(N, V, RV)                                                              \
  {                                                                                     \
    const R x = dtn * lam[N];                                                           \
    sL[V] = sL[V] + (R(.5) * (R(-1.) - x) * (RV) * cA[N] +                              \
                     R(.25) * (R(1.) + R(2.) * dtn * lam[N] + four3 * (x * x)) * (RV) * cB[N]); \
    sR[V] = sR[V] + (R(.5) * (R(1.) - x) * (RV) * cA[N] +                               \
                     R(.25) * (R(1.) - R(2.) * dtn * lam[N] + four3 * (x * x)) * (RV) * cB[N]); \
  }
  FX_TRACE(0, P_DENS, e0.rho)
  FX_TRACE(0, v1, -e0.cf)
  FX_TRACE(0, P_PRES, e0.rp)
  FX_TRACE(1, v2, R(1.))
  FX_TRACE(2, P_DENS, R(1.))
  FX_TRACE(3, v3, R(1.))
  FX_TRACE(4, P_DENS, e0.rho)
  FX_TRACE(4, v1, e0.cf)
  FX_TRACE(4, P_PRES, e0.rp)
#undef FX_TRACE
#pragma unroll
  for (int v = 0; v <= P_PRES; ++v) {
    Wm[v] = Vc[v] + div_const<12>(W6[v]) + sL[v];
    Wp[v] = Vc[v] + div_const<12>(W6[v]) + sR[v];
  }
}

template <int DIR, typename R>
__device__ __forceinline__ bool ppm_full(const DevParams& P, R dtn, R delta, const R* Vmm,
                                         const R* Vm, const R* Vc, const R* Vp, const R* Vpp,
                                         R flatC, const EigT<R>& e0, R Wp[8], R Wm[8]) {
  EigT<R> eP, eN;
  if (!eig_make<DIR>(Vp, eP)) return false;
  if (!eig_make<DIR>(Vm, eN)) return false;
  R dbN[8], db0[8], dbP[8];
  tvd_slope<DIR>(P, Vmm, Vm, Vc, eN, dbN);
  tvd_slope<DIR>(P, Vm, Vc, Vp, e0, db0);
  tvd_slope<DIR>(P, Vc, Vp, Vpp, eP, dbP);
  ppm_trace<DIR>(P, dtn, delta, Vm, Vc, Vp, Vmm[P_DENS], Vpp[P_DENS], dbN, db0, dbP, flatC, e0, Wp,
                 Wm);
  return true;
}

// ---- HLLC (hy_HLLC.F90:53-324) ----
template <int DIR, typename R>
__device__ __forceinline__ void prim2flx(const R* V, R fP, R F[6]) {
  const R u2 = V[P_VELX] * V[P_VELX] + V[P_VELY] * V[P_VELY] + V[P_VELZ] * V[P_VELZ];
  const R E = R(0.5) * V[P_DENS] * u2 + V[P_PRES] / (V[P_GAME] - R(1.));
  const R un = V[P_VELX + DIR];
  F[5] = V[P_PRES];
  F[0] = V[P_DENS] * un;
  F[1] = F[0] * V[P_VELX];
  F[2] = F[0] * V[P_VELY];
  F[3] = F[0] * V[P_VELZ];
  F[1 + DIR] = F[1 + DIR] + fP * V[P_PRES];
  F[4] = (E + V[P_PRES]) * un;
}

// returns 0 ok, 1 imaginary sound speed
template <int DIR, typename R>
__device__ __forceinline__ int hllc(const DevParams& P, const R* Vm, const R* Vp, R F[6]) {
  const R tiny = R(P.tiny), fP = R(P.fP);
  const R velNL = Vm[P_VELX + DIR], velNR = Vp[P_VELX + DIR];
  const R aL2 = Vm[P_GAMC] * Vm[P_PRES] / Vm[P_DENS];
  const R aR2 = Vp[P_GAMC] * Vp[P_PRES] / Vp[P_DENS];
  if ((Vm[P_DENS] < tiny && Vm[P_DENS] > R(0.)) || (Vp[P_DENS] < tiny && Vp[P_DENS] > R(0.)) ||
      (Vm[P_PRES] < tiny && Vm[P_PRES] > R(0.)) || (Vp[P_PRES] < tiny && Vp[P_PRES] > R(0.))) {
#pragma unroll
    for (int f = 0; f < 6; ++f) F[f] = R(0.);
    return 0;
  }
  if (aL2 < R(0.) || aR2 < R(0.)) return 1;
  const R cfL = sqrt(aL2), cfR = sqrt(aR2);
  const R SL = fmin(velNL - cfL, velNR - cfR);
  const R SR = fmax(velNL + cfL, velNR + cfR);
  const R tpL = Vm[P_PRES], tpR = Vp[P_PRES];
  R qStar = (Vp[P_DENS] * velNR * (SR - velNR) - Vm[P_DENS] * velNL * (SL - velNL) + tpL - tpR -
             R(0.) * R(0.) + R(0.) * R(0.));
  qStar = qStar / (Vp[P_DENS] * (SR - velNR) - Vm[P_DENS] * (SL - velNL));
  if (SL >= R(0.)) {
    prim2flx<DIR>(Vm, fP, F);
    return 0;
  }
  if (!(qStar < R(0.) && SR >= R(0.)) && !(SL < R(0.) && qStar >= R(0.))) {
    prim2flx<DIR>(Vp, fP, F);
    return 0;
  }
  const bool left = (SL < R(0.) && qStar >= R(0.));
  // element-wise select keeps both inputs in registers (a pointer select
  // between two private arrays would put them in scratch memory)
  R V[8];
#pragma unroll
  for (int v = 0; v < 8; ++v) V[v] = left ? Vm[v] : Vp[v];
  const R S = left ? SL : SR;
  const R velN = left ? velNL : velNR;
  const R tp = left ? tpL : tpR;
  const R numer = S - velN, denom = S - qStar;
  const R pStar = Vm[P_DENS] * (SL - velNL) * (qStar - velNL) + tpL;
  // the chosen side's flux, built in F itself (a second private array here
  // ends up in scratch memory after inlining)
  prim2flx<DIR>(V, fP, F);
  // conserved state of the chosen side (hy_prim2con.F90)
  const R u2 = V[P_VELX] * V[P_VELX] + V[P_VELY] * V[P_VELY] + V[P_VELZ] * V[P_VELZ];
  R Uc[5];
  Uc[0] = V[P_DENS];
  Uc[1] = V[P_DENS] * V[P_VELX];
  Uc[2] = V[P_DENS] * V[P_VELY];
  Uc[3] = V[P_DENS] * V[P_VELZ];
  Uc[4] = R(0.5) * V[P_DENS] * u2 + V[P_PRES] / (V[P_GAME] - R(1.)) + R(0.5) * R(0.);
  // the five quotients by denom (nonzero: S and qStar lie on either side of
  // zero or S is past it) share one reciprocal in FP64
  R Us[5], num[5];
#pragma unroll
  for (int m = 0; m < 4; ++m) num[m] = Uc[m] * numer;
  num[4] = Uc[4] * numer;
  const R work = pStar * qStar - tp * velN;
  bool shared = false;
  if constexpr (sizeof(R) == sizeof(double))
    shared = __any(window_pos(fabs(denom)) >= kWindow) == 0;
  R workQ;
  if (__builtin_expect(shared, 1)) {
    if constexpr (sizeof(R) == sizeof(double)) {
      const double rd = recip_rn(denom);
#pragma unroll
      for (int m = 0; m < 5; ++m) Us[m] = quot_r(num[m], denom, rd);
      workQ = quot_r(work, denom, rd);
    }
  } else {
#pragma unroll
    for (int m = 0; m < 5; ++m) Us[m] = num[m] / denom;
    workQ = work / denom;
  }
  const R dStar = Us[0];
  Us[4] = Us[4] + workQ;
  Us[1 + DIR] = dStar * qStar;
#pragma unroll
  for (int f = 0; f < 5; ++f) F[f] = F[f] + S * (Us[f] - Uc[f]);
  return 0;
}

// ---- HLL (hy_HLL.F90:82-165) ----
// conserved state (hy_prim2con.F90): dens, three momenta, total energy
template <typename R>
__device__ __forceinline__ void prim2con(const R* V, R Uc[5]) {
  const R u2 = V[P_VELX] * V[P_VELX] + V[P_VELY] * V[P_VELY] + V[P_VELZ] * V[P_VELZ];
  Uc[0] = V[P_DENS];
  Uc[1] = V[P_DENS] * V[P_VELX];
  Uc[2] = V[P_DENS] * V[P_VELY];
  Uc[3] = V[P_DENS] * V[P_VELZ];
  Uc[4] = R(0.5) * V[P_DENS] * u2 + V[P_PRES] / (V[P_GAME] - R(1.)) + R(0.5) * R(0.);
}

// returns 0 ok, 1 imaginary sound speed.  The fan average runs over all six
// slots; the pressure slot's state jump is zero (hy_HLL.F90:146).
template <int DIR, typename R>
__device__ __forceinline__ int hll(const DevParams& P, const R* Vm, const R* Vp, R F[6]) {
  const R tiny = R(P.tiny), fP = R(P.fP);
  const R velNL = Vm[P_VELX + DIR], velNR = Vp[P_VELX + DIR];
  const R aL2 = Vm[P_GAMC] * Vm[P_PRES] / Vm[P_DENS];
  const R aR2 = Vp[P_GAMC] * Vp[P_PRES] / Vp[P_DENS];
  if ((Vm[P_DENS] < tiny && Vm[P_DENS] > R(0.)) || (Vp[P_DENS] < tiny && Vp[P_DENS] > R(0.)) ||
      (Vm[P_PRES] < tiny && Vm[P_PRES] > R(0.)) || (Vp[P_PRES] < tiny && Vp[P_PRES] > R(0.))) {
#pragma unroll
    for (int f = 0; f < 6; ++f) F[f] = R(0.);
    return 0;
  }
  if (aL2 < R(0.) || aR2 < R(0.)) return 1;
  const R cfL = sqrt(aL2), cfR = sqrt(aR2);
  const R SL = fmin(velNL - cfL, velNR - cfR);
  const R SR = fmax(velNL + cfL, velNR + cfR);
  if (SL > R(0.)) {
    prim2flx<DIR>(Vm, fP, F);
    return 0;
  }
  if (SR < R(0.)) {
    prim2flx<DIR>(Vp, fP, F);
    return 0;
  }
  R FL[6], FR[6], UL[5], UR[5];
  prim2flx<DIR>(Vm, fP, FL);
  prim2flx<DIR>(Vp, fP, FR);
  prim2con(Vm, UL);
  prim2con(Vp, UR);
#pragma unroll
  for (int f = 0; f < 6; ++f) {
    const R dU = f < 5 ? UR[f] - UL[f] : R(0.0) - R(0.0);
    F[f] = (SR * FL[f] - SL * FR[f] + SR * SL * dU) / (SR - SL);
  }
  return 0;
}

// ---- exact Riemann solver for the gamma-law gas (no counterpart in the
// reference; it takes hy_HLLC.F90's contract).  Newton iteration on the
// exact pressure function (Toro, Riemann Solvers and Numerical Methods, 3rd
// ed., eqs. 4.6-4.9, derivative 4.37), seeded by a caller guess or by the
// two-shock guess (Toro eq. 9.42), sampled at x/t = 0 (Toro sec. 4.5).  The
// operation order follows the CPU oracle's restatement, except where a power
// follows from one already taken: the rarefaction derivative reuses the
// value's power, the density behind a rarefaction is gamma p / c^2, and the
// fan pressure's power is the density's times (c/ck)^2; and powers are taken
// as exp2(e log2 x) (pow_pos) where the oracle calls pow.

// x^e for x > 0 as exp2(e log2 x).  In FP64 this is about 130 instructions
// against pow's 230 (pow also handles signs, integer exponents and extra
// precision that positive pressure and sound-speed ratios do not need); its
// error, a few ulp, is far below the solver's 1e-12 convergence tolerance.
// In FP32 it is the hardware log2 and exp2.  x = 0 gives 0, as pow does for
// e > 0.
__device__ __forceinline__ double pow_pos(double x, double e) { return exp2(e * log2(x)); }
__device__ __forceinline__ float pow_pos(float x, float e) { return exp2f(e * log2f(x)); }

// The FP64 solver is bound by instruction issue, so it is built twice.  FAST
// forms its quotients and roots without range handling (quot, recip_rn,
// sqrt_fast): the same bits while the states are inside exact_window, which a
// wavefront checks once per problem.  The other build serves wavefronts with a
// state outside.  With what gamma and a side alone give taken out of the
// iteration, and one copy of the sampling for both sides: k_solve_update on 1024
// blocks of 16^3 1574 -> 1316 us, 4M seeded problems 1015 -> 880 us.
template <bool FAST> struct ExactOps {
  static __device__ __forceinline__ double div(double x, double y) {
    return FAST ? quot(x, y) : x / y;
  }
  // several quotients by y
  static __device__ __forceinline__ double recip(double y) { return FAST ? recip_rn(y) : y; }
  static __device__ __forceinline__ double divr(double x, double y, double r) {
    return FAST ? quot_r(x, y, r) : x / y;
  }
  static __device__ __forceinline__ double root(double x) { return FAST ? sqrt_fast(x) : sqrt(x); }
};

// Densities and pressures within 2^-96 .. 2^96, velocity differences up to 2^96,
// gamma - 1 within 2^-10 .. 2^10: with p* at most some 2^300 and an iterate of
// 1e-30 or more every quotient and divisor stays far inside 2^+-1000 and every
// root inside 2^+-410.
__device__ __forceinline__ bool exact_window(double g, double rl, double pl, double rr, double pr,
                                             double du) {
  constexpr double W = 0x1p+96;
  const double lo = fmin(fmin(rl, rr), fmin(pl, pr)), hi = fmax(fmax(rl, rr), fmax(pl, pr));
  const double g1 = g - 1.;
  return lo >= 1. / W && hi <= W && fabs(du) <= W && g1 >= 0x1p-10 && g1 <= 0x1p+10;
}

// what the pressure function takes from gamma alone, and from one side's state
struct ExactGas {
  double g, t1, e1, gr, gp1;   // 2/(g-1), (g-1)/(2g), (g-1)/(g+1), g+1
};
struct ExactSide {
  double rho, p, c;
  double fr, ir;   // rarefaction: 2/(g-1) c, 1/(rho c)
  double ak, bk;   // shock: 2/((g+1) rho), (g-1)/(g+1) p
};
template <bool FAST>
__device__ __forceinline__ ExactGas exact_gas(double g) {
  using O = ExactOps<FAST>;
  ExactGas G;
  G.g = g;
  G.gp1 = g + 1.;
  G.t1 = O::div(2., g - 1.);
  G.e1 = O::div(g - 1., 2. * g);
  G.gr = O::div(g - 1., G.gp1);
  return G;
}
template <bool FAST>
__device__ __forceinline__ ExactSide exact_side(const ExactGas& G, double rho, double p, double c) {
  using O = ExactOps<FAST>;
  ExactSide s;
  s.rho = rho;
  s.p = p;
  s.c = c;
  s.fr = G.t1 * c;
  s.ir = O::div(1., rho * c);
  s.ak = O::div(2., G.gp1 * rho);
  s.bk = G.gr * p;
  return s;
}

template <bool FAST>
__device__ __forceinline__ void exact_fk(double p, const ExactGas& G, const ExactSide& s, double& f,
                                         double& fd) {
  using O = ExactOps<FAST>;
  if (p <= s.p) {
    // rarefaction: the derivative's power is the value's divided by pratio,
    // since (g - 1)/(2g) + (g + 1)/(2g) = 1 (one pow instead of two)
    const double pratio = O::div(p, s.p);
    const double q = pow_pos(pratio, G.e1);
    f = s.fr * (q - 1.);
    fd = s.ir * O::div(q, pratio);
  } else {
    const double bp = s.bk + p, rb = O::recip(bp);
    const double qrt = O::root(O::divr(s.ak, bp, rb));
    f = (p - s.p) * qrt;
    fd = (1. - O::divr(0.5 * (p - s.p), bp, rb)) * qrt;
  }
}

template <bool FAST>
__device__ __forceinline__ double two_shock_guess(double ul, const ExactSide& L, double ur,
                                             const ExactSide& Q) {
  using O = ExactOps<FAST>;
  const double ppv = 0.5 * (L.p + Q.p) - 0.125 * (ur - ul) * (L.rho + Q.rho) * (L.c + Q.c);
  const double p0 = fmax(1.e-30, ppv);
  const double gl = O::root(O::div(L.ak, L.bk + p0));
  const double gr = O::root(O::div(Q.ak, Q.bk + p0));
  const double pts = O::div(gl * L.p + gr * Q.p - (ur - ul), gl + gr);
  return fmax(1.e-30, pts);
}

// Newton from the better of two starts: the pressure function is evaluated
// at both, and the iteration begins at the one with the smaller residual
// |f(p)| (its f and f' serve the first step).  pb <= 0 means no second
// start: plain Newton from pa, in the CPU oracle's operation order.
// Returns iterations, negative when maxit was reached; pick = 0 when pa was
// taken.
template <bool FAST>
__device__ __forceinline__ int exact_newton_pick(const ExactGas& G, const ExactSide& L,
                                                 const ExactSide& Q, double du, double pa, double pb,
                                                 double tol, int maxit, double& pstar, int& pick) {
  using O = ExactOps<FAST>;
  double fl, fld, fr, frd;
  exact_fk<FAST>(pa, G, L, fl, fld);
  exact_fk<FAST>(pa, G, Q, fr, frd);
  double p = pa;
  double f = fl + fr + du, fd = fld + frd;
  pick = 0;
  if (pb > 0.) {
    double gl, gld, gr, grd;
    exact_fk<FAST>(pb, G, L, gl, gld);
    exact_fk<FAST>(pb, G, Q, gr, grd);
    const double fb = gl + gr + du;
    if (!(fabs(f) <= fabs(fb))) {
      pick = 1;
      p = pb;
      f = fb;
      fd = gld + grd;
    }
  }
  for (int it = 1; it <= maxit; ++it) {
    if (it > 1) {
      exact_fk<FAST>(p, G, L, fl, fld);
      exact_fk<FAST>(p, G, Q, fr, frd);
      f = fl + fr + du;
      fd = fld + frd;
    }
    double pn = p - O::div(f, fd);
    if (!(pn > 0.)) pn = 1.e-30;
    const double change = 2. * fabs(O::div(pn - p, pn + p));
    p = pn;
    if (change <= tol) {
      pstar = p;
      return it;
    }
  }
  pstar = p;
  return -maxit;
}

struct ExactStats {
  unsigned long long iters, fallbacks;
};

// state at x/t = 0 (Toro sec. 4.5); leftside tells which input supplies the
// tangential velocities and gammas.  The right side is sampled as the left one
// of the mirrored problem (velocities negated, which is exact), so that
// wavefronts with faces on either side of the contact run one copy.
// FRESH: what a branch takes from gamma it forms again, from a copy that the
// compiler cannot see through: kept from exact_gas through the iteration, those
// values took the registers that k_face_solve's three waves per SIMD lack (14
// spilled of 168 on tiles of several classes: the exact solver's step on a
// three-level grid of 29.4M zones 27.8 ms instead of 24.7).  k_solve_update, at
// two waves, has them (1024 x 16^3 2561 us a step, 2569 with FRESH).
template <bool FAST, bool FRESH>
__device__ __forceinline__ void exact_sample(const ExactGas& G, const ExactSide& L, double ul,
                                             const ExactSide& Q, double ur, double pm, double um, double& r, double& u,
                                             double& pp, bool& leftside) {
  using O = ExactOps<FAST>;
  const bool left = 0. <= um;
  leftside = left;
  const double rk = left ? L.rho : Q.rho, pk = left ? L.p : Q.p, ck = left ? L.c : Q.c;
  const double v = left ? ul : -ur, w = left ? um : -um;
  const double pmk = O::div(pm, pk);
  double g = G.g;
  if constexpr (FRESH) asm("" : "+v"(g));
  if (left ? pm <= pk : !(pm > pk)) {
    if (0. <= v - ck) {
      r = rk; u = v; pp = pk;
    } else {
      const double cm = ck * pow_pos(pmk, G.e1);
      const double st = w - cm;
      // isentropic: rho = gamma p / c^2 behind the rarefaction
      if (left ? 0. > st : 0. >= st) {
        r = O::div(g * pm, cm * cm); u = w; pp = pm;
      } else {
        const double c = O::div(2., g + 1.) * (ck + (g - 1.) * 0.5 * v);
        u = left ? c : -(-c + 0.);   // a zero is +0 on either side
        // in the fan, (c/ck)^(2g/(g-1)) = (c/ck)^(2/(g-1)) (c/ck)^2
        const double x = O::div(c, ck);
        const double q = pow_pos(x, O::div(2., g - 1.)), s2 = x * x;
        r = rk * q;
        pp = pk * (q * s2);
      }
    }
  } else {
    const double gp1 = g + 1.;
    const double sk = v - ck * O::root(O::div(gp1, 2. * g) * pmk + G.e1);
    if (0. <= sk) {
      r = rk; u = v; pp = pk;
    } else {
      const double rp1 = O::recip(gp1);
      r = O::div(rk * (pmk + O::divr(g - 1., gp1, rp1)), O::divr(pmk * (g - 1.), gp1, rp1) + 1.);
      u = w; pp = pm;
    }
  }
  if (!left) u = -u;
}

// exact_riemann's problem once its states are known to be positive
template <bool FAST, bool SEEDED, bool FRESH>
__device__ __forceinline__ int exact_solve(const DevParams& P, double g, double rl, double ul, double pl, double rr, double ur,
                                           double pr, double guess, ExactStats& es, double& r, double& u, double& pp,
                                           bool& left) {
  using O = ExactOps<FAST>;
  const double cl = O::root(O::div(g * pl, rl)), cr = O::root(O::div(g * pr, rr));
  const ExactGas G = exact_gas<FAST>(g);
  if (G.t1 * (cl + cr) <= ur - ul) return 2;
  const double du = ur - ul;
  const ExactSide L = exact_side<FAST>(G, rl, pl, cl), Q = exact_side<FAST>(G, rr, pr, cr);
  const double ts = two_shock_guess<FAST>(ul, L, ur, Q);
  const double tol = P.exactTol;
  double pm;
  int it, pick;
  if constexpr (!SEEDED) {
    it = exact_newton_pick<FAST>(G, L, Q, du, ts, -1.0, tol, P.exactMaxIter, pm, pick);
    if (it < 0) es.fallbacks += 1;
  } else {
    double pb = guess;
    for (;;) {
      it = exact_newton_pick<FAST>(G, L, Q, du, ts, pb, tol, P.exactMaxIter, pm, pick);
      if (it < 0 && (pb > 0. || guess <= 0.)) es.fallbacks += 1;   // a restart counts once
      if (it >= 0 || pick == 0) break;
      es.iters += (unsigned long long)(-it);
      pb = -1.0;
    }
  }
  es.iters += (unsigned long long)(it < 0 ? -it : it);
  double fl, fld, fr, frd;
  exact_fk<FAST>(pm, G, L, fl, fld);
  exact_fk<FAST>(pm, G, Q, fr, frd);
  const double um = 0.5 * (ul + ur) + 0.5 * (fr - fl);
  exact_sample<FAST, FRESH>(G, L, ul, Q, ur, pm, um, r, u, pp, left);
  return 0;
}

// Exact solution at x/t = 0 of the face problem (rl, ul, pl | rr, ur, pr)
// with the face-normal velocities ul, ur; returns 0 ok, 1 non-positive state,
// 2 vacuum generated.  guess > 0 seeds Newton: it starts from the better of
// the seed and the two-shock guess, and a seeded start that does not
// converge restarts from the two-shock guess (counted as fallback).  One
// Newton loop serves both passes, which keeps a seeded kernel's register
// budget that of the unseeded one.  SEEDED = false ignores guess.
template <bool SEEDED, bool FRESH>
__device__ __forceinline__ int exact_riemann(const DevParams& P, double g, double rl, double ul, double pl, double rr, double ur,
                                             double pr, double guess, ExactStats& es, double& r, double& u,
                                             double& pp, bool& left) {
  if (!(rl > 0. && rr > 0. && pl > 0. && pr > 0.)) return 1;
  if (__builtin_expect(__all(exact_window(g, rl, pl, rr, pr, ur - ul)), 1))
    return exact_solve<true, SEEDED, FRESH>(P, g, rl, ul, pl, rr, ur, pr, guess, es, r, u, pp, left);
  return exact_solve<false, SEEDED, FRESH>(P, g, rl, ul, pl, rr, ur, pr, guess, es, r, u, pp, left);
}

// ---- the FP32 solver (mixed-precision mode): the pressure function, sampling
// and flux run in FP32, while the Newton iterate and its convergence test stay
// in FP64 (the iterate is rounded to FP32 only to evaluate the function).  Its
// expressions stand as they are written, apart from the FP64 ones: which of its
// quotients the compiler rounds correctly and which it forms from a reciprocal
// follows from how it merges the branches below, and the bits with it.

// Tolerance floor of the FP32 solve.  FP32 evaluations of the pressure
// function leave rounding noise of up to a few 1e-7 in p*, where Newton's
// relative change can stall; a change of 1e-5 already puts the next iterate
// (quadratic convergence) below FP32 resolution.
constexpr double kExactTolF32 = 1.e-5;

__device__ __forceinline__ void exact_fk_f32(float p, float rk, float pk, float ck, float g, float& f, float& fd) {
  if (p <= pk) {
    // rarefaction: the derivative's power is the value's divided by pratio,
    // since (g - 1)/(2g) + (g + 1)/(2g) = 1 (one pow instead of two)
    const float pratio = p / pk;
    const float q = pow_pos(pratio, (g - 1.f) / (2.f * g));
    f = 2.f / (g - 1.f) * ck * (q - 1.f);
    fd = (1.f / (rk * ck)) * (q / pratio);
  } else {
    const float ak = 2.f / ((g + 1.f) * rk);
    const float bk = (g - 1.f) / (g + 1.f) * pk;
    const float qrt = sqrt(ak / (bk + p));
    f = (p - pk) * qrt;
    fd = (1.f - 0.5f * (p - pk) / (bk + p)) * qrt;
  }
}

__device__ __forceinline__ float two_shock_guess_f32(float g, float rl, float ul, float pl, float cl, float rr, float ur, float pr, float cr) {
  const float ppv = 0.5f * (pl + pr) - 0.125f * (ur - ul) * (rl + rr) * (cl + cr);
  const float p0 = fmax(1.e-30f, ppv);
  const float gl = sqrt((2.f / ((g + 1.f) * rl)) / ((g - 1.f) / (g + 1.f) * pl + p0));
  const float gr = sqrt((2.f / ((g + 1.f) * rr)) / ((g - 1.f) / (g + 1.f) * pr + p0));
  const float pts = (gl * pl + gr * pr - (ur - ul)) / (gl + gr);
  return fmax(1.e-30f, pts);
}

__device__ __forceinline__ int exact_newton_pick_f32(float g, float rl, float pl, float cl, float rr, float pr, float cr, float du,
                                                 double pa, double pb, double tol, int maxit,
                                                 double& pstar, int& pick) {
  float fl, fld, fr, frd;
  exact_fk_f32(float(pa), rl, pl, cl, g, fl, fld);
  exact_fk_f32(float(pa), rr, pr, cr, g, fr, frd);
  double p = pa;
  float f = fl + fr + du, fd = fld + frd;
  pick = 0;
  if (pb > 0.) {
    float gl, gld, gr, grd;
    exact_fk_f32(float(pb), rl, pl, cl, g, gl, gld);
    exact_fk_f32(float(pb), rr, pr, cr, g, gr, grd);
    const float fb = gl + gr + du;
    if (!(fabs(f) <= fabs(fb))) {
      pick = 1;
      p = pb;
      f = fb;
      fd = gld + grd;
    }
  }
  for (int it = 1; it <= maxit; ++it) {
    if (it > 1) {
      exact_fk_f32(float(p), rl, pl, cl, g, fl, fld);
      exact_fk_f32(float(p), rr, pr, cr, g, fr, frd);
      f = fl + fr + du;
      fd = fld + frd;
    }
    double pn = p - double(f / fd);
    if (!(pn > 0.)) pn = 1.e-30;
    const double change = 2. * fabs((pn - p) / (pn + p));
    p = pn;
    if (change <= tol) {
      pstar = p;
      return it;
    }
  }
  pstar = p;
  return -maxit;
}

__device__ __forceinline__ void exact_sample_f32(float g, float rl, float ul, float pl, float cl, float rr, float ur, float pr, float cr,
                                             float pm, float um, float& r, float& u, float& pp, bool& leftside) {
  if (0.f <= um) {
    leftside = true;
    if (pm <= pl) {
      const float shl = ul - cl;
      if (0.f <= shl) { r = rl; u = ul; pp = pl; return; }
      const float cml = cl * pow_pos(pm / pl, (g - 1.f) / (2.f * g));
      const float stl = um - cml;
      // isentropic: rho = gamma p / c^2 behind the rarefaction
      if (0.f > stl) { r = g * pm / (cml * cml); u = um; pp = pm; return; }
      const float c = 2.f / (g + 1.f) * (cl + (g - 1.f) / 2.f * (ul - 0.f));
      u = 2.f / (g + 1.f) * (cl + (g - 1.f) / 2.f * ul + 0.f);
      // in the fan, (c/cl)^(2g/(g-1)) = (c/cl)^(2/(g-1)) (c/cl)^2
      const float q = pow_pos(c / cl, 2.f / (g - 1.f)), s2 = (c / cl) * (c / cl);
      r = rl * q;
      pp = pl * (q * s2);
      return;
    }
    const float pml = pm / pl;
    const float sl = ul - cl * sqrt((g + 1.f) / (2.f * g) * pml + (g - 1.f) / (2.f * g));
    if (0.f <= sl) { r = rl; u = ul; pp = pl; return; }
    r = rl * (pml + (g - 1.f) / (g + 1.f)) / (pml * (g - 1.f) / (g + 1.f) + 1.f);
    u = um; pp = pm;
    return;
  }
  leftside = false;
  if (pm > pr) {
    const float pmr = pm / pr;
    const float sr = ur + cr * sqrt((g + 1.f) / (2.f * g) * pmr + (g - 1.f) / (2.f * g));
    if (0.f >= sr) { r = rr; u = ur; pp = pr; return; }
    r = rr * (pmr + (g - 1.f) / (g + 1.f)) / (pmr * (g - 1.f) / (g + 1.f) + 1.f);
    u = um; pp = pm;
    return;
  }
  const float shr = ur + cr;
  if (0.f >= shr) { r = rr; u = ur; pp = pr; return; }
  const float cmr = cr * pow_pos(pm / pr, (g - 1.f) / (2.f * g));
  const float str = um + cmr;
  if (0.f <= str) { r = g * pm / (cmr * cmr); u = um; pp = pm; return; }
  const float c = 2.f / (g + 1.f) * (cr - (g - 1.f) / 2.f * (ur - 0.f));
  u = 2.f / (g + 1.f) * (-cr + (g - 1.f) / 2.f * ur + 0.f);
  const float q = pow_pos(c / cr, 2.f / (g - 1.f)), s2 = (c / cr) * (c / cr);
  r = rr * q;
  pp = pr * (q * s2);
}

// As exact_riemann.  Converges to max(exactTol, kExactTolF32), and a seed is held
// at 1e-30 or above, inside FP32's normal range.
template <bool SEEDED>
__device__ __forceinline__ int exact_riemann_f32(const DevParams& P, float g, float rl, float ul, float pl, float rr, float ur,
                                             float pr, double guess, ExactStats& es, float& r, float& u,
                                             float& pp, bool& left) {
  if (!(rl > 0.f && rr > 0.f && pl > 0.f && pr > 0.f)) return 1;
  const float cl = sqrt(g * pl / rl), cr = sqrt(g * pr / rr);
  if (2.f / (g - 1.f) * (cl + cr) <= ur - ul) return 2;
  const float du = ur - ul;
  const float ts = two_shock_guess_f32(g, rl, ul, pl, cl, rr, ur, pr, cr);
  const double tol = fmax(P.exactTol, kExactTolF32);
  double pm;
  int it, pick;
  if constexpr (!SEEDED) {
    it = exact_newton_pick_f32(g, rl, pl, cl, rr, pr, cr, du, double(ts), -1.0, tol, P.exactMaxIter,
                           pm, pick);
    if (it < 0) es.fallbacks += 1;
  } else {
    double pb = guess > 0. ? fmax(guess, 1.e-30) : guess;
    for (;;) {
      it = exact_newton_pick_f32(g, rl, pl, cl, rr, pr, cr, du, double(ts), pb, tol, P.exactMaxIter,
                             pm, pick);
      if (it < 0 && (pb > 0. || guess <= 0.)) es.fallbacks += 1;   // a restart counts once
      if (it >= 0 || pick == 0) break;
      es.iters += (unsigned long long)(-it);
      pb = -1.0;
    }
  }
  es.iters += (unsigned long long)(it < 0 ? -it : it);
  const float pmr = float(pm);
  float fl, fld, fr, frd;
  exact_fk_f32(pmr, rl, pl, cl, g, fl, fld);
  exact_fk_f32(pmr, rr, pr, cr, g, fr, frd);
  const float um = 0.5f * (ul + ur) + 0.5f * (fr - fl);
  exact_sample_f32(g, rl, ul, pl, cl, rr, ur, pr, cr, pmr, um, r, u, pp, left);
  return 0;
}

// prim2flx with the direction chosen at run time (same operations and
// order as prim2flx<DIR>)
template <typename R>
__device__ __forceinline__ void prim2flx_dir(int d, R r, R vx, R vy, R vz, R p, R game, R fP,
                                             R F[6]) {
  const R u2 = vx * vx + vy * vy + vz * vz;
  const R E = R(0.5) * r * u2 + p / (game - R(1.));
  const R un = d == 0 ? vx : (d == 1 ? vy : vz);
  F[5] = p;
  F[0] = r * un;
  F[1] = F[0] * vx;
  F[2] = F[0] * vy;
  F[3] = F[0] * vz;
  const R fp = fP * p;
  if (d == 0) F[1] = F[1] + fp;
  else if (d == 1) F[2] = F[2] + fp;
  else F[3] = F[3] + fp;
  F[4] = (E + p) * un;
}

// Godunov flux F[0..7] across a face normal to direction d from the exact
// solution, with the aux internal-energy fluxes (hy_getFaceFlux.F90:428-442).
// The face states sit in global memory as components 0..5 = dens, velx,
// vely, velz, pres, eint at Lb[q * s] (left) and Rb[q * s] (right); reading
// them with the run-time offset d keeps them out of private arrays, and one
// copy of the solver serves all directions.  gamc is the left cell's, game
// the cells' on either side.  The states and the solve are in R; F is FP64
// for the update.  FRESH as in exact_sample.  Returns exact_riemann's codes.
template <bool SEEDED, typename R, bool FRESH = true>
__device__ __forceinline__ int exact_face_flux(const DevParams& P, int d, const R* Lb,
                                               const R* Rb, long s, double gamc,
                                               double gameL, double gameR, double guess,
                                               double F[8], ExactStats& es) {
  const R rl = Lb[0], pl = Lb[4 * s], rr = Rb[0], pr = Rb[4 * s];
  const R ul = Lb[(1 + d) * s], ur = Rb[(1 + d) * s];
  R r, u, pp;
  bool left;
  int e;
  if constexpr (sizeof(R) == sizeof(double))
    e = exact_riemann<SEEDED, FRESH>(P, gamc, rl, ul, pl, rr, ur, pr, guess, es, r, u, pp, left);
  else
    e = exact_riemann_f32<SEEDED>(P, float(gamc), rl, ul, pl, rr, ur, pr, guess, es, r, u, pp, left);
  if (e) return e;
  // the sampled state takes its tangential velocities and game from the side
  // of the contact the face lies on
  const R* Sb = left ? Lb : Rb;
  R vx = Sb[s], vy = Sb[2 * s], vz = Sb[3 * s];
  if (d == 0) vx = u;
  else if (d == 1) vy = u;
  else vz = u;
  R Fr[6];
  prim2flx_dir(d, r, vx, vy, vz, pp, R(left ? gameL : gameR), R(P.fP), Fr);
#pragma unroll
  for (int q = 0; q < 6; ++q) F[q] = double(Fr[q]);
  F[6] = 0.;
  F[7] = 0.;
  if (P.aux) {
    if (Fr[0] > R(0.)) {
      F[7] = double(Fr[0] / rl);
      F[6] = double(Fr[0] * Lb[5 * s]);
    } else {
      F[7] = double(Fr[0] / rr);
      F[6] = double(Fr[0] * Rb[5 * s]);
    }
  }
  return 0;
}

// Gate of the learned seed: an interface is strong when its largest
// feature magnitude, max(|ln(rl/rr)|, |ln(pl/pr)|, |ur - ul| / c0) / 2 with
// c0^2 = gamma sqrt(pl pr) / sqrt(rl rr), reaches the gate.  The same test
// without logarithms or roots: with T = exp(2 gate) and K = 16 gate^4,
//   rl >= T rr  or  rr >= T rl  or  pl >= T pr  or  pr >= T pl
//   or  (ur - ul)^4 rl rr >= K gamma^2 pl pr.
struct SeedGate {
  double T, K;
};

__host__ __device__ inline SeedGate make_seed_gate(double gate) {
  const double g2 = gate * gate;
  return SeedGate{exp(2.0 * gate), 16.0 * g2 * g2};
}

__device__ __forceinline__ bool seed_gate_pass(const SeedGate& G, double g, double rl, double ul,
                                               double pl, double rr, double ur, double pr) {
  const double du = ur - ul, du2 = du * du;
  return rl >= G.T * rr || rr >= G.T * rl || pl >= G.T * pr || pr >= G.T * pl ||
         du2 * du2 * (rl * rr) >= G.K * (g * g) * (pl * pr);
}

// seed value of a face whose Newton iteration keeps the two-shock start
constexpr float kNoSeed = 3.0e38f;

// ---- gamma-law EOS, MODE_DENS_EI on one cell (Eos_getData.F90:189-215,
// eos_idealGamma.F90:323-333, Eos_putData.F90:197-210) ----
struct EosOut {
  double pres, temp, eint, ener, game;
};
// the internal energy the EOS takes, from the kinetic energy per mass
__device__ __forceinline__ double eos_ie(const DevParams& P, double ekin, double eintIn,
                                         double enerIn) {
  double ie = eintIn;
  if (enerIn - ekin > fmax(P.smallE, P.eintSwitch * ekin)) ie = enerIn - ekin;
  return fmax(ie, P.smallE);
}
// and what follows from it
__device__ __forceinline__ EosOut eos_of_ie(const DevParams& P, double dens, double ekin, double ie) {
  EosOut o;
  o.eint = ie;
  o.pres = dens * ie * P.gam1inv;
  o.temp = ie * P.ggprodinv * P.abar;
  o.ener = ie + ekin;
  o.game = o.pres / (ie * dens) + 1;
  return o;
}
__device__ __forceinline__ EosOut eos_dens_ei(const DevParams& P, double dens, double vx, double vy,
                                              double vz, double eintIn, double enerIn) {
  const double ekin = 0.5 * (vx * vx + vy * vy + vz * vz);
  return eos_of_ie(P, dens, ekin, eos_ie(P, ekin, eintIn, enerIn));
}

}  // namespace fx
