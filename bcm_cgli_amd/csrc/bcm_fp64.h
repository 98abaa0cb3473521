// Device functions the FP64 kernels share: correctly rounded division and square
// root, face reconstruction and the Roe-type flux.  Every function evaluates the
// reference expressions in the reference order (builds with -ffp-contract=off).
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>

#include "bcm_kernels.h"

namespace bcm {
namespace {

constexpr double KG = 1.4;          // K
constexpr double KM1 = 1.4 - 1;     // (K-1), folded exactly as the reference folds it
constexpr double RG = 287.0;        // R
constexpr double CVG = 717.5;       // Cv
constexpr double PRG = 0.72;        // Pr_L
constexpr int WG = 256;

__device__ __forceinline__ size_t sidx(int c, int v, int i, int j, int k) {
  return (size_t)c * CUBE_STRIDE + (size_t)v * PLANE + i * 400 + j * 20 + k;
}
__device__ __forceinline__ int fidx(int c, int i, int j, int k) {
  return c * PLANE + i * 400 + j * 20 + k;
}
// max(a,b) of the reference: (((a)>(b))?(a):(b)), NaN falls to b.
__device__ __forceinline__ double rmax(double a, double b) { return (a > b) ? a : b; }

// Correctly rounded division and square root without the range scaling that
// the compiler's own sequences carry for operands near the ends of the
// exponent range.
//
// A denominator's part (div_by) is its reciprocal r, from the hardware
// estimate r0 (relative error e0 below 2^-22) by one cubic step,
// r0 (1 + e0 + e0^2): what is left, e0^3, lies far below the last bit.  A
// quotient's part (div_sh) is the product a r, its exact remainder, one
// correction and the fixup that sets zeros, infinities, NaN and signs.
// Several quotients share one denominator's part.  The bits are those of a / b
// where the numerator is zero or at least 2^-969 in magnitude (below, its
// remainder is subnormal), the denominator and its reciprocal are normal numbers,
// and the quotient, if not zero, is normal and below 2^1023 (above, the product
// a r may overflow to infinity and the correction give NaN where the quotient is
// finite).  One correction does not suffice where r is not the rounded
// reciprocal, which a step from below cannot reach for a significand of all ones;
// there the hardware's estimate is that value, and the step keeps it.
// k_div_selftest compares at random, at such significands and near these limits.
// No flow reaches them: the smallest momenta are those at the front of a
// disturbance that spreads through a uniform field, above 1e-120 on rows of 24 to
// 120 cubes.  Against the scaled form: one instruction less per quotient (4), two
// less per denominator, no wait between a flag's producer and its consumer (with
// root below, the pushing flux kernel 1,345 -> 1,252 us on 2,048 cubes).
struct DivBy {
  double b, r;   // denominator and its reciprocal
};
__device__ __forceinline__ DivBy div_by(double b) {
  const double r0 = __builtin_amdgcn_rcp(b);
  const double e0 = __builtin_fma(-b, r0, 1.0);
  return DivBy{b, __builtin_fma(r0, __builtin_fma(e0, e0, e0), r0)};
}
__device__ __forceinline__ double div_sh(const DivBy& d, double a) {
  const double q = a * d.r;
  return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-d.b, q, a), d.r, q), d.b, a);
}
__device__ __forceinline__ double dvd(double a, double b) { return div_sh(div_by(b), a); }
// div_by of a value all lanes share, kept in scalar registers.
__device__ __forceinline__ DivBy div_by_uniform(double b) {
  const double r = div_by(b).r;
  return DivBy{b, __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(r)),
                                   __builtin_amdgcn_readfirstlane(__double2loint(r)))};
}
// Square root by Goldschmidt's coupled iteration for sqrt(x) and 1/(2 sqrt(x))
// from the hardware estimate of 1/sqrt(x), then two corrections by the exact
// residual x - s^2 (Markstein, "Software division and square root using
// Goldschmidt's algorithms", 2004).  Correctly rounded for x >= 2^-767; zero
// and +infinity are returned as they are, a negative x gives NaN.
__device__ __forceinline__ double root(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double s = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, s, 0.5);
  s = __builtin_fma(s, r, s);
  h = __builtin_fma(h, r, h);
  s = __builtin_fma(__builtin_fma(-s, s, x), h, s);
  s = __builtin_fma(__builtin_fma(-s, s, x), h, s);
  return __builtin_amdgcn_class(x, 0x260) ? x : s;   // -0, +0, +infinity
}

struct Prim {
  double u, v, w, T;
};

// ---------------------------------------------------------------------------
// Preconditioned Roe-type flux at one face (Flux.cpp:611-797; X :1061-1247,
// Y :1520-1695).  D is the face-normal axis; 3: the lane's own choice of y
// (ydir) or z, for lanes of one wave that evaluate faces of both axes.
template <int D>
__device__ __forceinline__ void roe_flux(const double (&L)[5], const double (&R)[5], double e,
                                         double (&F)[5], double& dP, bool ydir = false) {
  const double lr = L[0];
  const DivBy dl = div_by(lr);
  const double lq0 = div_sh(dl, L[1]), lq1 = div_sh(dl, L[2]), lq2 = div_sh(dl, L[3]);
  const double lVV = lq0 * lq0 + lq1 * lq1 + lq2 * lq2;
  const double lP = (L[4] - 0.5 * lr * lVV) * KM1;
  const double lC = div_sh(dl, KG * lP);
  const DivBy dk = div_by(KM1);
  const double lH = 0.5 * lVV + div_sh(dk, lC);
  const double rr = R[0];
  const DivBy dr = div_by(rr);
  const double rq0 = div_sh(dr, R[1]), rq1 = div_sh(dr, R[2]), rq2 = div_sh(dr, R[3]);
  const double rVV = rq0 * rq0 + rq1 * rq1 + rq2 * rq2;
  const double rP = (R[4] - 0.5 * rr * rVV) * KM1;
  const double rC = div_sh(dr, KG * rP);
  const double rH = 0.5 * rVV + div_sh(dk, rC);

  const double t5 = root(lr), t6 = root(rr), t4 = t5 + t6;
  const double rho = root(lr * rr);
  const DivBy d4 = div_by(t4);
  const double q0 = div_sh(d4, t5 * lq0 + t6 * rq0);
  const double q1 = div_sh(d4, t5 * lq1 + t6 * rq1);
  const double q2 = div_sh(d4, t5 * lq2 + t6 * rq2);
  const double VV = q0 * q0 + q1 * q1 + q2 * q2;
  const double H = div_sh(d4, t5 * lH + t6 * rH);
  const double C = (H - 0.5 * VV) * KM1;
  const DivBy dC = div_by(C);
  const double beta = rmax(div_sh(dC, VV), e);
  const bool ny = D == 3 ? ydir : D == 1, nz = D == 3 ? !ydir : D == 2;
  const double un = D == 0 ? q0 : (ny ? q1 : q2);
  const double lun = D == 0 ? lq0 : (ny ? lq1 : lq2);
  const double run = D == 0 ? rq0 : (ny ? rq1 : rq2);
  const double temp = 0.5 * (1 + beta) * un;
  const double S = 0.5 * root(4 * beta * C + un * un * (1 - beta) * (1 - beta));
  const double temp1 = div_sh(dC, dvd(dvd(rP - lP, rho), beta));
  const DivBy dS = div_by(S);
  const double tS = div_sh(dS, temp);
  const double temp2 = tS * (run - lun);
  const double temp3 = div_sh(dS, 0.5 * (1 - beta) * un * temp);
  const double an = fabs(un);
  const double deltaU = (S - temp3 - beta * an) * temp1 + temp2;
  const double deltaP = tS * (rP - lP) + (S - an + temp3) * rho * (run - lun);

  // Dissipation and the averaged physical flux; Ep = 1 multiplies exactly.
  const double fav0 = an * (R[0] - L[0]) + deltaU * rho;
  double fav1 = an * (R[1] - L[1]) + deltaU * rho * q0;
  double fav2 = an * (R[2] - L[2]) + deltaU * rho * q1;
  double fav3 = an * (R[3] - L[3]) + deltaU * rho * q2;
  if (D == 0) fav1 = fav1 + deltaP;
  if (ny) fav2 = fav2 + deltaP;
  if (nz) fav3 = fav3 + deltaP;
  const double fav4 = an * (R[4] - L[4]) + deltaU * rho * H + deltaP * un;
  F[0] = 0.5 * ((lr * lun + rr * run) - fav0);
  F[1] = D == 0 ? 0.5 * ((lr * lq0 * lq0 + lP + rr * rq0 * rq0 + rP) - fav1)
                : 0.5 * ((lr * lq0 * lun + rr * rq0 * run) - fav1);
  F[2] = ny ? 0.5 * ((lr * lq1 * lq1 + lP + rr * rq1 * rq1 + rP) - fav2)
                : 0.5 * ((lr * lq1 * lun + rr * rq1 * run) - fav2);
  F[3] = nz ? 0.5 * ((lr * lq2 * lq2 + lP + rr * rq2 * rq2 + rP) - fav3)
                : 0.5 * ((lr * lq2 * lun + rr * rq2 * run) - fav3);
  F[4] = 0.5 * ((lun * (3.5 * lP + 0.5 * lr * lVV) + run * (3.5 * rP + 0.5 * rr * rVV)) - fav4);
  dP = 0.5 * (lP + rP);
}

// ---------------------------------------------------------------------------
// Face-based formulation of the same flux (used by k_flux_march).
//
// The states at the face between cells p and p+1 depend only on the
// reconstruction order and on the six cells p-2..p+3: the reference's
// backward-face formulas of cell p+1 and forward-face formulas of cell p are
// the same expressions (Flux.cpp:499-562).  Only the order choice differs
// between the two views, so one evaluation serves both cells whenever their
// orders agree, with bitwise the same result.

// Order of face p+1/2 as cell p sees it (forward face, Flux.cpp:497,533).
__device__ __forceinline__ int order_fwd(int p, int fm1, int fp1, int fp2) {
  if (fp1 == 1 && fm1 == 1) return (p == 17 || fp2 != 1) ? 3 : 5;
  return 1;
}
// Order of face q-1/2 as cell q sees it (backward face, Flux.cpp:497,499).
__device__ __forceinline__ int order_bwd(int q, int fm2, int fm1, int fp1) {
  if (fp1 == 1 && fm1 == 1) return (q == 2 || fm2 != 1) ? 3 : 5;
  return 1;
}

// Face states of order 5, 3 or 1 (Flux.cpp:499-596) of the face between cells
// p and p+1; s(m, v) is variable v of cell p-2+m, read only where the order
// uses it.
template <typename S>
__device__ __forceinline__ void face_states(int order, S s, double (&L)[5], double (&R)[5]) {
  const double c6 = 1. / 6, c60 = 1. / 60;
  if (order == 5) {
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      const double s0 = s(0, v), s1 = s(1, v), s2 = s(2, v), s3 = s(3, v), s4 = s(4, v), s5 = s(5, v);
      L[v] = c60 * (2 * s0 - 13 * s1 + 47 * s2 + 27 * s3 - 3 * s4);
      R[v] = c60 * (-3 * s1 + 27 * s2 + 47 * s3 - 13 * s4 + 2 * s5);
    }
  } else if (order == 3) {
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      const double s1 = s(1, v), s2 = s(2, v), s3 = s(3, v), s4 = s(4, v);
      L[v] = c6 * (-s1 + 5 * s2 + 2 * s3);
      R[v] = c6 * (2 * s2 + 5 * s3 - s4);
    }
  } else {
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      L[v] = s(2, v);
      R[v] = s(3, v);
    }
  }
}

}  // namespace
}  // namespace bcm
