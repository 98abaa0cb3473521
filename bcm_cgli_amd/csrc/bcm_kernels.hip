// CDNA4 (gfx950) kernels of the BCM per-iteration hot path, FP64.
//
// Every kernel evaluates the reference expressions in the reference order and
// the library is built with -ffp-contract=off, so results are bitwise those
// of the reference's FP64 CPU path (checked against the oracle in tests/).
// Citations are file:line in the reference tree; "Flux.cpp" is
// BCM_Flux_XYZ_Viscous_Runge_kutta.cpp.
#include <hip/hip_runtime.h>
#include <math.h>
#include <type_traits>

#include "bcm_fp64.h"
#include "bcm_kernels.h"

namespace bcm {
namespace {

// Full-state access to an inner iterate.  FP64 storage holds the state
// itself; FP32 storage holds its deviation from the case's reference state.
struct NoOff {
  static constexpr bool exact = true;   // the reference's operations, bitwise
  __device__ explicit NoOff(const DevPhys&) {}
  __device__ double ld(const double* U, size_t o, int) const { return U[o]; }
  __device__ void st(double* U, size_t o, int, double x) const { U[o] = x; }
  __device__ double rt(double x, int) const { return x; }
};
struct RefOff {
  static constexpr bool exact = false;  // mixed path: operation order free
  double r[5];
  __device__ explicit RefOff(const DevPhys& ph) { ref_state(ph, r); }
  __device__ double ld(const float* U, size_t o, int v) const { return (double)U[o] + r[v]; }
  __device__ void st(float* U, size_t o, int v, double x) const { U[o] = (float)(x - r[v]); }
  // x as storage would return it.
  __device__ double rt(double x, int v) const { return (double)(float)(x - r[v]) + r[v]; }
};
template <typename T> struct OffOf;
template <> struct OffOf<double> { using type = NoOff; };
template <> struct OffOf<float> { using type = RefOff; };

template <typename T> struct Vec2;
template <> struct Vec2<double> { using type = double2; };
template <> struct Vec2<float> { using type = float2; };

// Inviscid flux difference of one cell along axis D (Flux.cpp:367-806 for Z):
// upwind-biased face states of 5th, 3rd or 1st order depending on the cell
// position and the neighbour flags, then the two face fluxes.
template <int D>
__device__ __forceinline__ void axis_flux(const double* __restrict__ U,
                                          const int8_t* __restrict__ fws, int c, int i, int j,
                                          int k, double e, double (&Rf)[5], double& dPb,
                                          double& dPf) {
  constexpr int st = D == 0 ? 400 : (D == 1 ? 20 : 1);
  const int pos = D == 0 ? i : (D == 1 ? j : k);
  const size_t b = sidx(c, 0, i, j, k);
  const int8_t* fb = fws + fidx(c, i, j, k);
  const int fm2 = fb[-2 * st], fm1 = fb[-st], fp1 = fb[st], fp2 = fb[2 * st];
  double s[7][5];
#pragma unroll
  for (int o = -2; o <= 2; ++o)
#pragma unroll
    for (int v = 0; v < 5; ++v) s[o + 3][v] = U[b + (size_t)v * PLANE + o * st];
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    s[0][v] = pos > 2 ? U[b + (size_t)v * PLANE - 3 * st] : 0.0;
    s[6][v] = pos < 17 ? U[b + (size_t)v * PLANE + 3 * st] : 0.0;
  }
  const double c6 = 1. / 6, c60 = 1. / 60;
  double ML[5], MR[5], MLi[5], MRi[5];
  if (fp1 == 1 && fm1 == 1) {
    if (pos == 2 || fm2 != 1) {
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        ML[v] = c6 * (-s[1][v] + 5 * s[2][v] + 2 * s[3][v]);
        MR[v] = c6 * (2 * s[2][v] + 5 * s[3][v] - s[4][v]);
      }
    } else {
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        ML[v] = c60 * (2 * s[0][v] - 13 * s[1][v] + 47 * s[2][v] + 27 * s[3][v] - 3 * s[4][v]);
        MR[v] = c60 * (-3 * s[1][v] + 27 * s[2][v] + 47 * s[3][v] - 13 * s[4][v] + 2 * s[5][v]);
      }
    }
    if (pos == 17 || fp2 != 1) {
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        MLi[v] = c6 * (-s[2][v] + 5 * s[3][v] + 2 * s[4][v]);
        MRi[v] = c6 * (2 * s[3][v] + 5 * s[4][v] - s[5][v]);
      }
    } else {
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        MLi[v] = c60 * (2 * s[1][v] - 13 * s[2][v] + 47 * s[3][v] + 27 * s[4][v] - 3 * s[5][v]);
        MRi[v] = c60 * (-3 * s[2][v] + 27 * s[3][v] + 47 * s[4][v] - 13 * s[5][v] + 2 * s[6][v]);
      }
    }
  } else {
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      ML[v] = s[2][v];
      MR[v] = s[3][v];
      MLi[v] = s[3][v];
      MRi[v] = s[4][v];
    }
  }
  double Fb[5], Ff[5];
  roe_flux<D>(ML, MR, e, Fb, dPb);
  roe_flux<D>(MLi, MRi, e, Ff, dPf);
#pragma unroll
  for (int v = 0; v < 5; ++v) Rf[v] = Ff[v] - Fb[v];
}


// Neighbour primitives as the viscous block computes them (T = P/(rho*R)).
__device__ __forceinline__ Prim nb_prim(const double* __restrict__ U, size_t b) {
  const double r = U[b];
  Prim p;
  p.u = U[b + PLANE] / r;
  p.v = U[b + 2 * PLANE] / r;
  p.w = U[b + 3 * PLANE] / r;
  const double P = (U[b + 4 * PLANE] - 0.5 * r * (p.u * p.u + p.v * p.v + p.w * p.w)) * KM1;
  p.T = P / (r * RG);
  return p;
}

// Slot of a neighbour offset (a,b,c) in {-1,0,1}^3 in a 27-entry table.
__device__ __forceinline__ constexpr int nslot(int a, int b, int c) {
  return (a + 1) * 9 + (b + 1) * 3 + (c + 1);
}

// Viscous flux through the face of axis D on side SIDE (-1 backward,
// +1 forward), Flux.cpp:1946-2272.
template <int D, int SIDE>
__device__ __forceinline__ void visc_face(const Prim (&q)[27], const Prim& me, double T0,
                                          double mu_L, double inv, double (&L)[5]) {
  constexpr int o0 = D == 0 ? SIDE : 0, o1 = D == 1 ? SIDE : 0, o2 = D == 2 ? SIDE : 0;
  const Prim f = q[nslot(o0, o1, o2)];
  const double Tf = 0.5 * (me.T + f.T);
  const double temp = dvd(Tf, T0);
  const double mu = dvd(mu_L * temp * root(temp) * (T0 + 110.), Tf + 110.);
  double g[3][4];
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    if (t == D) {
      if (SIDE < 0) {
        g[t][0] = (me.u - f.u) * inv;
        g[t][1] = (me.v - f.v) * inv;
        g[t][2] = (me.w - f.w) * inv;
        g[t][3] = (me.T - f.T) * inv;
      } else {
        g[t][0] = (f.u - me.u) * inv;
        g[t][1] = (f.v - me.v) * inv;
        g[t][2] = (f.w - me.w) * inv;
        g[t][3] = (f.T - me.T) * inv;
      }
    } else {
      const int p0 = t == 0 ? 1 : 0, p1 = t == 1 ? 1 : 0, p2 = t == 2 ? 1 : 0;
      const Prim& A = q[nslot(p0, p1, p2)];
      const Prim& B = q[nslot(p0 + o0, p1 + o1, p2 + o2)];
      const Prim& Cm = q[nslot(-p0, -p1, -p2)];
      const Prim& Dm = q[nslot(-p0 + o0, -p1 + o1, -p2 + o2)];
      g[t][0] = (A.u + B.u - Cm.u - Dm.u) / 4 * inv;
      g[t][1] = (A.v + B.v - Cm.v - Dm.v) / 4 * inv;
      g[t][2] = (A.w + B.w - Cm.w - Dm.w) / 4 * inv;
      g[t][3] = (A.T + B.T - Cm.T - Dm.T) / 4 * inv;
    }
  }
  const double uf = 0.5 * (me.u + f.u), vf = 0.5 * (me.v + f.v), wf = 0.5 * (me.w + f.w);
  const double div = g[0][0] + g[1][1] + g[2][2];
  double sg[3];
#pragma unroll
  for (int m = 0; m < 3; ++m)
    sg[m] = (m == D) ? mu * (2 * g[D][D] - 2.0 / 3.0 * div) : mu * (g[m][D] + g[D][m]);
  L[1] = sg[0];
  L[2] = sg[1];
  L[3] = sg[2];
  L[4] = uf * sg[0] + vf * sg[1] + wf * sg[2] + mu * CVG * KG * g[D][3] / (PRG);
}

// ---------------------------------------------------------------------------
// Flux, residual and preconditioned stage increment of one interior cell
// (Flux.cpp:331-2398).  Grid: (16 i-planes, cubes), 256 lanes = 16 j x 16 k.
__global__ __launch_bounds__(WG) void k_flux(const double* __restrict__ U,
                                             const double* __restrict__ U1,
                                             const double* __restrict__ U1q,
                                             const int8_t* __restrict__ fws,
                                             const double* __restrict__ cube_size,
                                             double* __restrict__ Rku, double* __restrict__ Res,
                                             PhysTab pt, double deltaT, double deltaTau,
                                             double e) {
  const int c = blockIdx.y + 1;
  const int cc = pt.cube_case[c];
  if (cc < 0) return;
  const DevPhys ph = pt.phys[cc];
  const int i = blockIdx.x + 2;
  const int j = (threadIdx.x >> 4) + 2;
  const int k = (threadIdx.x & 15) + 2;
  const double dx = cube_size[c] / 16;
  const double dy = dx, dz = dx;
  const double inv = 1. / dx;
  const size_t b = sidx(c, 0, i, j, k);
  const int IF = fws[fidx(c, i, j, k)];

  double u[5];
#pragma unroll
  for (int v = 0; v < 5; ++v) u[v] = U[b + (size_t)v * PLANE];

  // Inviscid part.
  double Rx[5], Ry[5], Rz[5], dPxb, dPxf, dPyb, dPyf, dPzb, dPzf;
  axis_flux<2>(U, fws, c, i, j, k, e, Rz, dPzb, dPzf);
  axis_flux<0>(U, fws, c, i, j, k, e, Rx, dPxb, dPxf);
  axis_flux<1>(U, fws, c, i, j, k, e, Ry, dPyb, dPyf);
  double Rf[5];
#pragma unroll
  for (int v = 0; v < 5; ++v) Rf[v] = -(Rx[v] / dx + Ry[v] / dy + Rz[v] / dz);

  // Viscous part: primitives of the 6 face and 12 edge neighbours.
  Prim q[27];
#pragma unroll
  for (int a = -1; a <= 1; ++a)
#pragma unroll
    for (int bb = -1; bb <= 1; ++bb)
#pragma unroll
      for (int cc = -1; cc <= 1; ++cc) {
        const int nz = (a != 0) + (bb != 0) + (cc != 0);
        if (nz == 1 || nz == 2) q[nslot(a, bb, cc)] = nb_prim(U, b + a * 400 + bb * 20 + cc);
      }
  Prim me;
  const double rho = u[0];
  me.u = u[1] / u[0];
  me.v = u[2] / u[0];
  me.w = u[3] / u[0];
  {
    const double VV = me.u * me.u + me.v * me.v + me.w * me.w;
    const double P = (u[4] - 0.5 * rho * VV) * KM1;
    me.T = P / rho / RG;
  }
  double Lxb[5], Lxf[5], Lyb[5], Lyf[5], Lzb[5], Lzf[5];
  visc_face<0, -1>(q, me, ph.T0, ph.mu_L, inv, Lxb);
  visc_face<0, +1>(q, me, ph.T0, ph.mu_L, inv, Lxf);
  visc_face<1, -1>(q, me, ph.T0, ph.mu_L, inv, Lyb);
  visc_face<1, +1>(q, me, ph.T0, ph.mu_L, inv, Lyf);
  visc_face<2, -1>(q, me, ph.T0, ph.mu_L, inv, Lzb);
  visc_face<2, +1>(q, me, ph.T0, ph.mu_L, inv, Lzf);
  double vF[5];
#pragma unroll
  for (int v = 1; v < 5; ++v)
    vF[v] = (Lxf[v] - Lxb[v]) * inv + (Lyf[v] - Lyb[v]) * inv + (Lzf[v] - Lzb[v]) * inv;

  // Residual with the dual-time source.
  double Rk[5];
  const DivBy d2t = div_by(2 * deltaT);
  {
    const double uu0 = U1[b], uq0 = U1q[b];
    Rk[0] = div_sh(d2t, -(3 * u[0] - 4 * uu0 + uq0)) + Rf[0];
  }
#pragma unroll
  for (int v = 1; v < 5; ++v) {
    const double uu = U1[b + (size_t)v * PLANE], uq = U1q[b + (size_t)v * PLANE];
    const double Rp = div_sh(d2t, -(3 * u[v] - 4 * uu + uq));
    Rk[v] = Rp + Rf[v] + vF[v];
  }

  // Closed-form preconditioner D = M (Gamma + 3 dtau/(2 dT) M)^-1 (Flux.cpp:2295-2343).
  const double U_ = u[1] / u[0], V_ = u[2] / u[0], W_ = u[3] / u[0];
  const double VV = U_ * U_ + V_ * V_ + W_ * W_;
  const double P = (u[4] - 0.5 * rho * VV) * KM1;
  const double C = KG * P / rho;
  const double T = P / rho;
  const double H = 0.5 * VV + C / KM1;
  const double beta = rmax(VV / C, e);
  const double temp = KG * T * (2 * deltaT + 3 * deltaTau) * (2 * deltaT + 3 * beta * deltaTau);
  const double temp2 = KM1 * (beta - 1) * deltaT * deltaT;
  const double temp3 = H - H * KG - VV + KG * (T + VV);
  double out[5];
  if (IF == 1) {
    const DivBy dT = div_by(temp);
    const double d11 = div_sh(dT, (2 * deltaT * (-2 * (-KM1 * (H - VV) - temp3 * beta) * deltaT + 3 * KG * T * beta * deltaTau)));
    const double d12 = div_sh(dT, (-4 * U_ * temp2));
    const double d13 = div_sh(dT, (-4 * V_ * temp2));
    const double d14 = div_sh(dT, (-4 * W_ * temp2));
    const double d15 = div_sh(dT, (4 * temp2));
    out[0] = deltaTau * (d11 * Rk[0] + d12 * Rk[1] + d13 * Rk[2] + d14 * Rk[3] + d15 * Rk[4]);
    const double d21 = div_sh(dT, (4 * U_ * temp3 * (beta - 1) * deltaT * deltaT));
    const double d22 = div_sh(dT, (2 * deltaT * (2 * KG * (T - U_ * U_ * (beta - 1)) * deltaT + 2 * U_ * U_ * (beta - 1) * deltaT + 3 * KG * T * beta * deltaTau)));
    const double d23 = div_sh(dT, (-4 * U_ * V_ * temp2));
    const double d24 = div_sh(dT, (-4 * U_ * W_ * temp2));
    const double d25 = div_sh(dT, (4 * U_ * temp2));
    out[1] = deltaTau * (d21 * Rk[0] + d22 * Rk[1] + d23 * Rk[2] + d24 * Rk[3] + d25 * Rk[4]);
    const double d31 = div_sh(dT, (4 * V_ * temp3 * (beta - 1) * deltaT * deltaT));
    const double d33 = div_sh(dT, (2 * deltaT * (2 * KG * (T - V_ * V_ * (beta - 1)) * deltaT + 2 * V_ * V_ * (beta - 1) * deltaT + 3 * KG * T * beta * deltaTau)));
    const double d34 = div_sh(dT, (-4 * V_ * W_ * temp2));
    const double d35 = div_sh(dT, (4 * V_ * temp2));
    out[2] = deltaTau * (d31 * Rk[0] + d23 * Rk[1] + d33 * Rk[2] + d34 * Rk[3] + d35 * Rk[4]);
    const double d41 = div_sh(dT, (4 * W_ * temp3 * (beta - 1) * deltaT * deltaT));
    const double d44 = div_sh(dT, (2 * deltaT * (2 * KG * (T - W_ * W_ * (beta - 1)) * deltaT + 2 * W_ * W_ * (beta - 1) * deltaT + 3 * KG * T * beta * deltaTau)));
    const double d45 = div_sh(dT, (4 * W_ * temp2));
    out[3] = deltaTau * (d41 * Rk[0] + d24 * Rk[1] + d34 * Rk[2] + d44 * Rk[3] + d45 * Rk[4]);
    const double d51 = div_sh(dT, (4 * H * temp3 * (beta - 1) * deltaT * deltaT));
    const double d52 = div_sh(dT, (-4 * H * U_ * temp2));
    const double d53 = div_sh(dT, (-4 * H * V_ * temp2));
    const double d54 = div_sh(dT, (-4 * H * W_ * temp2));
    const double d55 = div_sh(dT, (2 * deltaT * (2 * H * KM1 * (beta - 1) * deltaT + KG * T * (2 * deltaT + 3 * beta * deltaTau))));
    out[4] = deltaTau * (d51 * Rk[0] + d52 * Rk[1] + d53 * Rk[2] + d54 * Rk[3] + d55 * Rk[4]);
  } else {
#pragma unroll
    for (int v = 0; v < 5; ++v) out[v] = 0;
  }
#pragma unroll
  for (int v = 0; v < 5; ++v) Rku[b + (size_t)v * PLANE] = out[v];
  if (IF < 1) {
    Res[b] = -(-(dPxf - dPxb) / dx + vF[1]) * dx * dy * dz;
    Res[b + PLANE] = -(-(dPzf - dPzb) / dz + vF[3]) * dx * dy * dz;
  }
}

// RK stage update of fluid cells (Flux.cpp:2417-2599).  At RK3 each block
// also writes its partial sums of the five change norms (:2530-2566) and of
// the two force-density components (:2603-2625; body_only: of the cells a flux
// kernel just wrote, whatever the others hold).
__global__ __launch_bounds__(WG) void k_update(int RK, double* __restrict__ U,
                                               double* __restrict__ U1p1,
                                               double* __restrict__ U1p2,
                                               const double* __restrict__ Rku,
                                               const double* __restrict__ Res,
                                               const int8_t* __restrict__ fws,
                                               const int* __restrict__ cube_case,
                                               double* __restrict__ partials, int body_only) {
  const int c = blockIdx.y + 1;
  if (cube_case[c] < 0) return;
  const int i = blockIdx.x + 2;
  const int j = (threadIdx.x >> 4) + 2;
  const int k = (threadIdx.x & 15) + 2;
  const size_t b = sidx(c, 0, i, j, k);
  const bool fluid = fws[fidx(c, i, j, k)] == 1;
  if (RK == 1) {
    if (fluid)
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        const double x = U[b + (size_t)v * PLANE] + Rku[b + (size_t)v * PLANE];
        U[b + (size_t)v * PLANE] = x;
        U1p1[b + (size_t)v * PLANE] = x;
      }
    return;
  }
  if (RK == 2) {
    if (fluid)
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        const size_t o = b + (size_t)v * PLANE;
        const double x = 0.75 * U[o] + 0.25 * U1p1[o] + 0.25 * Rku[o];
        U[o] = x;
        U1p2[o] = x;
      }
    return;
  }
  double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (fluid) {
    double u[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) u[v] = U[b + (size_t)v * PLANE];
    const double ro = u[0];
    const double uo = u[1] / ro, vo = u[2] / ro, wo = u[3] / ro;
    const double VVo = uo * uo + vo * vo + wo * wo;
    const double Po = (u[4] - 0.5 * ro * VVo) * KM1;
    const double To = Po / ro;
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      const size_t o = b + (size_t)v * PLANE;
      u[v] = 1.0 / 3.0 * u[v] + 2.0 / 3.0 * U1p2[o] + 2.0 / 3.0 * Rku[o];
      U[o] = u[v];
    }
    const double r = u[0];
    const double un = u[1] / r, vn = u[2] / r, wn = u[3] / r;
    const double VV = un * un + vn * vn + wn * wn;
    const double P = (u[4] - 0.5 * r * VV) * KM1;
    const double T = P / r;
    acc[0] = (P - Po) * (P - Po);
    acc[1] = (un - uo) * (un - uo);
    acc[2] = (vn - vo) * (vn - vo);
    acc[3] = (wn - wo) * (wn - wo);
    acc[4] = (T - To) * (T - To);
  }
  if (!body_only || fws[fidx(c, i, j, k)] < 1) {
    acc[5] = Res[b];
    acc[6] = Res[b + PLANE];
  }
  // The row the marching flux kernels write for this plane, bitwise.
  __shared__ double red[WG / 64][8];
  const int t = threadIdx.x;
  const double s = wave_sum8(acc);
  if ((t & 7) == 0) red[t >> 6][(t >> 3) & 7] = s;
  __syncthreads();
  if (t < 8) {
    double r = red[0][t];
#pragma unroll
    for (int w = 1; w < WG / 64; ++w) r += red[w][t];
    partials[((size_t)blockIdx.y * gridDim.x + blockIdx.x) * 8 + t] = r;
  }
}

// Final norm reduction (Flux.cpp:2627-2652 at one rank): er[1..7] of one case
// per block from its cubes' rows of 8 partial sums, stride rows apart: 16 rows
// per cube (one per plane), already summed into the first for the pool's first
// `single` cubes.  Eight lanes read a row; a cube's rows are summed in order,
// then the cubes in an order fixed relative to the case's first cube, so a case
// gives the same bits alone and next to other cases, in any number of runs.
//
// Bound: one CU's loads for one large case (2,048 cubes: 14 us, 21 when every
// cube had 16 rows, folded by a kernel of its own), latencies for a small one (8
// cubes: 4.6 us, 9 in two kernels).
constexpr int REDUCE_WG = 1024;
__global__ __launch_bounds__(REDUCE_WG) void k_reduce(const double* __restrict__ partials,
                                                      int stride, int single,
                                                      const CaseDesc* __restrict__ cases,
                                                      const DevPhys* __restrict__ phys,
                                                      double* __restrict__ er_all) {
  __shared__ double sh[REDUCE_WG / 64][8];
  const CaseDesc cd = cases[blockIdx.x];
  const DevPhys ph = phys[cd.slot];
  const int t = threadIdx.x;
  const double* rows = partials + (size_t)(cd.first - 1) * stride * 8 + (t & 7);
  double acc = 0;
  for (int q = t / 8; q < cd.n; q += REDUCE_WG / 8) {
    const double* r = rows + (size_t)q * stride * 8;
    double s = r[0];
    if (cd.first + q > single) {
      double x[15];
#pragma unroll
      for (int b = 0; b < 15; ++b) x[b] = r[(b + 1) * 8];
#pragma unroll
      for (int b = 0; b < 15; ++b) s += x[b];
    }
    acc += s;
  }
#pragma unroll
  for (int off = 32; off >= 8; off >>= 1) acc += __shfl_down(acc, off, 64);
  if ((t & 63) < 8) sh[t >> 6][t & 7] = acc;
  __syncthreads();
  if (t < 7) {
    double s = sh[0][t];
#pragma unroll
    for (int w = 1; w < REDUCE_WG / 64; ++w) s += sh[w][t];
    double* er = er_all + (size_t)cd.slot * 8;
    const double DN = 1. / (cd.mpi_ncube * 16 * 16 * 16);
    if (t == 0) er[0] = 0;
    er[t + 1] = t < 5 ? sqrt(s) * DN : s / (0.5 * ph.rho0 * ph.U0 * ph.U0 * 2.602);
  }
}

// ---------------------------------------------------------------------------
// ---------------------------------------------------------------------------
// Edge passes and domain boundary conditions of one cube by the calling
// workgroup (OPEN_WG lanes): edge-ghost averaging (Interface.cpp:5640-5732)
// where asked for, then X (BCM_X_boundary_condition.cpp:43-118), Y
// (BCM_Y_boundary_condition.cpp:36-80) and Z (BCM_Z_boundary_condition.cpp:42-92).
// m bits: 1 x-min, 2 x-max, 4 y-min, 8 y-max, 16 z-min, 32 z-max.
//
// Pass by pass each of the six would read what the one before wrote: a chain
// of up to six memory round trips for a few kilobytes.  Every cell written
// has a closed form in the state before the first pass (a copy of a copy is a
// copy of the first source, an edge mean's sources are face ghost cells or
// such means), so all cells are loaded, one barrier passes, and all are
// stored; a cell that a later pass overwrites is not stored by the earlier
// one.  1024 lanes leave at most one cell of each pass to a lane.  A cube with
// three BC faces 6 us, pass by pass 9.5; the opening of 2,048 cubes (872 with
// BCs) in FP64 28 us, with 256 lanes pass by pass 43.
// Of the edge passes only the listed cells are formed: those the z-BC copies
// (four of the plane k = 2 or 17 of such a face; listed wherever there is one)
// and those the IB fill reads.  The passes belong to the exchange after the last
// update, so where they read face ghost cells that the BCs write they read the
// previous stage's: from `before`, the copy of the iterate that holds them (U
// itself where no pushing flux kernel ran since).
constexpr int OPEN_WG = 1024;
template <typename T>
__device__ __forceinline__ void edge_bc_cube(T* U, const T* before, int c, const int16_t* edges,
                                             int nedge, int m, const DevPhys& ph) {
  using T2 = typename Vec2<T>::type;
  const typename OffOf<T>::type F(ph);
  const int t = threadIdx.x;
  T* const Uc = U + (size_t)c * CUBE_STRIDE;
  const T* const Bc = before + (size_t)c * CUBE_STRIDE;
  auto at = [](int v, int i, int j, int k) { return v * PLANE + i * 400 + j * 20 + k; };
  // Nearest interior index of 1 (2) or 18 (17).
  auto near = [](int q) { return q == 1 ? 2 : 17; };
  bool de = t < 5 * nedge;
  const int ecell = de ? edges[t / 5] : 0, ev = t % 5;
  // Face ghost cell as the last exchange's edge passes read it.
  auto face = [&](int v, int i, int j, int k) {
    const bool bc = (i == 1 && (m & 1)) || (i == 18 && (m & 2)) || (j == 1 && (m & 4)) ||
                    (j == 18 && (m & 8)) || (k == 1 && (m & 16)) || (k == 18 && (m & 32));
    return (bc ? Bc : Uc)[at(v, i, j, k)];
  };
  // x-min inflow state from the interior state next to it, as stored.
  auto inflow = [&](const T (&q)[5], T (&o)[5]) {
    const double rho = F.ld(q, 0, 0);
    const double uu = F.ld(q, 1, 1) / rho;
    const double vv = F.ld(q, 2, 2) / rho;
    const double ww = F.ld(q, 3, 3) / rho;
    double VV = uu * uu + vv * vv + ww * ww;
    const double P = (F.ld(q, 4, 4) - 0.5 * rho * VV) * KM1;
    VV = ph.Uin * ph.Uin + ph.V0 * ph.V0 + ph.W0 * ph.W0;
    const double E = P / KM1 + 0.5 * rho * VV;
    o[0] = q[0];
    F.st(o, 1, 1, rho * ph.Uin);
    F.st(o, 2, 2, rho * ph.V0);
    F.st(o, 3, 3, rho * ph.W0);
    F.st(o, 4, 4, E);
  };
  // Source row i of a BC copy along x, and whether it passes the inflow.
  auto x_source = [&](int i, bool& in) {
    in = i < 2 && (m & 1);
    return in ? 2 : (i > 17 && (m & 2) ? 17 : i);
  };

  // X: (j, k) of side t / 256 (the other half of the lanes has none).
  const int xs = t >> 8, xj = ((t >> 4) & 15) + 2, xk = (t & 15) + 2;
  const bool dx = xs < 2 && (m & (1 << xs));
  T x[5];
  if (dx)
#pragma unroll
    for (int v = 0; v < 5; ++v) x[v] = Uc[at(v, xs ? 17 : 2, xj, xk)];

  // Y: (i, k), i = 0..19, of side t / 512.
  const int side = t >> 9, w = t & 511;
  const int yi = w >> 4, yk = (w & 15) + 2;
  const bool dy = w < 320 && (m & (4 << side));
  bool yin = false;
  T y[5];
  if (dy) {
    const int i = x_source(yi, yin);
#pragma unroll
    for (int v = 0; v < 5; ++v) y[v] = Uc[at(v, i, side ? 17 : 2, yk)];
  }

  // Z: (i, j) of side t / 512.  Interior planes of a face marked ZBC_IN_FLUX
  // get their z-BC from the flux kernel.
  const int zi = w / 20, zj = w % 20, zk = side ? 17 : 2;
  bool dz = w < 400 && (m & (16 << side)) &&
            !(zi >= 2 && zi <= 17 && (m & (ZBC_IN_FLUX << side)));
  bool zin = false;
  T z[5];
  if (dz) {
    // Where the Y-BC wrote the source plane its own source, where that (or
    // the cell itself) is in a row of the X-BC the source of that.  A k-edge
    // cell is copied by the lane that forms it.
    const int j = zj < 2 && (m & 4) ? 2 : (zj > 17 && (m & 8) ? 17 : zj);
    int i = zi;
    if (j >= 2 && j <= 17) i = x_source(zi, zin);
    dz = !(nedge > 0 && (i == 1 || i == 18) && (j == 1 || j == 18));
    if (dz)
#pragma unroll
      for (int v = 0; v < 5; ++v) z[v] = Uc[at(v, i, j, zk)];
  }

  // Edges: a listed cell's variable t % 5 by lane t (at most 200 cells), the
  // mean of two face ghost cells, or at a cube corner of the j-edge and the
  // i-edge cell next to it.
  bool corner = false;
  int zcopy = 0;   // 1 (2): z-min (z-max) copies the cell
  T ea, eb, ec;
  if (de) {
    const int i = ecell / 400, j = ecell / 20 % 20, k = ecell % 20;
    const bool gi = i == 1 || i == 18, gj = j == 1 || j == 18, gk = k == 1 || k == 18;
    corner = gi && gj && gk;
    if (corner) {
      // j-edge (i, near j, k) from ea and ec, i-edge (near i, j, k) from eb
      // and ec.
      ea = face(ev, i, near(j), near(k));
      eb = face(ev, near(i), j, near(k));
      ec = face(ev, near(i), near(j), k);
    } else {
      // (For each pair of ghost layers the cell one step in from either.)
      ea = gk ? face(ev, i, j, near(k)) : face(ev, i, near(j), k);
      eb = gi ? face(ev, near(i), j, k) : face(ev, i, near(j), k);
    }
    // Cells the BCs overwrite.
    const bool zinner = i >= 2 && i <= 17;
    if (!gk) {
      de = !((j == 1 && (m & 4)) || (j == 18 && (m & 8)));
      zcopy = k == 2 && (m & 16) ? 1 : (k == 17 && (m & 32) ? 2 : 0);
    } else {
      de = !((k == 1 && (m & 16) && !(zinner && (m & ZBC_IN_FLUX))) ||
             (k == 18 && (m & 32) && !(zinner && (m & (ZBC_IN_FLUX << 1)))));
    }
  }
  __syncthreads();   // all loads have returned

  if (de) {
    if (corner) {
      ea = 0.5 * (ea + ec);
      eb = 0.5 * (eb + ec);
    }
    const T x = 0.5 * (ea + eb);
    const int dst = ev * PLANE + ecell;
    Uc[dst] = x;
    if (zcopy) {
      // dst is the k = 2 (17) cell; its z ghost cells are k = 0, 1 (18, 19).
      T o = x;
      if (zcopy == 1 && ev == 3) F.st(&o, 0, 3, -F.ld(&o, 0, 3));
      T2 q;
      q.x = q.y = o;
      *reinterpret_cast<T2*>(Uc + dst + (zcopy == 1 ? -2 : 1)) = q;
    }
  }
  if (dx) {
    T o[5];
    if (xs)
#pragma unroll
      for (int v = 0; v < 5; ++v) o[v] = x[v];
    else
      inflow(x, o);
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      Uc[at(v, xs ? 18 : 0, xj, xk)] = o[v];
      Uc[at(v, xs ? 19 : 1, xj, xk)] = o[v];
    }
  }
  if (dy) {
    T o[5];
    if (yin)
      inflow(y, o);
    else
#pragma unroll
      for (int v = 0; v < 5; ++v) o[v] = y[v];
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      Uc[at(v, yi, side ? 18 : 0, yk)] = o[v];
      Uc[at(v, yi, side ? 19 : 1, yk)] = o[v];
    }
  }
  if (dz) {
    T o[5];
    if (zin)
      inflow(z, o);
    else
#pragma unroll
      for (int v = 0; v < 5; ++v) o[v] = z[v];
    if (!side) F.st(o, 3, 3, -F.ld(o, 3, 3));
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      // Both ghost cells at once: rows are a multiple of two values long.
      T2 q;
      q.x = q.y = o[v];
      *reinterpret_cast<T2*>(Uc + at(v, zi, zj, side ? 18 : 0)) = q;
    }
  }
}

template <typename T>
__global__ __launch_bounds__(OPEN_WG) void k_bc(T* __restrict__ U, const int* __restrict__ cubes,
                                                const uint8_t* __restrict__ masks, PhysTab pt) {
  const int c = cubes[blockIdx.x];
  edge_bc_cube<T>(U, U, c, nullptr, 0, masks[blockIdx.x], pt.phys[pt.cube_case[c]]);
}

// Ghost regions the BCs wrote, from the copy of the iterate that a pushing flux
// kernel read to the one it wrote, which no BC pass has seen: one boundary cube
// per workgroup, once per step.  (When each flux kernel copied them in its last
// lines, a stage's took 24.6 us instead of 19.1 on 8 cubes in FP64 and 529 instead
// of 493 on 2,048 mixed.)
template <typename T>
__global__ __launch_bounds__(OPEN_WG) void k_carry_bc(const T* __restrict__ Uin,
                                                      T* __restrict__ Uout,
                                                      const int* __restrict__ cubes,
                                                      const uint8_t* __restrict__ cube_mask,
                                                      PhysTab pt) {
  const int c = cubes[blockIdx.x];
  const DevPhys ph = pt.phys[pt.cube_case[c]];
  copy_bc_regions(Uin, Uout, c, cube_mask[c], ph.rho0 * ph.W0);
}

// ---------------------------------------------------------------------------
// Immersed-boundary ghost fill (BCM_Ghostcell_minus.cpp:72-489).  The
// reference walks the minus list then the plus list in order, writing in
// place; entries here come grouped per cube into dependency levels built on
// the host (an entry's level is above every earlier entry it reads from or
// whose corners it overwrites), so all entries of one level run in parallel
// and levels are separated by workgroup barriers.  Interpolation corners
// always lie in the ghost cell's own padded cube.
//
// The fill is a chain of latencies (one entry's arithmetic per level, table
// and state loads before it), so all that can be is taken out of the chain.
// A corner's density, velocity and pressure depend on its cell alone: they
// are formed once per staged cell, at the load, and once per entry for the
// levels above, and a level only reads and combines them, eight lanes to an
// entry.  A cube's tables start from one record; the next level's entries and
// the bounds of the one after load during a level, whose barrier leaves memory
// operations in flight; ghost cells go back to memory once, at the end.  A
// level takes 0.85 us with few entries and 1.9 with 126 (2.2 us when each entry
// formed its corners' primitives in one lane and every level waited for its
// table loads), the opening of a stage with a sphere inside one cube (7 levels)
// 11.5 us of 20, of a body on 7 cubes with one of 2040 slots 12.5 of 75 (then on
// memory, beyond 1536 slots).
// A value is rounded to storage precision before a later level reads it, as
// memory would round it, so the fill on memory (cubes of more slots than
// GHOST_LDS_SLOTS) gives the same results.

// What the fill in LDS reads of an entry: the weights, the corners' slots (two
// to a word), and its own slot with the corner that is the ghost cell.
struct GhostEntryR {
  double w[8];
  int lc[4], lg_self;
  __device__ int slot(int m) const { return (m & 1 ? lc[m / 2] >> 16 : lc[m / 2] & 0xffff); }
};
__device__ __forceinline__ GhostEntryR load_entry(const GhostEntry* p) {
  GhostEntryR r;
  const int* q = reinterpret_cast<const int*>(p->lc);
#pragma unroll
  for (int m = 0; m < 8; ++m) r.w[m] = p->w[m];
#pragma unroll
  for (int m = 0; m < 4; ++m) r.lc[m] = q[m];
  r.lg_self = q[4];
  return r;
}

// Density, velocity and pressure of a conserved state.
template <typename OFF>
__device__ __forceinline__ void corner_prim(const double (&q)[5], double (&p)[5]) {
  const double r = q[0];
  p[0] = r;
  if constexpr (OFF::exact) {
    p[1] = q[1] / r;
    p[2] = q[2] / r;
    p[3] = q[3] / r;
  } else {
    // One reciprocal per corner instead of three divisions.
    const double ir = 1.0 / r;
    p[1] = q[1] * ir;
    p[2] = q[2] * ir;
    p[3] = q[3] * ir;
  }
  const double VV = p[1] * p[1] + p[2] * p[2] + p[3] * p[3];
  p[4] = (q[4] - 0.5 * r * VV) * KM1;
}

// Conserved state of a ghost cell, by eight lanes that all return it: lane
// r < 5 of them interpolates quantity r (density, velocity, pressure) from the
// corners' values x with the weights w, in the order of a GhostEntry; self: the
// last corner is the ghost cell.
__device__ __forceinline__ void ghost_state(const double (&w)[8], const double (&x)[8], bool self,
                                            double rho0, double P0, double (&o)[5]) {
  const int r = threadIdx.x & 7;
  const bool scalar = r == 0 || r >= 4;
  const double off = r == 0 ? rho0 : (r >= 4 ? P0 : 0.0);
  // (Subtracting an offset of zero changes no value.)
  double s = w[0] * (x[0] - off);
#pragma unroll
  for (int m = 1; m < 7; ++m) s = s + w[m] * (x[m] - off);
  double z;
  if (self) {
    // The ghost cell is an interpolation corner (:192-449).
    const double qt = s / ((scalar ? 1 : 2) - w[7]);
    z = scalar ? (w[7] > 0.9999 ? x[7] : qt + off) : qt;
  } else {
    s = s + w[7] * (x[7] - off);
    z = scalar ? s + off : s;
  }
  const int l0 = threadIdx.x & 56;
  const double rho = __shfl(z, l0), uu = __shfl(z, l0 + 1), vv = __shfl(z, l0 + 2),
               ww = __shfl(z, l0 + 3), P = __shfl(z, l0 + 4);
  const double VV = uu * uu + vv * vv + ww * ww;
  o[0] = rho;
  if (self) {
    o[1] = rho * uu;
    o[2] = rho * vv;
    o[3] = rho * ww;
    o[4] = P / KM1 + 0.5 * rho * VV;
  } else {
    o[1] = 0.5 * rho * uu;
    o[2] = 0.5 * rho * vv;
    o[3] = 0.5 * rho * ww;
    o[4] = P / KM1 + 0.5 * rho * 0.25 * VV;
  }
}
// The r-th of five values, by selection (values, as a reference to an array
// would become an index into memory).
__device__ __forceinline__ double pick(double a0, double a1, double a2, double a3, double a4,
                                       int r) {
  const double x = r == 1 ? a1 : a0, y = r == 3 ? a3 : a2;
  return r > 3 ? a4 : (r > 1 ? y : x);
}

// Eight lanes share an entry.  Entry of a lane in a level of n entries
// starting at e (a lane without one loads the level's first, which it does
// not use).
constexpr int GHOST_PASS = OPEN_WG / 8;
__device__ __forceinline__ int entry_of(int e, int n) {
  const int q = threadIdx.x / 8;
  return e + (q < n ? q : 0);
}

// What a lane can load of a cube's fill before the state it reads is final:
// its first staged cell (the last one where it has none), its entry of the
// first level, and the ghost cell it stores (-1: none).
struct GhostFirst {
  int cell, out;
  GhostEntryR E;
};
__device__ __forceinline__ void ghost_first(const GhostTables& gt, const GhostCube& g,
                                            GhostFirst& f) {
  if (g.nread < 0) return;
  const int t = threadIdx.x;
  f.cell = gt.read[g.read0 + (t < g.nread ? t : g.nread - 1)];
  f.out = gt.out[g.ent0 + (t < g.ne ? t : 0)];
  f.E = load_entry(gt.ent + entry_of(g.ent0, g.n1));
}

// Barrier for values exchanged through LDS: unlike __syncthreads it leaves
// loads and stores of memory in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// IB fill of one cube in LDS by the calling workgroup.  prim holds the
// primitives of slot n in prim[v * cap + n]; the conserved values of entry a
// follow in cons[v * ne + a].
template <typename T>
__device__ __forceinline__ void ghost_lds(T* __restrict__ U, const GhostTables& gt,
                                          const GhostCube& g, const GhostFirst& f,
                                          const DevPhys& ph, double* gsm) {
  using OFF = typename OffOf<T>::type;
  const OFF F(ph);
  const int t = threadIdx.x;
  const size_t base = (size_t)g.cube * CUBE_STRIDE;
  const int cap = g.ne + g.nread;
  double* prim = gsm;
  double* cons = gsm + 5 * cap;
  for (int n = t; n < g.nread; n += OPEN_WG) {
    const int cell = n < OPEN_WG ? f.cell : gt.read[g.read0 + n];
    double a[5], p[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) a[v] = F.ld(U, base + (size_t)v * PLANE + cell, v);
    corner_prim<OFF>(a, p);
#pragma unroll
    for (int v = 0; v < 5; ++v) prim[v * cap + g.ne + n] = p[v];
  }
  lds_barrier();
  // The value of an entry goes to LDS conserved for the store to memory and
  // as primitives for the levels above.
  const int r = t & 7, rv = r < 5 ? r : 4;
  auto fill_entry = [&](const GhostEntryR& E) {
    double x[8], o[5], p[5];
#pragma unroll
    for (int m = 0; m < 8; ++m) x[m] = prim[rv * cap + E.slot(m)];
    ghost_state(E.w, x, (E.lg_self >> 16) < 8, ph.rho0, ph.P0, o);
#pragma unroll
    for (int v = 0; v < 5; ++v) o[v] = F.rt(o[v], v);
    corner_prim<OFF>(o, p);
    const int lg = E.lg_self & 0xffff;
    if (r < 5) {
      cons[r * g.ne + lg] = pick(o[0], o[1], o[2], o[3], o[4], r);
      prim[r * cap + lg] = pick(p[0], p[1], p[2], p[3], p[4], r);
    }
  };
  // Levels run one after the other, each taking one entry's latency.  The
  // lane's entry of the next level is loaded while the current one is
  // computed, the bounds of the level after that as well.
  const int end = g.lev0 + g.nlev;
  GhostEntryR Enext = f.E;
  int e0 = g.ent0, e1 = g.ent0 + g.n1;
  int e2 = gt.level_off[min(g.lev0 + 2, end)];
  for (int lv = g.lev0; lv < end; ++lv) {
    const GhostEntryR E = Enext;
    const int e3 = gt.level_off[min(lv + 3, end)];
    if (e1 < e2) Enext = load_entry(gt.ent + entry_of(e1, e2 - e1));
    if (e0 + t / 8 < e1) fill_entry(E);
    for (int n = e0 + t / 8 + GHOST_PASS; n < e1; n += GHOST_PASS) fill_entry(load_entry(gt.ent + n));
    lds_barrier();
    e0 = e1;
    e1 = e2;
    e2 = e3;
  }
  // The last value of each ghost cell goes back to memory.
  for (int a = t; a < g.ne; a += OPEN_WG) {
    const int cell = a < OPEN_WG ? f.out : gt.out[g.ent0 + a];
    if (cell < 0) continue;
#pragma unroll
    for (int v = 0; v < 5; ++v) F.st(U, base + (size_t)v * PLANE + cell, v, cons[v * g.ne + a]);
  }
}

// IB fill of one cube in place on memory: an entry's eight lanes form a corner's
// primitives each.
template <typename T>
__device__ __forceinline__ void ghost_memory(T* __restrict__ U, const GhostTables& gt,
                                             const GhostCube& g, const DevPhys& ph) {
  using OFF = typename OffOf<T>::type;
  const OFF F(ph);
  const size_t base = (size_t)g.cube * CUBE_STRIDE;
  const int r = threadIdx.x & 7, l0 = threadIdx.x & 56;
  for (int lv = g.lev0; lv < g.lev0 + g.nlev; ++lv) {
    const int e1 = gt.level_off[lv + 1];
    for (int n = gt.level_off[lv] + threadIdx.x / 8; n < e1; n += GHOST_PASS) {
      const GhostEntry& E = gt.ent[n];
      // Corner of the entry's r-th weight.
      const int m = E.self > 7 ? r : r == 7 ? E.self : r + (r >= E.self);
      const int a = (m == 1 || m == 4 || m == 5 || m == 7);
      const int bq = (m == 2 || m == 4 || m == 6 || m == 7);
      const int cq = (m == 3 || m == 5 || m == 6 || m == 7);
      const size_t at = base + (E.pi + a) * 400 + (E.pj + bq) * 20 + (E.pk + cq);
      double q[5], p[5], w[8], x[8], o[5];
#pragma unroll
      for (int v = 0; v < 5; ++v) q[v] = F.ld(U, at + (size_t)v * PLANE, v);
      corner_prim<OFF>(q, p);
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        w[m] = E.w[m];
#pragma unroll
        for (int v = 0; v < 5; ++v) {
          const double y = __shfl(p[v], l0 + m);
          x[m] = v == 0 || r == v ? y : (v == 4 && r > 4 ? y : x[m]);
        }
      }
      ghost_state(w, x, E.self < 8, ph.rho0, ph.P0, o);
      // Every corner has been read: the eight lanes are in one wave, and no
      // other entry of the level reads or writes the cell.
      const size_t go = base + E.gi * 400 + E.gj * 20 + E.gk;
      if (r == 0)
#pragma unroll
        for (int v = 0; v < 5; ++v) F.st(U, go + (size_t)v * PLANE, v, o[v]);
    }
    __syncthreads();
  }
}

template <typename T>
__device__ __forceinline__ void ghost_cube(T* __restrict__ U, const GhostTables& gt,
                                           const GhostCube& g, GhostFirst& f, const DevPhys& ph,
                                           double* gsm) {
  if (g.nread >= 0)
    ghost_lds(U, gt, g, f, ph, gsm);
  else
    ghost_memory(U, gt, g, ph);
}

template <typename T>
__global__ __launch_bounds__(OPEN_WG) void k_ghost(T* __restrict__ U, GhostTables gt, PhysTab pt) {
  extern __shared__ double gsm[];
  const GhostCube g = gt.cubes[blockIdx.x];
  GhostFirst f;
  ghost_first(gt, g, f);
  ghost_cube(U, gt, g, f, pt.phys[pt.cube_case[g.cube]], gsm);
}

// Edge-ghost averaging of one cube in the reference's three sequential passes
// (Interface.cpp:5640-5732): i-edges, then j-edges, then k-edges.  Called by a
// whole workgroup; the face ghosts it reads must be complete.  A pass reads
// face ghost cells and writes edge cells only, so each lane loads both of its
// items (w = t and t + 256) before storing either.
template <typename T>
__device__ __forceinline__ void edge_fill(T* __restrict__ U, int c) {
  const int t = threadIdx.x;
  // Pass a (0: i-edges at (j,k) in {1,18}^2, i = 2..17; 1: j-edges at (i,k),
  // j = 1..18; 2: k-edges at (i,j), k = 1..18).  Item w: edge e = w & 3,
  // variable v = (w >> 2) % 5, position along the edge (w >> 2) / 5.
  auto pass = [&](auto axis) {
    constexpr int A = decltype(axis)::value;
    constexpr int n = (A == 0 ? 16 : 18) * 4 * 5, p0 = A == 0 ? 2 : 1;
    T xa[2], xb[2];
    size_t dst[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int w = t + h * WG;
      if (w >= n) continue;
      const int q = (w >> 2) / 5 + p0, e = w & 3, v = (w >> 2) % 5;
      size_t a, b;
      if (A == 0) {
        if (e == 0) a = sidx(c, v, q, 1, 2), b = sidx(c, v, q, 2, 1);
        else if (e == 1) a = sidx(c, v, q, 18, 2), b = sidx(c, v, q, 17, 1);
        else if (e == 2) a = sidx(c, v, q, 1, 17), b = sidx(c, v, q, 2, 18);
        else a = sidx(c, v, q, 18, 17), b = sidx(c, v, q, 17, 18);
        dst[h] = sidx(c, v, q, (e == 1 || e == 3) ? 18 : 1, (e >= 2) ? 18 : 1);
      } else if (A == 1) {
        if (e == 0) a = sidx(c, v, 1, q, 2), b = sidx(c, v, 2, q, 1);
        else if (e == 1) a = sidx(c, v, 2, q, 18), b = sidx(c, v, 1, q, 17);
        else if (e == 2) a = sidx(c, v, 17, q, 1), b = sidx(c, v, 18, q, 2);
        else a = sidx(c, v, 17, q, 18), b = sidx(c, v, 18, q, 17);
        dst[h] = sidx(c, v, (e >= 2) ? 18 : 1, q, (e == 1 || e == 3) ? 18 : 1);
      } else {
        if (e == 0) a = sidx(c, v, 1, 2, q), b = sidx(c, v, 2, 1, q);
        else if (e == 1) a = sidx(c, v, 2, 18, q), b = sidx(c, v, 1, 17, q);
        else if (e == 2) a = sidx(c, v, 17, 1, q), b = sidx(c, v, 18, 2, q);
        else a = sidx(c, v, 17, 18, q), b = sidx(c, v, 18, 17, q);
        dst[h] = sidx(c, v, (e >= 2) ? 18 : 1, (e == 1 || e == 3) ? 18 : 1, q);
      }
      xa[h] = U[a];
      xb[h] = U[b];
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
      if (t + h * WG < n) U[dst[h]] = 0.5 * (xa[h] + xb[h]);
  };
  pass(std::integral_constant<int, 0>());
  __syncthreads();
  pass(std::integral_constant<int, 1>());
  __syncthreads();
  pass(std::integral_constant<int, 2>());
}

// ---------------------------------------------------------------------------
// Cube-to-cube halo of equal-size neighbours as a gather into each cube's own
// face layers (Interface.cpp:1745-1782, 2604-2641, 3474-3511), then the
// cube's edge-ghost averaging in the reference's three sequential passes
// (:5640-5732).  Sources are interior layers, which nothing in this kernel
// writes, so cubes proceed independently.
template <typename T>
__global__ __launch_bounds__(WG) void k_halo_edge(T* __restrict__ U,
                                                  const HaloSrc* __restrict__ srcs,
                                                  const int* __restrict__ cube_case) {
  using T2 = typename Vec2<T>::type;
  const int c = blockIdx.x + 1;
  if (cube_case[c] < 0) return;
  const HaloSrc hs = srcs[c];
  const int t = threadIdx.x;
  const int p = (t >> 4) + 2, r = (t & 15) + 2;
  // All loads first, then all stores: one memory round trip per lane.  The
  // two layers of a z-face are adjacent in k and move as one 2-element vector
  // (rows start 16-byte aligned for FP64 and 8-byte aligned for FP32).
  // Faces without a neighbour read their own cube (discarded) so that every
  // load is unconditional.
  const int sx0 = hs.src[0], sx1 = hs.src[1], sy0 = hs.src[2], sy1 = hs.src[3];
  const int sz0 = hs.src[4], sz1 = hs.src[5];
  const int ax0 = sx0 > 0 ? sx0 : c, ax1 = sx1 > 0 ? sx1 : c, ay0 = sy0 > 0 ? sy0 : c,
            ay1 = sy1 > 0 ? sy1 : c, az0 = sz0 > 0 ? sz0 : c, az1 = sz1 > 0 ? sz1 : c;
  T x0[2][5], x1[2][5], y0[2][5], y1[2][5], z0[2][5], z1[2][5];
#pragma unroll
  for (int l = 0; l < 2; ++l)
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      x0[l][v] = U[sidx(ax0, v, 16 + l, p, r)];
      x1[l][v] = U[sidx(ax1, v, 2 + l, p, r)];
      y0[l][v] = U[sidx(ay0, v, p, 16 + l, r)];
      y1[l][v] = U[sidx(ay1, v, p, 2 + l, r)];
    }
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    const T2 a = *reinterpret_cast<const T2*>(U + sidx(az0, v, p, r, 16));
    const T2 b = *reinterpret_cast<const T2*>(U + sidx(az1, v, p, r, 2));
    z0[0][v] = a.x;
    z0[1][v] = a.y;
    z1[0][v] = b.x;
    z1[1][v] = b.y;
  }
#pragma unroll
  for (int l = 0; l < 2; ++l)
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      if (sx0 > 0) U[sidx(c, v, l, p, r)] = x0[l][v];
      if (sx1 > 0) U[sidx(c, v, 18 + l, p, r)] = x1[l][v];
      if (sy0 > 0) U[sidx(c, v, p, l, r)] = y0[l][v];
      if (sy1 > 0) U[sidx(c, v, p, 18 + l, r)] = y1[l][v];
    }
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    T2 a, b;
    a.x = z0[0][v];
    a.y = z0[1][v];
    b.x = z1[0][v];
    b.y = z1[1][v];
    if (sz0 > 0) *reinterpret_cast<T2*>(U + sidx(c, v, p, r, 0)) = a;
    if (sz1 > 0) *reinterpret_cast<T2*>(U + sidx(c, v, p, r, 18)) = b;
  }
  __syncthreads();
  edge_fill(U, c);
}

// Pre-flux halo refresh.  Between the post-update exchange and the next
// stage's pre-flux exchange the only interior cells that change are the IB
// ghost cells written by the ghost fill, and the domain BCs only write ghost
// layers that no gather writes.  The full gather therefore reduces to copying
// those ghost cells that lie in a neighbour's source layers, followed by the
// edge passes, which read face ghosts the BCs may have changed.
template <typename T>
__global__ __launch_bounds__(WG) void k_halo_sparse(T* __restrict__ U,
                                                    const int2* __restrict__ pairs, int n) {
  const int g = blockIdx.x * WG + threadIdx.x;
  if (g >= n) return;
  const int2 pr = pairs[g];  // (source flat cell, destination flat cell), cube*8000 + cell
  const size_t so = (size_t)(pr.x / PLANE) * CUBE_STRIDE + pr.x % PLANE;
  const size_t dd = (size_t)(pr.y / PLANE) * CUBE_STRIDE + pr.y % PLANE;
#pragma unroll
  for (int v = 0; v < 5; ++v) U[dd + (size_t)v * PLANE] = U[so + (size_t)v * PLANE];
}

template <typename T>
__global__ __launch_bounds__(WG) void k_edge(T* __restrict__ U,
                                             const int* __restrict__ cube_case) {
  if (cube_case[blockIdx.x + 1] < 0) return;
  edge_fill(U, blockIdx.x + 1);
}

// Edge passes of the listed cubes only.
template <typename T>
__global__ __launch_bounds__(WG) void k_edge_list(T* __restrict__ U, const int* __restrict__ list) {
  edge_fill(U, list[blockIdx.x]);
}

// Opening of a stage after a flux kernel that wrote its face halos into the
// neighbours (flux_push), in one launch: per item, a cube's edge passes of the
// post-update exchange and the domain BCs of the next stage, then its IB fill.
// Both touch only the cube's own cells, so cubes proceed independently, each in
// the reference's order.  Every item gets the LDS of the pool's largest fill: a
// fill of 2,040 slots (80 KB, so one workgroup per CU) next to the 872 boundary
// cubes of 2,048 leaves the launch at 26 us.
template <typename T>
__global__ __launch_bounds__(OPEN_WG) void k_open(T* U, const T* before,
                                                  const OpenItem* __restrict__ items,
                                                  const int16_t* __restrict__ edges,
                                                  GhostTables gt,
                                                  const DevPhys* __restrict__ phys) {
  extern __shared__ double gsm[];
  const OpenItem it = items[blockIdx.x];
  const DevPhys ph = phys[it.slot];
  const bool shell = it.mask || it.nedge;
  if (shell) edge_bc_cube(U, before, it.g.cube, edges + it.edge0, it.nedge, it.mask, ph);
  if (it.g.nlev == 0) return;
  // The fill's tables load while the stores above complete.
  GhostFirst f;
  ghost_first(gt, it.g, f);
  if (shell) __syncthreads();
  ghost_cube(U, gt, it.g, f, ph, gsm);
}

// Two-level faces (BCM_Interface.cpp:1790-2600 for x, :2651-3470 for y,
// :3518-4360 for z): one task per workgroup.  Injection copies storage values
// (the FP32 iterate holds deviations from one reference state per case, and
// both cubes of a face belong to the same case); restriction sums the 8 full
// states in the reference's order, (0,0,0) (1,0,0) (0,1,0) (0,0,1) (1,1,0)
// (1,0,1) (0,1,1) (1,1,1) of (i,j,k) offsets, and scales by 0.125.
template <typename T>
__global__ __launch_bounds__(WG) void k_halo_ml(T* __restrict__ U,
                                                const MlTaskDev* __restrict__ tasks,
                                                PhysTab pt) {
  const MlTaskDev t = tasks[blockIdx.x];
  const int A = t.axis, T0 = A == 0 ? 1 : 0, T1 = A == 2 ? 1 : 2;
  const int o0 = (t.slot == 2 || t.slot == 4) ? 8 : 0;
  const int o1 = (t.slot == 3 || t.slot == 4) ? 8 : 0;
  int d[3], q[3];
  if (!t.restrict_) {
    for (int n = threadIdx.x; n < 2 * 256; n += WG) {
      const int l = n >> 8, p = ((n >> 4) & 15) + 2, r = (n & 15) + 2;
      d[A] = t.hi ? 18 + l : l;
      d[T0] = p;
      d[T1] = r;
      q[A] = t.hi ? 2 : 17;
      q[T0] = p / 2 + 1 + o0;
      q[T1] = r / 2 + 1 + o1;
      const size_t dd = sidx(t.dst, 0, d[0], d[1], d[2]);
      const size_t so = sidx(t.src, 0, q[0], q[1], q[2]);
#pragma unroll
      for (int v = 0; v < 5; ++v) U[dd + (size_t)v * PLANE] = U[so + (size_t)v * PLANE];
    }
    return;
  }
  const typename OffOf<T>::type F(pt.phys[pt.cube_case[t.dst]]);
  for (int n = threadIdx.x; n < 2 * 64; n += WG) {
    const int l = n >> 6, p = ((n >> 3) & 7) + 2, r = (n & 7) + 2;
    d[A] = t.hi ? 18 + l : l;
    d[T0] = p + o0;
    d[T1] = r + o1;
    q[A] = t.hi ? 2 * (l + 1) : 14 + 2 * l;
    q[T0] = (p - 1) * 2;
    q[T1] = (r - 1) * 2;
    const size_t dd = sidx(t.dst, 0, d[0], d[1], d[2]);
    const size_t b = sidx(t.src, 0, q[0], q[1], q[2]);
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      const size_t o = b + (size_t)v * PLANE;
      double s = F.ld(U, o, v);
      s = s + F.ld(U, o + 400, v);
      s = s + F.ld(U, o + 20, v);
      s = s + F.ld(U, o + 1, v);
      s = s + F.ld(U, o + 420, v);
      s = s + F.ld(U, o + 401, v);
      s = s + F.ld(U, o + 21, v);
      s = s + F.ld(U, o + 421, v);
      F.st(U, dd + (size_t)v * PLANE, v, 0.125 * s);
    }
  }
}

// Physical-time shift of interior cells (main.cpp:1292-1315).
__global__ __launch_bounds__(WG) void k_shift(const double* __restrict__ U,
                                              double* __restrict__ U1,
                                              double* __restrict__ U1q,
                                              const int* __restrict__ cube_case) {
  const int c = blockIdx.y + 1;
  if (cube_case[c] < 0) return;
  const int i = blockIdx.x + 2;
  const int j = (threadIdx.x >> 4) + 2;
  const int k = (threadIdx.x & 15) + 2;
  const size_t b = sidx(c, 0, i, j, k);
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    const size_t o = b + (size_t)v * PLANE;
    U1q[o] = U1[o];
    U1[o] = U[o];
  }
}

__global__ __launch_bounds__(WG) void k_aos_to_soa(const double* __restrict__ aos,
                                                   double* __restrict__ soa, int ncells) {
  const int g = blockIdx.x * WG + threadIdx.x;
  if (g >= ncells) return;
  const int c = g / PLANE, cell = g % PLANE;
#pragma unroll
  for (int v = 0; v < 5; ++v) soa[(size_t)c * CUBE_STRIDE + (size_t)v * PLANE + cell] = aos[(size_t)g * 5 + v];
}

__global__ __launch_bounds__(WG) void k_soa_to_aos(const double* __restrict__ soa,
                                                   double* __restrict__ aos, int ncells) {
  const int g = blockIdx.x * WG + threadIdx.x;
  if (g >= ncells) return;
  const int c = g / PLANE, cell = g % PLANE;
#pragma unroll
  for (int v = 0; v < 5; ++v) aos[(size_t)g * 5 + v] = soa[(size_t)c * CUBE_STRIDE + (size_t)v * PLANE + cell];
}

}  // namespace

// ---------------------------------------------------------------------------
int update_blocks(int ncube) { return 16 * (ncube - 1); }

template <typename T>
void launch_bc_t(hipStream_t s, T* U, const int* cubes, const uint8_t* masks, int n, PhysTab pt) {
  if (n > 0) hipLaunchKernelGGL(k_bc<T>, dim3(n), dim3(OPEN_WG), 0, s, U, cubes, masks, pt);
}
void launch_bc(hipStream_t s, double* U, const int* cubes, const uint8_t* masks, int n,
               PhysTab pt) {
  launch_bc_t(s, U, cubes, masks, n, pt);
}
void launch_bc(hipStream_t s, float* U, const int* cubes, const uint8_t* masks, int n,
               PhysTab pt) {
  launch_bc_t(s, U, cubes, masks, n, pt);
}

template <typename T>
void launch_ghost_t(hipStream_t s, T* U, const GhostTables& g, PhysTab pt) {
  if (g.ncubes <= 0) return;
  const size_t shmem = (size_t)g.max_slots * 5 * sizeof(double);
  hipLaunchKernelGGL(k_ghost<T>, dim3(g.ncubes), dim3(OPEN_WG), shmem, s, U, g, pt);
}
void launch_ghost(hipStream_t s, double* U, const GhostTables& g, PhysTab pt) {
  launch_ghost_t(s, U, g, pt);
}
void launch_ghost(hipStream_t s, float* U, const GhostTables& g, PhysTab pt) {
  launch_ghost_t(s, U, g, pt);
}

template <typename T>
void launch_open_t(hipStream_t s, T* U, const T* before, const OpenItem* items, int n,
                   const int16_t* edges, const GhostTables& g, const DevPhys* phys) {
  if (n <= 0) return;
  const size_t shmem = (size_t)g.max_slots * 5 * sizeof(double);
  hipLaunchKernelGGL(k_open<T>, dim3(n), dim3(OPEN_WG), shmem, s, U, before, items,
                     edges, g, phys);
}
void launch_open(hipStream_t s, double* U, const double* before, const OpenItem* items, int n,
                 const int16_t* edges, const GhostTables& g, const DevPhys* phys) {
  launch_open_t(s, U, before, items, n, edges, g, phys);
}
void launch_open(hipStream_t s, float* U, const float* before, const OpenItem* items, int n,
                 const int16_t* edges, const GhostTables& g, const DevPhys* phys) {
  launch_open_t(s, U, before, items, n, edges, g, phys);
}

template <typename T>
void launch_carry_bc_t(hipStream_t s, const T* Uin, T* Uout, const int* cubes, int n,
                       const uint8_t* cube_mask, PhysTab pt) {
  if (n > 0)
    hipLaunchKernelGGL(k_carry_bc<T>, dim3(n), dim3(OPEN_WG), 0, s, Uin, Uout, cubes, cube_mask,
                       pt);
}
void launch_carry_bc(hipStream_t s, const double* Uin, double* Uout, const int* cubes, int n,
                     const uint8_t* cube_mask, PhysTab pt) {
  launch_carry_bc_t(s, Uin, Uout, cubes, n, cube_mask, pt);
}
void launch_carry_bc(hipStream_t s, const float* Uin, float* Uout, const int* cubes, int n,
                     const uint8_t* cube_mask, PhysTab pt) {
  launch_carry_bc_t(s, Uin, Uout, cubes, n, cube_mask, pt);
}

template <typename T>
void launch_edge_t(hipStream_t s, T* U, int ncube, const int* cube_case) {
  if (ncube > 1) hipLaunchKernelGGL(k_edge<T>, dim3(ncube - 1), dim3(WG), 0, s, U, cube_case);
}
template <typename T>
void launch_halo_ml_t(hipStream_t s, T* U, const MlTaskDev* tasks, int ntask, PhysTab pt) {
  if (ntask > 0) hipLaunchKernelGGL(k_halo_ml<T>, dim3(ntask), dim3(WG), 0, s, U, tasks, pt);
}
void launch_halo_ml(hipStream_t s, double* U, const MlTaskDev* tasks, int ntask, PhysTab pt) {
  launch_halo_ml_t(s, U, tasks, ntask, pt);
}
void launch_halo_ml(hipStream_t s, float* U, const MlTaskDev* tasks, int ntask, PhysTab pt) {
  launch_halo_ml_t(s, U, tasks, ntask, pt);
}
void launch_edge(hipStream_t s, double* U, int ncube, const int* cube_case) {
  launch_edge_t(s, U, ncube, cube_case);
}
void launch_edge(hipStream_t s, float* U, int ncube, const int* cube_case) {
  launch_edge_t(s, U, ncube, cube_case);
}

template <typename T>
void launch_halo_edge_t(hipStream_t s, T* U, const HaloSrc* src, int ncube, const int* cube_case) {
  if (ncube > 1)
    hipLaunchKernelGGL(k_halo_edge<T>, dim3(ncube - 1), dim3(WG), 0, s, U, src, cube_case);
}
void launch_halo_edge(hipStream_t s, double* U, const HaloSrc* src, int ncube,
                      const int* cube_case) {
  launch_halo_edge_t(s, U, src, ncube, cube_case);
}
void launch_halo_edge(hipStream_t s, float* U, const HaloSrc* src, int ncube,
                      const int* cube_case) {
  launch_halo_edge_t(s, U, src, ncube, cube_case);
}

template <typename T>
void launch_halo_pairs_t(hipStream_t s, T* U, const int2* pairs, int npairs) {
  if (npairs > 0)
    hipLaunchKernelGGL(k_halo_sparse<T>, dim3((npairs + WG - 1) / WG), dim3(WG), 0, s, U, pairs,
                       npairs);
}
void launch_halo_pairs(hipStream_t s, double* U, const int2* pairs, int npairs) {
  launch_halo_pairs_t(s, U, pairs, npairs);
}
void launch_halo_pairs(hipStream_t s, float* U, const int2* pairs, int npairs) {
  launch_halo_pairs_t(s, U, pairs, npairs);
}

template <typename T>
void launch_edge_list_t(hipStream_t s, T* U, const int* list, int n) {
  if (n > 0) hipLaunchKernelGGL(k_edge_list<T>, dim3(n), dim3(WG), 0, s, U, list);
}
void launch_edge_list(hipStream_t s, double* U, const int* list, int n) {
  launch_edge_list_t(s, U, list, n);
}
void launch_edge_list(hipStream_t s, float* U, const int* list, int n) {
  launch_edge_list_t(s, U, list, n);
}

void launch_flux(hipStream_t s, const double* U, const double* U1, const double* U1q,
                 const int8_t* fws, const double* cube_size, double* Rku, double* Res,
                 int ncube, PhysTab pt, double deltaT, double deltaTau, double e) {
  if (ncube > 1)
    hipLaunchKernelGGL(k_flux, dim3(16, ncube - 1), dim3(WG), 0, s, U, U1, U1q, fws, cube_size,
                       Rku, Res, pt, deltaT, deltaTau, e);
}

__global__ __launch_bounds__(WG) void k_copy_d(const double* __restrict__ src,
                                               double* __restrict__ dst, size_t n) {
  for (size_t g = (size_t)blockIdx.x * WG + threadIdx.x; g < n; g += (size_t)gridDim.x * WG)
    dst[g] = src[g];
}

namespace {
// DivBy/div_sh against a / b and root against sqrt: per thread one denominator
// and four numerators from a seeded hash, with random signs; about one numerator
// in 16 is a signed zero.  Of four threads one each takes
//   0: random significands, exponents in [-126, 126];
//   1: significands next to 1, 1.5 and 2 (all ones), the same exponents;
//   2: numerators next to the smallest division is right for, 2^-969 to 2^-965,
//      over denominators in 2^-24 to 2^24, half of either with significands as in
//      1, and roots of 2^-767 to 2^-763;
//   3: numerators and denominators of exponents in [-480, 480].
__device__ __forceinline__ unsigned long long mix64(unsigned long long x) {
  x += 0x9e3779b97f4a7c15ull;
  x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
  x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
  return x ^ (x >> 31);
}
// A value with exponent in [lo, lo + n) from the bits of r; ends: its significand
// at most 3 units off 1, 1.5 or 2.
__device__ __forceinline__ double test_value(unsigned long long r, int lo, int n, bool ends) {
  long long m = (long long)(r >> 12);
  if (ends) {
    const int at = (int)(m % 3), by = (int)(m / 3 % 4);
    m = at == 0 ? by : at == 1 ? (1ll << 51) - 2 + by : (1ll << 52) - 1 - by;
  }
  const double v = ldexp(1.0 + (double)m * 0x1p-52, lo + (int)((r >> 1) % n));
  return (r & 1) ? -v : v;
}
__global__ __launch_bounds__(WG) void k_div_selftest(unsigned long long seed, int n,
                                                     unsigned long long* __restrict__ bad) {
  const int g = blockIdx.x * WG + threadIdx.x;
  if (g >= n) return;
  const unsigned long long base = mix64(seed ^ ((unsigned long long)g << 20));
  const int kind = g & 3;
  auto ends = [&](unsigned long long r) { return kind == 1 || (kind == 2 && (r >> 32 & 1)); };
  auto den = [&](unsigned long long r) {
    return kind < 2 ? test_value(r, -126, 253, ends(r))
                    : kind == 2 ? test_value(r, -24, 49, ends(r)) : test_value(r, -480, 961, false);
  };
  auto num = [&](unsigned long long r) {
    return kind == 2 ? test_value(r, -969, 5, ends(r)) : den(r);
  };
  const double b = den(mix64(base));
  double a[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    a[k] = num(mix64(base + 1 + k));
    if ((mix64(base + 10 + k) & 15) == 0) a[k] = (k & 1) ? -0.0 : 0.0;
  }
  const DivBy d = div_by(b);
  unsigned long long nb = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    nb += __double_as_longlong(div_sh(d, a[k])) != __double_as_longlong(a[k] / b);
  const unsigned long long q = mix64(base + 5);
  const double x = fabs(kind == 2 ? test_value(q, -767, 5, ends(q)) : a[0]);
  nb += __double_as_longlong(root(x)) != __double_as_longlong(sqrt(x));
  if (nb) atomicAdd(bad, nb);
}
}  // namespace

int div_selftest(unsigned long long seed, int n, unsigned long long* mismatches) {
  unsigned long long* d = nullptr;
  if (n < 0 || hipMalloc((void**)&d, sizeof(unsigned long long)) != hipSuccess) return 1;
  int rc = hipMemset(d, 0, sizeof(unsigned long long)) != hipSuccess;
  if (!rc && n > 0) hipLaunchKernelGGL(k_div_selftest, dim3((n + WG - 1) / WG), dim3(WG), 0, 0, seed, n, d);
  rc = rc || hipGetLastError() != hipSuccess ||
       hipMemcpy(mismatches, d, sizeof(unsigned long long), hipMemcpyDeviceToHost) != hipSuccess;
  (void)hipFree(d);
  return rc;
}

void launch_copy_d(hipStream_t s, const double* src, double* dst, size_t n) {
  if (n == 0) return;
  const size_t blocks = (n + WG - 1) / WG;
  hipLaunchKernelGGL(k_copy_d, dim3(blocks < 65536 ? (unsigned)blocks : 65536u), dim3(WG), 0, s,
                     src, dst, n);
}

void launch_update(hipStream_t s, int RK, double* U, double* U1p1, double* U1p2,
                   const double* Rku, const double* Res, const int8_t* fws, int ncube,
                   const int* cube_case, double* partials, bool body_only) {
  if (ncube > 1)
    hipLaunchKernelGGL(k_update, dim3(16, ncube - 1), dim3(WG), 0, s, RK, U, U1p1, U1p2, Rku,
                       Res, fws, cube_case, partials, body_only ? 1 : 0);
}

void launch_reduce(hipStream_t s, const double* partials, int stride, int single,
                   const CaseDesc* cases, int ncases, const DevPhys* phys, double* er) {
  if (ncases > 0)
    hipLaunchKernelGGL(k_reduce, dim3(ncases), dim3(REDUCE_WG), 0, s, partials, stride, single,
                       cases, phys, er);
}

void launch_shift(hipStream_t s, const double* U, double* U1, double* U1q, int ncube,
                  const int* cube_case) {
  if (ncube > 1)
    hipLaunchKernelGGL(k_shift, dim3(16, ncube - 1), dim3(WG), 0, s, U, U1, U1q, cube_case);
}

void launch_aos_to_soa(hipStream_t s, const double* aos, double* soa, int ncube) {
  const int n = ncube * PLANE;
  hipLaunchKernelGGL(k_aos_to_soa, dim3((n + WG - 1) / WG), dim3(WG), 0, s, aos, soa, n);
}

void launch_soa_to_aos(hipStream_t s, const double* soa, double* aos, int ncube) {
  const int n = ncube * PLANE;
  hipLaunchKernelGGL(k_soa_to_aos, dim3((n + WG - 1) / WG), dim3(WG), 0, s, soa, aos, n);
}

}  // namespace bcm
