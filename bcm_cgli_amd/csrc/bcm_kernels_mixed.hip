// Mixed-precision form of the per-iteration hot path for gfx950.
//
// FP32: the inner iterate U1_ (storage and arithmetic), the inviscid and
// viscous fluxes, the residual, the preconditioner and the RK stages.  The
// iterate is stored as its deviation d = U1_ - Uref from the case's freestream
// state Uref, and fluxes are formed as F(U) - F(Uref) from deviations only, so
// the FP32 rounding applies to the deviations (small away from the body)
// rather than to the full state, whose pressure and energy carry a large
// constant offset at these Mach numbers.
// FP64: the physical time levels U1 and U1q, the dual-time source
// -(3u - 4U1 + U1q)/(2 dT) (a difference of nearly equal states; its constant
// part 3 Uref - 4 U1 + U1q is formed once per physical step, at the shift), the
// norms and force sums, and the IB interpolation (bcm_kernels.hip, FP64
// arithmetic on the FP32 iterate).  The algorithm is the reference's
// (BCM_Flux_XYZ_Viscous_Runge_kutta.cpp:326-2655, cited as Flux.cpp); the
// operation order is free here, so divisions become reciprocal multiplies and
// square roots the hardware approximations.
//
// Kernel shape: one workgroup of 256 lanes per cube or run of its planes, a lane
// per (j,k), marching along i (k_flux_mixed below).  The kernel reads
// one copy of the iterate and writes the other, so each cell's RK update is
// stored as soon as it is computed: no stage increment array, no RK scratch
// arrays; the two layers next to a face with a neighbour are written into
// the neighbour's ghost layers as well, which replaces the face part of the
// post-update halo exchange.  The reference's RK2/RK3 read U1p1
// and U1p2, which equal U1_ at every fluid cell when those stages run (only
// ghost and non-fluid cells change in between), so the stages use U1_.
#include <hip/hip_runtime.h>
#include <math.h>

#include "bcm_kernels.h"

namespace bcm {
namespace {

constexpr int WG = 256;
constexpr float KGf = 1.4f;
constexpr float KM1f = 0.4f;
constexpr float IKM1f = 2.5f;          // 1/(K-1)
constexpr float IRGf = 1.0f / 287.0f;  // 1/R
constexpr float HEATf = 717.5f * 1.4f / 0.72f;   // Cv K / Pr
constexpr double KM1d = 1.4 - 1;

__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float fsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ float fmaxr(float a, float b) { return (a > b) ? a : b; }

// Reference (freestream) state of a case in FP32 and the quantities derived
// from it that the perturbation forms below need.
struct RefF {
  float rho, u[3], m[3], E, P, PoR, T;   // PoR = P0/rho0, T = P0/(rho0 R)
};

__device__ __forceinline__ RefF make_ref(const DevPhys& ph) {
  double r[5];
  ref_state(ph, r);
  RefF f;
  f.rho = (float)r[0];
  f.u[0] = (float)ph.Uin;
  f.u[1] = (float)ph.V0;
  f.u[2] = (float)ph.W0;
  for (int k = 0; k < 3; ++k) f.m[k] = (float)r[k + 1];
  f.E = (float)r[4];
  f.P = (float)ph.P0;
  f.PoR = (float)(ph.P0 / ph.rho0);
  f.T = (float)(ph.P0 / (ph.rho0 * 287.0));
  return f;
}

// One state d = U - Uref in perturbation form: density and its reciprocal,
// velocity u = u0 + du, pressure P = P0 + dP, total enthalpy H.  du and dP are
// formed from the deviations only (no difference of nearly equal numbers):
//   du = (dm - u0 drho) / rho,
//   dP = (K-1) (dE - (drho |u|^2 + rho0 sum du (u + u0)) / 2).
struct Side {
  float r, ir, du[3], u[3], dP, P, H;
};

__device__ __forceinline__ void side(const float (&d)[5], const RefF& rf, Side& s) {
  s.r = rf.rho + d[0];
  s.ir = frcp(s.r);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    s.du[k] = (d[k + 1] - rf.u[k] * d[0]) * s.ir;
    s.u[k] = rf.u[k] + s.du[k];
  }
  const float VV = s.u[0] * s.u[0] + s.u[1] * s.u[1] + s.u[2] * s.u[2];
  const float dke = 0.5f * (d[0] * VV + rf.rho * (s.du[0] * (s.u[0] + rf.u[0]) +
                                                  s.du[1] * (s.u[1] + rf.u[1]) +
                                                  s.du[2] * (s.u[2] + rf.u[2])));
  s.dP = KM1f * (d[4] - dke);
  s.P = rf.P + s.dP;
  s.H = 0.5f * VV + KGf * s.P * s.ir * IKM1f;
}

// Preconditioned Roe-type flux at a face with normal axis d (Flux.cpp:611-797)
// in perturbation form: F returns F(U) - F(Uref), which differs from the flux
// by a constant that cancels in every face difference of the residual.
//   mass      dm_d
//   momentum  dm_m u_d + m0_m du_d + dP [m = d]
//   energy    du_d (E + P) + u0_d (dE + dP)
// The dissipation is built from differences R - L as in the reference.  dP
// returns the deviation of the face pressure average.
// D is the face-normal axis; 3: the lane's own choice of y (ydir) or z.
template <int D>
__device__ __forceinline__ void roe_f(const float (&L)[5], const float (&R)[5], float e,
                                      const RefF& rf, float (&F)[5], float& dP, bool ydir = false) {
  Side l, r;
  side(L, rf, l);
  side(R, rf, r);
  const float t5 = fsqrt(l.r), t6 = fsqrt(r.r), it4 = frcp(t5 + t6);
  const float rho = t5 * t6;
  float q[3];
#pragma unroll
  for (int m = 0; m < 3; ++m) q[m] = (t5 * l.u[m] + t6 * r.u[m]) * it4;
  const float VV = q[0] * q[0] + q[1] * q[1] + q[2] * q[2];
  const float H = (t5 * l.H + t6 * r.H) * it4;
  const float C = (H - 0.5f * VV) * KM1f;
  const float beta = fmaxr(VV * frcp(C), e);
  const bool normal[3] = {D == 0, D == 3 ? ydir : D == 1, D == 3 ? !ydir : D == 2};
  auto pick = [&](const float (&x)[3]) { return D == 0 ? x[0] : (normal[1] ? x[1] : x[2]); };
  const float un = pick(q), lun = pick(l.u), run = pick(r.u), ldu = pick(l.du), rdu = pick(r.du);
  const float u0n = pick(rf.u);
  const float Ln = D == 0 ? L[1] : (normal[1] ? L[2] : L[3]);
  const float Rn = D == 0 ? R[1] : (normal[1] ? R[2] : R[3]);
  const float temp = 0.5f * (1 + beta) * un;
  const float S = 0.5f * fsqrt(4 * beta * C + un * un * (1 - beta) * (1 - beta));
  const float iS = frcp(S);
  const float dPr = r.dP - l.dP, dun = rdu - ldu;
  const float temp1 = dPr * frcp(rho * beta * C);
  const float tS = temp * iS;
  const float temp3 = 0.5f * (1 - beta) * un * tS;
  const float an = fabsf(un);
  const float deltaU = (S - temp3 - beta * an) * temp1 + tS * dun;
  const float deltaP = tS * dPr + (S - an + temp3) * rho * dun;
  const float dUr = deltaU * rho;
  F[0] = 0.5f * ((Ln + Rn) - (an * (R[0] - L[0]) + dUr));
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const float fav = an * (R[m + 1] - L[m + 1]) + dUr * q[m] + (normal[m] ? deltaP : 0.f);
    const float cen = (L[m + 1] * lun + rf.m[m] * ldu) + (R[m + 1] * run + rf.m[m] * rdu) +
                      (normal[m] ? l.dP + r.dP : 0.f);
    F[m + 1] = 0.5f * (cen - fav);
  }
  const float EPl = rf.E + rf.P + L[4] + l.dP, EPr = rf.E + rf.P + R[4] + r.dP;
  const float cenE = (ldu * EPl + u0n * (L[4] + l.dP)) + (rdu * EPr + u0n * (R[4] + r.dP));
  const float fav4 = an * (R[4] - L[4]) + dUr * H + deltaP * un;
  F[4] = 0.5f * (cenE - fav4);
  dP = 0.5f * (l.dP + r.dP);
}

// Face states of order 5, 3 or 1 (Flux.cpp:499-596) from six cells s0..s5 =
// p-2..p+3 of the face between p and p+1, as weighted sums with the order's
// weights (zero for the cells an order does not use), so that lanes of one
// wave with different orders run the same instructions:
//   5: L = (2 s0 - 13 s1 + 47 s2 + 27 s3 - 3 s4) / 60,
//      R = (-3 s1 + 27 s2 + 47 s3 - 13 s4 + 2 s5) / 60
//   3: L = (-s1 + 5 s2 + 2 s3) / 6,  R = (2 s2 + 5 s3 - s4) / 6
//   1: L = s2, R = s3.
// Cells outside an order's stencil must hold finite values (callers pass
// an in-range cell in their place).
struct ReconW {
  float a0, a1, a2, a3, a4, b1, b2, b3, b4, b5;
};
__device__ __forceinline__ ReconW recon_weights(int order) {
  const bool o5 = order == 5, o3 = order == 3;
  ReconW w;
  w.a0 = o5 ? 2.f / 60 : 0.f;
  w.a1 = o5 ? -13.f / 60 : (o3 ? -1.f / 6 : 0.f);
  w.a2 = o5 ? 47.f / 60 : (o3 ? 5.f / 6 : 1.f);
  w.a3 = o5 ? 27.f / 60 : (o3 ? 2.f / 6 : 0.f);
  w.a4 = o5 ? -3.f / 60 : 0.f;
  w.b1 = o5 ? -3.f / 60 : 0.f;
  w.b2 = o5 ? 27.f / 60 : (o3 ? 2.f / 6 : 0.f);
  w.b3 = o5 ? 47.f / 60 : (o3 ? 5.f / 6 : 1.f);
  w.b4 = o5 ? -13.f / 60 : (o3 ? -1.f / 6 : 0.f);
  w.b5 = o5 ? 2.f / 60 : 0.f;
  return w;
}
__device__ __forceinline__ void recon(const ReconW& w, float s0, float s1, float s2, float s3,
                                      float s4, float s5, float& L, float& R) {
  L = w.a0 * s0 + w.a1 * s1 + w.a2 * s2 + w.a3 * s3 + w.a4 * s4;
  R = w.b1 * s1 + w.b2 * s2 + w.b3 * s3 + w.b4 * s4 + w.b5 * s5;
}

__device__ __forceinline__ int order_fwd(int p, int fm1, int fp1, int fp2) {
  if (fp1 == 1 && fm1 == 1) return (p == 17 || fp2 != 1) ? 3 : 5;
  return 1;
}
__device__ __forceinline__ int order_bwd(int q, int fm2, int fm1, int fp1) {
  if (fp1 == 1 && fm1 == 1) return (q == 2 || fm2 != 1) ? 3 : 5;
  return 1;
}

// LDS layouts.  Lane t of a workgroup owns cell (j, k) with k = t % 16 + 2
// and j = 2 + w + 4 q for wave w = t / 64 and q = (t / 16) % 4: the four
// 16-cell rows a wave reads at once lie 4 rows apart, so row strides of 20
// (staged plane, primitive ring) put them on distinct LDS banks.
constexpr int PRW = 20;           // row stride of the primitive ring
constexpr int PR = 18 * PRW;      // primitive plane, j,k in [1,18]
constexpr int NFY = 4 * 80;       // y-face slots (17 rows of 16 in 4 blocks of 5 rows)
__device__ __forceinline__ int ring_idx(int jj, int kk) { return (jj - 1) * PRW + (kk - 1); }
// y-face between rows p and p+1 at k = kk (p = 1..17): block (p-1) % 4, row
// (p-1) / 4 in it, so a wave's rows are consecutive slots.
__device__ __forceinline__ int fy_idx(int p, int kk) {
  return ((p - 1) & 3) * 80 + ((p - 1) >> 2) * 16 + (kk - 2);
}
// States of the face between cells p and p+1 of a line whose cell p-2+m holds
// s(m, v): every order's weighted sum over the six cells (a lane's order may
// differ from its neighbour's).  An order below 5 does not use p-2 and p+3.
template <typename S>
__device__ __forceinline__ void face_states(int order, S s, float (&L)[5], float (&R)[5]) {
  const ReconW w = recon_weights(order);
#pragma unroll
  for (int v = 0; v < 5; ++v)
    recon(w, s(0, v), s(1, v), s(2, v), s(3, v), s(4, v), s(5, v), L[v], R[v]);
}

// The same along a line of the staged plane, st floats apart; base is cell p.
// Orders below 5 read cell p in place of the cells they do not use (which may
// lie beyond the plane).
__device__ __forceinline__ void plane_states(const float* cp, int base, int st, int order,
                                             float (&L)[5], float (&R)[5]) {
  const int o0 = order == 5 ? -2 * st : 0, o5 = order == 5 ? 3 * st : 0;
  face_states(order, [&](int m, int v) {
    return cp[v * 400 + base + (m == 0 ? o0 : m == 5 ? o5 : (m - 2) * st)];
  }, L, R);
}

// Viscous flux through the face between cell P and P + e_D (Flux.cpp:1946-2272,
// forward-face formulas of P): one evaluation serves both adjacent cells.  D as
// for roe_f.  ring holds deviations of u, v, w, T; rm, r0 and rp are the ring
// offsets of P in the plane before, its own and the next (rm unused for D = 0).
// L receives the x, y, z stress and the energy flux.
template <int D>
__device__ __forceinline__ void visc_face(const float (*ring)[3 * PR], int rm, int r0, int rp,
                                          const RefF& rf, float inv, float iT0, float muL,
                                          float sut, float (&L)[4], bool ydir = false) {
  // Ring steps of the face normal and of the in-plane tangents.
  const int sn = D == 1 ? PRW : D == 2 ? 1 : ydir ? PRW : 1;
  float me[4], fv[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    me[m] = ring[m][r0];
    fv[m] = D == 0 ? ring[m][rp] : ring[m][r0 + sn];
  }
  const float Tf = rf.T + 0.5f * (me[3] + fv[3]);
  const float temp = Tf * iT0;
  const float mu = muL * temp * fsqrt(temp) * sut * frcp(Tf + 110.f);
  const float q = 0.25f * inv;
  float gn[4], gx[4], gy[4], gz[4];   // gradients along the normal and the axes
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const float* a = ring[m];
    gn[m] = (fv[m] - me[m]) * inv;
    if (D == 0) {
      gx[m] = gn[m];
      gy[m] = (a[r0 + PRW] + a[rp + PRW] - a[r0 - PRW] - a[rp - PRW]) * q;
      gz[m] = (a[r0 + 1] + a[rp + 1] - a[r0 - 1] - a[rp - 1]) * q;
    } else {
      gx[m] = (a[rp] + a[rp + sn] - a[rm] - a[rm + sn]) * q;
      // The other in-plane axis.
      const int so = D == 1 ? 1 : D == 2 ? PRW : ydir ? 1 : PRW;
      const float go = (a[r0 + so] + a[r0 + sn + so] - a[r0 - so] - a[r0 + sn - so]) * q;
      if (D == 3) {
        gy[m] = ydir ? gn[m] : go;
        gz[m] = ydir ? go : gn[m];
      } else {
        gy[m] = D == 1 ? gn[m] : go;
        gz[m] = D == 1 ? go : gn[m];
      }
    }
  }
  const float uf = rf.u[0] + 0.5f * (me[0] + fv[0]), vf = rf.u[1] + 0.5f * (me[1] + fv[1]),
              wf = rf.u[2] + 0.5f * (me[2] + fv[2]);
  const float div = gx[0] + gy[1] + gz[2];
  const bool normal[3] = {D == 0, D == 3 ? ydir : D == 1, D == 3 ? !ydir : D == 2};
  // d/dm of the normal velocity, m = x, y, z.
  const float nx = D == 0 ? gx[0] : (normal[1] ? gx[1] : gx[2]);
  const float ny = D == 0 ? gy[0] : (normal[1] ? gy[1] : gy[2]);
  const float nz = D == 0 ? gz[0] : (normal[1] ? gz[1] : gz[2]);
  const float gd[3] = {nx, ny, nz};
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const float dia = 2 * gn[m] - (2.0f / 3.0f) * div, off = gn[m] + gd[m];
    L[m] = mu * (D == 3 ? (normal[m] ? dia : off) : m == D ? dia : off);
  }
  L[3] = uf * L[0] + vf * L[1] + wf * L[2] + mu * HEATf * gn[3];
}

// An address as a uniform base and a 32-bit byte offset per lane.
template <typename T>
__device__ __forceinline__ T& at_byte(T* base, unsigned off) {
  using B = std::conditional_t<std::is_const_v<T>, const char, char>;
  return *reinterpret_cast<T*>(reinterpret_cast<B*>(base) + off);
}

// One workgroup of 256 lanes marches through a run of a cube's i-planes, in two
// phases per plane:
//  1. the plane's 272 y-faces and 272 z-faces, inviscid and viscous, once each;
//     meanwhile the next plane's conserved values go from memory straight into
//     the other LDS buffer, and the lane's column cell three planes ahead and the
//     border cells two planes ahead into registers;
//  2. the primitives two planes ahead into the ring slot of the plane behind,
//     the x-face i+1/2 from the lane's column (two planes behind and two ahead
//     in registers, two in LDS), the differences, the residual, the increment,
//     the update and its stores.
//
// Runs: with nseg > 1 each cube's interior planes 2..17 are split into nseg runs
// of 16/nseg planes, one workgroup each (more workgroups when few cubes are
// resident).  A run starting at i0 > 2 first executes one prologue iteration at
// i0 - 1 that only forms the x-face i0 - 1/2 (inviscid and viscous) the run
// carries into its first plane: the same loop body, and so the same instructions
// and bits, as the unsegmented march computes it with.  Norm partials are one row
// per plane, so every result is bitwise the same for every nseg.
//
// Bound: vector instructions, 1,654 per cell (70% of the issue rate over the
// launch).  Two workgroups per CU: a third (46 KB of LDS, 168 registers with 25
// spilled) gives the same rate, 624 us on 2,048 cubes against 555.  Against a
// march that kept the whole column in registers, two face arrays more in LDS and
// a boundary round per axis: 570 -> 555 us on 2,048 cubes, 51 -> 45 on 125.  (476
// and 43 with what followed: quartered last cubes, BC regions carried by a kernel
// of their own, another schedule.  Bursts of some hundred launches; runs of seconds
// take 500 to 520 on 2,048.)
__global__ __launch_bounds__(WG, 2) void k_flux_mixed(
    float* __restrict__ U, float* __restrict__ Uout, const HaloSrc* __restrict__ halo,
    const uint8_t* __restrict__ cube_mask, const double* __restrict__ Bsrc,
    const int8_t* __restrict__ fws, const double* __restrict__ cube_size, PhysTab pt,
    double deltaT, double deltaTau, double e_d, int RK, double* __restrict__ partials,
    IbRefresh ib, Runs runs, int ncube) {
  __shared__ __align__(16) float cp[2][5 * 400];   // conserved values of planes i, i+1
  __shared__ int8_t fl[2][400];                    // flags of planes i, i+1
  __shared__ float pr[4][3 * PR];                  // u, v, w, T of planes i-1..i+1
  __shared__ float fy[9][NFY];                     // y-faces: flux, viscous flux
  __shared__ float fzb[10][16];                    // z-faces before k = 2: flux, pressure, viscous
  __shared__ double red[WG / 64][8];               // RK 3: norm sums of the waves
  __shared__ double tot[8];                        // and, of a whole cube, of its planes

  const RunOf run = run_of(runs, blockIdx.x);
  const int c = run.cube, seg = run.seg;
  if (c >= ncube) return;
  const int cc = pt.cube_case[c];
  if (cc < 0) return;
  const DevPhys ph = pt.phys[cc];
  // Planes i0..i1 of this run; the march starts at `start`.
  const int len = 16 / run.nseg;
  const int i0 = 2 + seg * len, i1 = i0 + len - 1;
  const int start = i0 == 2 ? 2 : i0 - 1;
  const double dxd = cube_size[c] / 16;
  const float inv = (float)(1.0 / dxd), vol = (float)(dxd * dxd * dxd);
  const float e = (float)e_d;
  const RefF rf = make_ref(ph);
  const float iT0 = (float)(1.0 / ph.T0), muL = (float)ph.mu_L;
  const float sut = (float)(ph.T0 + 110.);
  const double i2dT = 1.0 / (2 * deltaT);
  const float dT = (float)deltaT, dtau = (float)deltaTau;
  const float* Uc = U + (size_t)c * CUBE_STRIDE;
  const HaloSrc hs = halo[c];
  const int8_t* __restrict__ Fc = fws + (size_t)c * PLANE;
  // ZBC_IN_FLUX faces: the z-ghost cells (k = 0, 1 or 18, 19) of the interior
  // planes are taken as the z-BC sets them, from the cell k = 2 (w negated) or
  // 17 of the same row.
  const int zm = cube_mask[c];
  const bool zlo = (zm & ZBC_IN_FLUX) != 0, zhi = (zm & (ZBC_IN_FLUX << 1)) != 0;
  const double r3 = ph.rho0 * ph.W0;
  refresh_cube(U, ib, c);

  // The lane's cell, re-formed at the top of every plane iteration (below).
  int t = threadIdx.x;
  int j, k, col;
  auto lane = [&] {
    j = 2 + (t >> 6) + 4 * ((t >> 4) & 3);
    k = (t & 15) + 2;
    col = j * 20 + k;
  };
  lane();
  // The wave whose lanes 0..31 evaluate the faces next to the first ghost
  // layers (an extra round), and the one that forms the border primitives:
  // another wave for every workgroup, so that each SIMD has its share.
  const int wbnd = (blockIdx.x / 8) & 3, wbrd = wbnd ^ 2;

  // Plane p's conserved values from memory straight into buffer p & 1: 500
  // pieces of 16 bytes, piece q of a wave to the wave's LDS base (m0) + 16
  // lane.  In asm, since the compiler would wait for the copy before the next
  // read of any LDS array; wait_loads and a barrier stand between a copy and
  // its readers.
  auto stage = [&](int p) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const unsigned q = t + h * WG;
      if (q < 500) {
        const unsigned off = q / 100 * (4 * PLANE) + q % 100 * 16;
        const unsigned dst = __builtin_amdgcn_readfirstlane(
            (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)&cp[p & 1][0] +
            16 * ((t & ~63) + h * WG));
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :: "s"(dst), "v"(off), "s"(Uc + p * 400)
                     : "memory", "m0");
      }
    }
  };
  auto wait_loads = [] { __builtin_amdgcn_s_waitcnt(0xF70); };   // vmcnt(0)
  auto column = [&](int p, float (&q)[5]) {
#pragma unroll
    for (int v = 0; v < 5; ++v) q[v] = at_byte(Uc + v * PLANE + p * 400, 4u * col);
  };
  // ZBC_IN_FLUX: the staged plane's z-ghost cells, 4 per row of 20.
  auto fix_z = [&](int p) {
    const int row = t >> 2, q = t & 3;
    if (t >= 80 || !(q < 2 ? zlo : zhi)) return;
    float* b = cp[p & 1] + row * 20;
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      const float x = b[v * 400 + (q < 2 ? 2 : 17)];
      b[v * 400 + (q < 2 ? q : q + 16)] = v == 3 && q < 2 ? zbc_neg(x, r3) : x;
    }
  };
  // Deviations of the viscous block's primitives u, v, w and T = P/(rho R) of a
  // cell from the reference state, into ring offset o:
  // dT = (dP - (P0/rho0) drho) / (rho R).
  auto put_prims = [&](int o, const float (&q)[5]) {
    Side sd;
    side(q, rf, sd);
    pr[0][o] = sd.du[0];
    pr[1][o] = sd.du[1];
    pr[2][o] = sd.du[2];
    pr[3][o] = (sd.dP - rf.PoR * q[0]) * sd.ir * IRGf;
  };
  // Border cells of a primitive plane other than its corners: lane l of wave
  // wbrd.  Their conserved values are loaded a phase before they are used.  In
  // the ghost planes 1 and 18 they are edge ghost cells, the mean of two face
  // ghost cells (loaded where they are used, once per cube each).
  const int bl = t & 63, bm = (bl & 15) + 2;
  const int bj = bl < 16 ? 1 : bl < 32 ? 18 : bm, bk = bl < 32 ? bm : bl < 48 ? 1 : 18;
  const bool border = (t >> 6) == wbrd;
  // A border cell of an interior plane as ZBC_IN_FLUX faces have it.
  const bool blo = zlo && bk == 1, bhi = zhi && bk == 18;
  const int bcell = bj * 20 + (blo ? 2 : bhi ? 17 : bk);
  auto load_border = [&](int p, float (&q)[5]) {
    if (border && p >= 2 && p <= 17)
#pragma unroll
      for (int v = 0; v < 5; ++v) q[v] = at_byte(Uc + v * PLANE + p * 400, 4u * bcell);
  };
  auto fill_border = [&](int p, int slot, float (&q)[5]) {
    if (!border) return;
    if (p == 1 || p == 18) {
      int ea, eb;
      edge_sources(p, bj, bk, ea, eb);   // true: no corner among these cells
      // eb lies in the interior plane 2 or 17, ea in the ghost plane.
      if (blo || bhi) eb += blo ? 1 : -1;
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        const float x = Uc[v * PLANE + ea], y = Uc[v * PLANE + eb];
        q[v] = 0.5f * (x + (v == 3 && blo ? zbc_neg(y, r3) : y));
      }
    } else if (blo) {
      q[3] = zbc_neg(q[3], r3);
    }
    put_prims(slot + ring_idx(bj, bk), q);
  };
  // The four corners of interior plane p, edge ghost cells that only the
  // plane's own viscous faces read, from the staged plane.
  auto fill_corners = [&](int p, int slot) {
    const int l = t & 63;
    if ((t >> 6) != (wbrd ^ 1) || l >= 4) return;
    const float* b = cp[p & 1];
    const int jj = l & 2 ? 18 : 1, kk = l & 1 ? 18 : 1, jn = l & 2 ? 17 : 2, kn = l & 1 ? 17 : 2;
    const bool lo = zlo && kk == 1, hi = zhi && kk == 18;
    float q[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      const float x = b[v * 400 + jj * 20 + kn], y = b[v * 400 + jn * 20 + (lo || hi ? kn : kk)];
      q[v] = 0.5f * (x + (v == 3 && lo ? zbc_neg(y, r3) : y));
    }
    put_prims(slot + ring_idx(jj, kk), q);
  };
  int fo[2] = {0, 0};   // the lane's two flags of the plane to stage
  auto load_flags = [&](int p) {
    fo[0] = Fc[p * 400 + (unsigned)t];
    if (t < 400 - WG) fo[1] = Fc[p * 400 + WG + (unsigned)t];
  };
  auto store_flags = [&](int p) {
    fl[p & 1][t] = (int8_t)fo[0];
    if (t < 400 - WG) fl[p & 1][WG + t] = (int8_t)fo[1];
  };

  // ---- before the march: plane `start` staged, primitives of start-1, start
  // and start+1, the column's registers ----
  float p2[5], p1[5], n2[5];   // the lane's column cells of planes i-2, i-1, i+2
  float bq[5] = {1, 0, 0, 0, 0};   // border cell of plane i+2
  unsigned fb = 0;             // flags of planes i-2..i+2 equal to 1, bits 0..4
  {
    stage(start);
    load_flags(start);
    float own[2][5], b0[5] = {1, 0, 0, 0, 0}, b1[5] = {1, 0, 0, 0, 0}, b2[5] = {1, 0, 0, 0, 0};
    column(start - 2, p2);
    column(start - 1, p1);
    column(start, own[0]);
    column(start + 1, own[1]);
    column(start + 2, n2);
    load_border(start - 1, b0);
    load_border(start, b1);
    load_border(start + 1, b2);
#pragma unroll
    for (int m = 0; m < 4; ++m) fb |= (Fc[(start - 2 + m) * 400 + (unsigned)col] == 1) << m;
    const int o = ring_idx(j, k);
    put_prims(o, p1);
    put_prims(PR + o, own[0]);
    put_prims(2 * PR + o, own[1]);
    fill_border(start - 1, 0, b0);
    fill_border(start, PR, b1);
    fill_border(start + 1, 2 * PR, b2);
    store_flags(start);
    wait_loads();
    __syncthreads();
    // (Interior planes only: ghost planes' z-ghost cells are as the BCs left
    // them, and no run starts there.)
    if (zlo || zhi) fix_z(start);
    fill_corners(start, PR);
    __syncthreads();
  }
  float cF[5] = {0, 0, 0, 0, 0}, cdP = 0.f;   // x-face before plane i
  float cL[4] = {0, 0, 0, 0};                 // and its viscous flux
  int corder = -1;
  int sl0 = 0, sl1 = PR, sl2 = 2 * PR;        // ring slots of planes i-1, i, i+1

#pragma unroll 1
  for (int i = start; i <= i1; ++i) {
    // The lane index passes through an empty asm statement, so the quantities
    // derived from it are computed inside the iteration that uses them rather
    // than held across it.
    asm volatile("" : "+v"(t));
    lane();
    const bool pro = i < i0;    // prologue: only the x-face i + 1/2
    const float* __restrict__ cpi = cp[i & 1];
    const int8_t* __restrict__ fli = fl[i & 1];
    const int ro = ring_idx(j, k);

    // ---- phase 1: y- and z-faces of plane i ----
    // The row of the plane before, from the waves' sums: after the barrier that
    // closed that plane, before the one ahead of this plane's sums.
    if (RK == 3 && i > i0 && t < 8) {
      double s = red[0][t];
#pragma unroll
      for (int w = 1; w < WG / 64; ++w) s += red[w][t];
      if (run.nseg == 1)   // (in the order k_reduce adds rows)
        tot[t] = i == i0 + 1 ? s : tot[t] + s;
      else
        partials[((size_t)(c - 1) * MIXED_ROWS_PER_CUBE + (i - 3)) * 8 + t] = s;
    }
    stage(i + 1);
    load_flags(i + 1);
    float n3[5];
    column(min(i + 3, 19), n3);   // (plane 20 is not used: order 3 or 1 there)
    const int f2 = Fc[(i + 2) * 400 + (unsigned)col];
    load_border(i + 2, bq);
    // The viscous x-face before plane 2 (plane 1's ring slot is refilled in
    // phase 2).
    if (i == 2) visc_face<0>(pr, 0, sl0 + ro, sl1 + ro, rf, inv, iT0, muL, sut, cL);
    float zF[5], dPzf, zL[4];
    if (!pro) {
      const int8_t* f = fli + col;
      float L[5], R[5], F[5], dP, Lv[4];
      plane_states(cpi, col, 20, order_fwd(j, f[-20], f[20], f[40]), L, R);
      roe_f<1>(L, R, e, rf, F, dP);
      visc_face<1>(pr, sl0 + ro, sl1 + ro, sl2 + ro, rf, inv, iT0, muL, sut, Lv);
      const int g = fy_idx(j, k);
#pragma unroll
      for (int v = 0; v < 5; ++v) fy[v][g] = F[v];
#pragma unroll
      for (int v = 0; v < 4; ++v) fy[5 + v][g] = Lv[v];
      plane_states(cpi, col, 1, order_fwd(k, f[-1], f[1], f[2]), L, R);
      roe_f<2>(L, R, e, rf, zF, dPzf);
      visc_face<2>(pr, sl0 + ro, sl1 + ro, sl2 + ro, rf, inv, iT0, muL, sut, zL);
      // The 16 y-faces and 16 z-faces next to the first ghost layers.
      if ((t >> 6) == wbnd && (t & 63) < 32) {
        const bool ydir = t & 16;
        const int a = (t & 15) + 2, st = ydir ? 20 : 1;
        const int base = ydir ? 20 + a : a * 20 + 1;
        const int rb = ydir ? ring_idx(1, a) : ring_idx(a, 1);
        const int8_t* fa = fli + base;
        plane_states(cpi, base, st, order_bwd(2, fa[-st], fa[0], fa[2 * st]), L, R);
        roe_f<3>(L, R, e, rf, F, dP, ydir);
        visc_face<3>(pr, sl0 + rb, sl1 + rb, sl2 + rb, rf, inv, iT0, muL, sut, Lv, ydir);
        if (ydir) {
          const int gb = fy_idx(1, a);
#pragma unroll
          for (int v = 0; v < 5; ++v) fy[v][gb] = F[v];
#pragma unroll
          for (int v = 0; v < 4; ++v) fy[5 + v][gb] = Lv[v];
        } else {
#pragma unroll
          for (int v = 0; v < 5; ++v) fzb[v][a - 2] = F[v];
          fzb[5][a - 2] = dP;
#pragma unroll
          for (int v = 0; v < 4; ++v) fzb[6 + v][a - 2] = Lv[v];
        }
      }
    }
    wait_loads();
    __syncthreads();

    // ---- phase 2 ----
    // This cell's FP64 source constant Bv = 3 Uref - 4 U1 + U1q, first used in
    // the residual.
    const size_t row = (size_t)c * CUBE_STRIDE + i * 400;
    double Bv[5] = {0, 0, 0, 0, 0};
    if (!pro) {
#pragma unroll
      for (int v = 0; v < 5; ++v) Bv[v] = at_byte(Bsrc + row + v * PLANE, 8u * col);
    }
    // Primitives of plane i+2 into the ring slot of plane i-1, whose last
    // readers were the viscous y- and z-faces of plane i.
    store_flags(i + 1);
    if (i + 2 <= i1 + 1) {
      put_prims(sl0 + ro, n2);
      fill_border(i + 2, sl0, bq);
    }
    if (i < i1) {
      fill_corners(i + 1, sl2);
      if (zlo || zhi) fix_z(i + 1);
    }
    float u[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) u[v] = cpi[v * 400 + col];
    fb |= (unsigned)(f2 == 1) << 4;
    const auto is = [&](int m) { return (int)(fb >> m & 1); };
    // ---- inviscid x: forward face from the column, backward carried ----
    float Rx[5], px, pz;   // px, pz: face pressure differences
    {
      float n1[5];
      const float* cpn = cp[~i & 1];
#pragma unroll
      for (int v = 0; v < 5; ++v) n1[v] = cpn[v * 400 + col];
      auto at = [&](int m, int v) {
        return m == 0 ? p2[v] : m == 1 ? p1[v] : m == 2 ? u[v] : m == 3 ? n1[v] : m == 4 ? n2[v] : n3[v];
      };
      const int of = order_fwd(i, is(1), is(3), is(4));
      float L[5], R[5], Ff[5], dPf;
      face_states(of, at, L, R);
      roe_f<0>(L, R, e, rf, Ff, dPf);
      const int ob = order_bwd(i, is(0), is(1), is(3));
      if (!pro && (i == 2 || ob != corder)) {
        float q3[5];
        column(max(i - 3, 0), q3);   // (plane -1 is not used: order 3 or 1)
        face_states(ob, [&](int m, int v) { return m == 0 ? q3[v] : at(m - 1, v); }, L, R);
        roe_f<0>(L, R, e, rf, cF, cdP);
      }
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        Rx[v] = Ff[v] - cF[v];
        cF[v] = Ff[v];
      }
      px = dPf - cdP;
      cdP = dPf;
      corder = of;
    }
    float vF[5] = {0, 0, 0, 0, 0};
    {
      float Lf[4];
      visc_face<0>(pr, 0, sl1 + ro, sl2 + ro, rf, inv, iT0, muL, sut, Lf);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        vF[v + 1] = Lf[v] - cL[v];
        cL[v] = Lf[v];
      }
    }
    if (!pro) {
      const int8_t* f = fli + col;
      const int IF = f[0];
      float Ry[5], Rz[5];
      {
        float Fb[5], dPu;
        const int ff = fy_idx(j, k), fbk = fy_idx(j - 1, k);
        const int ob = order_bwd(j, f[-40], f[-20], f[20]);
        if (j == 2 || ob == order_fwd(j - 1, f[-40], f[0], f[20])) {
#pragma unroll
          for (int v = 0; v < 5; ++v) Fb[v] = fy[v][fbk];
        } else {
          float L[5], R[5];
          plane_states(cpi, col - 20, 20, ob, L, R);
          roe_f<1>(L, R, e, rf, Fb, dPu);
        }
#pragma unroll
        for (int v = 0; v < 5; ++v) Ry[v] = fy[v][ff] - Fb[v];
#pragma unroll
        for (int v = 0; v < 4; ++v) vF[v + 1] += fy[5 + v][ff] - fy[5 + v][fbk];
      }
      {
        // The z-face behind comes from the lane behind in the row of 16, the
        // first lane's from LDS.
        float Fb[10];
#pragma unroll
        for (int v = 0; v < 10; ++v) {
          const float x = v < 5 ? zF[v] : v == 5 ? dPzf : zL[v - 6];
          Fb[v] = __int_as_float(__builtin_amdgcn_update_dpp(
              __float_as_int(fzb[v][j - 2]), __float_as_int(x), 0x111, 0xf, 0xf, false));
        }
        const int ob = order_bwd(k, f[-2], f[-1], f[1]);
        if (!(k == 2 || ob == order_fwd(k - 1, f[-2], f[0], f[1]))) {
          float L[5], R[5], F[5];
          plane_states(cpi, col - 1, 1, ob, L, R);
          roe_f<2>(L, R, e, rf, F, Fb[5]);
#pragma unroll
          for (int v = 0; v < 5; ++v) Fb[v] = F[v];
        }
#pragma unroll
        for (int v = 0; v < 5; ++v) Rz[v] = zF[v] - Fb[v];
        pz = dPzf - Fb[5];
#pragma unroll
        for (int v = 0; v < 4; ++v) vF[v + 1] = (vF[v + 1] + (zL[v] - Fb[6 + v])) * inv;
      }

      // ---- residual with the FP64 dual-time source ----
      float Rk[5];
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        const double Rp = -(3.0 * (double)u[v] + Bv[v]) * i2dT;
        const float Rf = -(Rx[v] + Ry[v] + Rz[v]) * inv + (v == 0 ? 0.f : vF[v]);
        Rk[v] = (float)(Rp + (double)Rf);
      }

      // ---- preconditioned increment (Flux.cpp:2295-2375) and RK update ----
      double pn[8] = {0, 0, 0, 0, 0, 0, 0, 0};   // the cell's norm and force terms
      float nv[5];
#pragma unroll
      for (int v = 0; v < 5; ++v) nv[v] = u[v];
      if (IF == 1) {
        Side me;
        side(u, rf, me);
        const float U_ = me.u[0], V_ = me.u[1], W_ = me.u[2];
        const float irho = me.ir;
        const float VV = U_ * U_ + V_ * V_ + W_ * W_;
        const float P = me.P;
        const float C = KGf * P * irho;
        const float T = P * irho;
        const float H = 0.5f * VV + C * IKM1f;
        const float beta = fmaxr(VV * frcp(C), e);
        const float bm1 = beta - 1;
        const float itemp = frcp(KGf * T * (2 * dT + 3 * dtau) * (2 * dT + 3 * beta * dtau));
        const float temp2 = KM1f * bm1 * dT * dT;
        const float temp3 = H - H * KGf - VV + KGf * (T + VV);
        const float kTbt = 3 * KGf * T * beta * dtau;
        const float a4 = 4 * temp2 * itemp;              // 4 temp2 / temp
        const float b4 = 4 * temp3 * bm1 * dT * dT * itemp;
        const float d11 = 2 * dT * (-2 * (-KM1f * (H - VV) - temp3 * beta) * dT + kTbt) * itemp;
        const float dmm[3] = {
            2 * dT * (2 * KGf * (T - U_ * U_ * bm1) * dT + 2 * U_ * U_ * bm1 * dT + kTbt) * itemp,
            2 * dT * (2 * KGf * (T - V_ * V_ * bm1) * dT + 2 * V_ * V_ * bm1 * dT + kTbt) * itemp,
            2 * dT * (2 * KGf * (T - W_ * W_ * bm1) * dT + 2 * W_ * W_ * bm1 * dT + kTbt) * itemp};
        const float d55 = 2 * dT * (2 * H * KM1f * bm1 * dT + KGf * T * (2 * dT + 3 * beta * dtau)) * itemp;
        const float vel[3] = {U_, V_, W_};
        // Row 0: d11, -a4 U, -a4 V, -a4 W, a4.  Rows 1..3 (velocity m): b4 vm,
        // -a4 vm vn off-diagonal, dmm on the diagonal, a4 vm.  Row 4: b4 H,
        // -a4 H U, -a4 H V, -a4 H W, d55.
        const float sv = U_ * Rk[1] + V_ * Rk[2] + W_ * Rk[3];
        float out[5];
        out[0] = dtau * (d11 * Rk[0] - a4 * sv + a4 * Rk[4]);
#pragma unroll
        for (int m = 0; m < 3; ++m)
          out[m + 1] = dtau * (b4 * vel[m] * Rk[0] - a4 * vel[m] * (sv - vel[m] * Rk[m + 1]) +
                               dmm[m] * Rk[m + 1] + a4 * vel[m] * Rk[4]);
        out[4] = dtau * (b4 * H * Rk[0] - a4 * H * sv + d55 * Rk[4]);
        float un[5];
        if (RK == 1) {
#pragma unroll
          for (int v = 0; v < 5; ++v) un[v] = u[v] + out[v];
        } else if (RK == 2) {
#pragma unroll
          for (int v = 0; v < 5; ++v) un[v] = 0.75f * u[v] + 0.25f * u[v] + 0.25f * out[v];
        } else {
#pragma unroll
          for (int v = 0; v < 5; ++v)
            un[v] = (1.0f / 3.0f) * u[v] + (2.0f / 3.0f) * u[v] + (2.0f / 3.0f) * out[v];
        }
#pragma unroll
        for (int v = 0; v < 5; ++v) nv[v] = un[v];
        if (RK == 3) {
          // Change norms in FP64 (Flux.cpp:2530-2566).
          double uref[5], fo5[5], fn[5];
          ref_state(ph, uref);
#pragma unroll
          for (int v = 0; v < 5; ++v) {
            fo5[v] = (double)u[v] + uref[v];
            fn[v] = (double)un[v] + uref[v];
          }
          const double ro5 = fo5[0], iro = 1.0 / ro5;
          const double uo = fo5[1] * iro, vo = fo5[2] * iro, wo = fo5[3] * iro;
          const double Po = (fo5[4] - 0.5 * ro5 * (uo * uo + vo * vo + wo * wo)) * KM1d;
          const double r = fn[0], ir = 1.0 / r;
          const double uu = fn[1] * ir, vv = fn[2] * ir, ww = fn[3] * ir;
          const double Pn = (fn[4] - 0.5 * r * (uu * uu + vv * vv + ww * ww)) * KM1d;
          const double dTn = Pn * ir - Po * iro;
          pn[0] = (Pn - Po) * (Pn - Po);
          pn[1] = (uu - uo) * (uu - uo);
          pn[2] = (vv - vo) * (vv - vo);
          pn[3] = (ww - wo) * (ww - wo);
          pn[4] = dTn * dTn;
        }
      } else if (IF < 1 && RK == 3) {
        // Force density of non-fluid cells (Flux.cpp:2395-2398), summed at RK 3.
        pn[5] = (double)(-(-px * inv + vF[1]) * vol);
        pn[6] = (double)(-(-pz * inv + vF[3]) * vol);
      }
      // Every interior cell goes to Uout; cells next to a face with a
      // neighbour also go to that neighbour's ghost layers.
      {
        const int nx = i <= 3 ? hs.src[0] : (i >= 16 ? hs.src[1] : 0);
        const int ny = j <= 3 ? hs.src[2] : (j >= 16 ? hs.src[3] : 0);
        const int nz = k <= 3 ? hs.src[4] : (k >= 16 ? hs.src[5] : 0);
        const int o = i * 400 + col;
        const int oy = o + (j <= 3 ? 16 * 20 : -16 * 20);
        const int oz = o + (k <= 3 ? 16 : -16);
        const size_t rx = (size_t)nx * CUBE_STRIDE + (i <= 3 ? i + 16 : i - 16) * 400;
#pragma unroll
        for (int v = 0; v < 5; ++v) {
          at_byte(Uout + row + v * PLANE, 4u * col) = nv[v];
          if (nx > 0) at_byte(Uout + rx + v * PLANE, 4u * col) = nv[v];
        }
        if (ny > 0) {
          float* O = Uout + (size_t)ny * CUBE_STRIDE + oy;
#pragma unroll
          for (int v = 0; v < 5; ++v) O[v * PLANE] = nv[v];
        }
        if (nz > 0) {
          float* O = Uout + (size_t)nz * CUBE_STRIDE + oz;
#pragma unroll
          for (int v = 0; v < 5; ++v) O[v * PLANE] = nv[v];
        }
      }
      if (RK == 3) {
        const double s = wave_sum8(pn);
        if ((t & 7) == 0) red[t >> 6][(t >> 3) & 7] = s;
      }
    }  // !pro

    // ---- advance the column, the flags and the ring ----
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      p2[v] = p1[v];
      p1[v] = u[v];
      n2[v] = n3[v];
    }
    fb >>= 1;
    const int s = sl0;
    sl0 = sl1;
    sl1 = sl2;
    sl2 = s;
    __syncthreads();
  }
  if (RK == 3 && t < 8) {
    double s = red[0][t];
#pragma unroll
    for (int w = 1; w < WG / 64; ++w) s += red[w][t];
    const size_t row = (size_t)(c - 1) * MIXED_ROWS_PER_CUBE;
    if (run.nseg == 1)
      partials[row * 8 + t] = tot[t] + s;
    else
      partials[(row + i1 - 2) * 8 + t] = s;
  }
}

__global__ __launch_bounds__(WG) void k_shift_mixed(const float* __restrict__ U,
                                                    double* __restrict__ U1,
                                                    double* __restrict__ U1q,
                                                    double* __restrict__ Bsrc, PhysTab pt) {
  const int c = blockIdx.y + 1;
  const int cc = pt.cube_case[c];
  if (cc < 0) return;
  double ref[5];
  ref_state(pt.phys[cc], ref);
  const int i = blockIdx.x + 2;
  const int j = (threadIdx.x >> 4) + 2;
  const int k = (threadIdx.x & 15) + 2;
  const size_t b = (size_t)c * CUBE_STRIDE + i * 400 + j * 20 + k;
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    const size_t o = b + (size_t)v * PLANE;
    const double q = U1[o], n = (double)U[o] + ref[v];
    U1q[o] = q;
    U1[o] = n;
    Bsrc[o] = 3.0 * ref[v] - 4.0 * n + q;
  }
}

// Bsrc <- 3 Uref - 4 U1 + U1q on the interior cells of cubes first + blockIdx.y.
__global__ __launch_bounds__(WG) void k_bsrc_mixed(const double* __restrict__ U1,
                                                   const double* __restrict__ U1q,
                                                   double* __restrict__ Bsrc, int first,
                                                   PhysTab pt) {
  const int c = first + blockIdx.y;
  const int cc = pt.cube_case[c];
  if (cc < 0) return;
  double ref[5];
  ref_state(pt.phys[cc], ref);
  const int i = blockIdx.x + 2;
  const int j = (threadIdx.x >> 4) + 2;
  const int k = (threadIdx.x & 15) + 2;
  const size_t b = (size_t)c * CUBE_STRIDE + i * 400 + j * 20 + k;
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    const size_t o = b + (size_t)v * PLANE;
    Bsrc[o] = 3.0 * ref[v] - 4.0 * U1[o] + U1q[o];
  }
}

struct Ref5 {
  double r[5];
};

__global__ __launch_bounds__(WG) void k_copy_f(const float* __restrict__ src,
                                               float* __restrict__ dst, size_t n) {
  for (size_t g = (size_t)blockIdx.x * WG + threadIdx.x; g < n; g += (size_t)gridDim.x * WG)
    dst[g] = src[g];
}

__global__ __launch_bounds__(WG) void k_aos_to_soa_f(const double* __restrict__ aos,
                                                     float* __restrict__ soa, int ncells,
                                                     Ref5 ref) {
  const int g = blockIdx.x * WG + threadIdx.x;
  if (g >= ncells) return;
  const int c = g / PLANE, cell = g % PLANE;
#pragma unroll
  for (int v = 0; v < 5; ++v)
    soa[(size_t)c * CUBE_STRIDE + (size_t)v * PLANE + cell] =
        (float)(aos[(size_t)g * 5 + v] - ref.r[v]);
}

__global__ __launch_bounds__(WG) void k_soa_to_aos_f(const float* __restrict__ soa,
                                                     double* __restrict__ aos, int ncells,
                                                     Ref5 ref) {
  const int g = blockIdx.x * WG + threadIdx.x;
  if (g >= ncells) return;
  const int c = g / PLANE, cell = g % PLANE;
#pragma unroll
  for (int v = 0; v < 5; ++v)
    aos[(size_t)g * 5 + v] =
        (double)soa[(size_t)c * CUBE_STRIDE + (size_t)v * PLANE + cell] + ref.r[v];
}

}  // namespace

int launch_flux_mixed(hipStream_t s, float* Uin, float* Uout, const HaloSrc* halo,
                       const uint8_t* cube_mask, const double* Bsrc, const int8_t* fws,
                       const double* cube_size, int ncube, PhysTab pt, double deltaT,
                       double deltaTau, double e, int RK, double* partials, IbRefresh ib, int nseg) {
  if (ncube <= 1) return 0;
  const Runs runs = runs_for(ncube, nseg);
  hipLaunchKernelGGL(k_flux_mixed, run_grid(runs, ncube), dim3(WG), 0, s, Uin, Uout, halo,
                     cube_mask, Bsrc, fws, cube_size, pt, deltaT, deltaTau, e, RK, partials, ib,
                     runs, ncube);
  return single_rows(runs, ncube);
}

// Runs per cube of the mixed flux kernel; the chip holds 512 of its workgroups.
// Most runs that fit at once to 128 cubes (8 cubes: 14 us in 16 runs, 106 in one;
// 64: 28 in 8; 128: 46 in 4, 112 in one); above, a run's prologue stands against
// the last wave of workgroups: 8 runs to 200 cubes (180: 62 us, 66 in 4), 4 to
// 370 (343: 104, 112 in 2), 2 to 560 (512: 146, 150 in 4, 154 in one), then one
// with quartered last cubes (runs_for; 576: 154, 171 in 2; 1,000: 254, 271 in 2).
int mixed_runs(int n) {
  return n <= 32 ? 16 : n <= 64 ? 8 : n <= 128 ? 4 : n <= 200 ? 8 : n <= 370 ? 4 : n <= 560 ? 2
       : 1;
}

void launch_copy_f(hipStream_t s, const float* src, float* dst, size_t n) {
  if (n == 0) return;
  const size_t blocks = (n + WG - 1) / WG;
  hipLaunchKernelGGL(k_copy_f, dim3(blocks < 65536 ? (unsigned)blocks : 65536u), dim3(WG), 0, s,
                     src, dst, n);
}

void launch_shift_mixed(hipStream_t s, const float* U, double* U1, double* U1q, double* Bsrc,
                        int ncube, PhysTab pt) {
  if (ncube > 1)
    hipLaunchKernelGGL(k_shift_mixed, dim3(16, ncube - 1), dim3(WG), 0, s, U, U1, U1q, Bsrc, pt);
}

void launch_bsrc_mixed(hipStream_t s, const double* U1, const double* U1q, double* Bsrc, int first,
                       int n, PhysTab pt) {
  if (n > 0)
    hipLaunchKernelGGL(k_bsrc_mixed, dim3(16, n), dim3(WG), 0, s, U1, U1q, Bsrc, first, pt);
}

void launch_aos_to_soa_f(hipStream_t s, const double* aos, float* soa, int ncube,
                         const double* ref5) {
  const int n = ncube * PLANE;
  Ref5 r;
  for (int v = 0; v < 5; ++v) r.r[v] = ref5[v];
  hipLaunchKernelGGL(k_aos_to_soa_f, dim3((n + WG - 1) / WG), dim3(WG), 0, s, aos, soa, n, r);
}

void launch_soa_to_aos_f(hipStream_t s, const float* soa, double* aos, int ncube,
                         const double* ref5) {
  const int n = ncube * PLANE;
  Ref5 r;
  for (int v = 0; v < 5; ++v) r.r[v] = ref5[v];
  hipLaunchKernelGGL(k_soa_to_aos_f, dim3((n + WG - 1) / WG), dim3(WG), 0, s, soa, aos, n, r);
}

}  // namespace bcm
