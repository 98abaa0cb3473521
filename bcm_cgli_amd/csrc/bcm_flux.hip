// Marching FP64 flux kernel for gfx950: flux, residual, preconditioned
// increment and (but for FLUX_ONLY) the RK update of one stage.  Every
// expression is the reference's, in its order, so results are bitwise those of
// the reference's FP64 CPU path.  "Flux.cpp" is
// BCM_Flux_XYZ_Viscous_Runge_kutta.cpp.
#include <hip/hip_runtime.h>

#include "bcm_fp64.h"
#include "bcm_kernels.h"

namespace bcm {
namespace {

// What the kernel does with a cell's increment.
enum March {
  FLUX_ONLY,   // stores it in Rku; several runs of planes per cube
  IN_PLACE,    // stores it and applies the RK update in place; one run per cube
  PUSH         // writes the update to the other copy of the iterate; several runs
};

constexpr int PR_ROW = 18, PR_PLANE = 18 * PR_ROW;   // primitives of j,k in [1,18]
constexpr int NFY = 17 * 16;                         // y-faces of one plane

struct MarchArgs {
  double* U;
  const double *U1, *U1q;
  const int8_t* fws;
  const double* cube_size;
  double *Rku, *Res;
  PhysTab pt;
  double deltaT, deltaTau, e;
  Runs runs;
  int RK, ncube;
  double *U1p1, *U1p2, *partials, *Uout;
  const HaloSrc* halo;
  const uint8_t* cube_mask;
  IbRefresh ib;
  bool rku;   // AUX: store Rku1 and Residual1
};

// An address as a uniform base and a 32-bit offset per lane (no 64-bit vector
// arithmetic).
template <typename T>
__device__ __forceinline__ T& at_byte(T* base, unsigned off) {
  using B = std::conditional_t<std::is_const_v<T>, const char, char>;
  return *reinterpret_cast<T*>(reinterpret_cast<B*>(base) + off);
}

// One workgroup of 256 lanes, lane (j,k), marches through a run of a cube's
// i-planes.  Per plane, in two phases closed by one barrier each:
//  1. the plane's 272 y-faces and 272 z-faces, once each, from its conserved
//     values in LDS; meanwhile the next plane's go from memory straight into the
//     other LDS buffer and the lane's column cell three planes ahead into
//     registers;
//  2. the next plane's primitives (u, v, w, T) into a 3-plane LDS ring, each
//     computed once instead of once per neighbour; the x-face i+1/2 from the
//     lane's column (two planes behind and two ahead in registers, two in LDS);
//     the cell's y- and z-differences;
// then, with nothing left to exchange, the viscous terms, the residual, the
// increment and the update.  No phase waits for a load issued in it: at two
// waves per SIMD a memory latency is not covered by the other wave.
// A cell whose backward-face order differs from its neighbour's forward-face
// order evaluates its own backward face, as the reference does.
//
// PUSH: the update is written to Uout, with every interior cell (non-fluid
// cells unchanged) and, for the two layers next to a face with an equal-size
// neighbour, into that neighbour's ghost layers: the face part of the
// post-update exchange.  It uses U for U1p1 (RK2) and U1p2 (RK3): those equal
// U1_ bitwise at fluid cells during a stage sequence, since only ghost and
// non-fluid cells change between stages.  It reads none of Rku1, U1p1, U1p2
// and Residual1 back and stores them only with AUX, which the engine asks for
// in the last inner iteration of a step; Rku1 and Residual1, which every stage
// overwrites, then in the step's last stage only (2,048 cubes: 1,268 us with
// them in each stage, 1,119 without, 993 without AUX).  The edge ghost cells the viscous
// stencil reads are not read from memory (no edge pass runs between the
// stage's face updates and this kernel) but formed as the pre-flux exchange's
// edge passes would leave them, the mean of two face ghost cells: the corners
// of an interior plane, and the border cells other than the corners of the
// ghost planes 1 and 18.  ZBC_IN_FLUX faces: the z-ghost cells (k = 0, 1 or 18,
// 19) of the interior planes are taken as the z-BC sets them, from the cell
// k = 2 (w negated) or 17 of the same row.
//
// Runs: a run's first plane needs the x-face before it (evaluated before the
// march) and two primitive planes; nothing else is done twice.
//
// Bound: vector instructions, 2,797 per cell (68% of the issue rate); 253 VGPRs
// and 76 KB of LDS give two workgroups per CU.  Against a march that loaded the plane's and the
// column's cells in the iteration that uses them, with three barriers and one
// boundary round per axis: 1,252 -> 1,004 us on 2,048 cubes (PUSH), 1,487 ->
// 1,072 (IN_PLACE).  (PUSH 947 with quartered last cubes and without the copy of
// the BC regions.  These are bursts of some hundred launches; runs of seconds
// take 960 to 1,080.)
template <March MODE, bool AUX>
__global__ __launch_bounds__(WG, 2) void k_flux_march(const MarchArgs A) {
  __shared__ __align__(16) double cp[2][5 * 400];   // conserved values of planes i, i+1
  __shared__ double pr[4][3 * PR_PLANE];            // u, v, w, T = P/(rho R)
  __shared__ double fy[5][NFY];
  __shared__ double fzb[6][16];                     // z-faces before k = 2: flux, pressure
  __shared__ int8_t fl[2][400];                     // flags of planes i, i+1
  __shared__ double red[WG / 64][8];                // RK 3: norm sums of the waves
  __shared__ double tot[8];                         // and of the cube's planes
  const int RK = A.RK;
  const RunOf run = run_of(A.runs, blockIdx.x);
  const int c = run.cube, seg = run.seg;
  if (c >= A.ncube) return;
  const int cc = A.pt.cube_case[c];
  if (cc < 0) return;
  const DevPhys ph = A.pt.phys[cc];
  const double deltaT = A.deltaT, deltaTau = A.deltaTau, e = A.e;
  const int len = 16 / run.nseg;
  const int i0 = 2 + seg * len, i1 = i0 + len - 1;
  const double dx = A.cube_size[c] / 16;
  const double inv = 1. / dx;
  const double inv4 = 0.25 * inv;   // (x / 4) inv = x (inv / 4): the scaling by 1/4 is exact
  // x / 2^n equals x * 2^-n exactly: use the multiply when dx is a power of two.
  int ex;
  const bool pow2 = frexp(dx, &ex) == 0.5;
  const DivBy ddx = div_by_uniform(dx), dT0 = div_by_uniform(ph.T0), d2t = div_by_uniform(2 * deltaT);
  const double* Uc = A.U + (size_t)c * CUBE_STRIDE;
  const int8_t* __restrict__ Fc = A.fws + (size_t)c * PLANE;
  HaloSrc hs;
  if (MODE == PUSH) hs = A.halo[c];
  const int zm = MODE == PUSH ? A.cube_mask[c] : 0;
  const bool zlo = zm & ZBC_IN_FLUX, zhi = zm & (ZBC_IN_FLUX << 1);
  if (MODE == PUSH) refresh_cube(A.U, A.ib, c);

  // The lane's indices, re-formed at the top of every plane iteration (below).
  int t = threadIdx.x;
  int j = (t >> 4) + 2, k = (t & 15) + 2, col = j * 20 + k;
  // The wave whose lanes 0..31 evaluate the faces next to the first ghost
  // layers (an extra round), and the one that forms the border primitives:
  // another wave for every workgroup, so that each SIMD has its share.
  const int wbnd = (blockIdx.x / 8) & 3, wbrd = wbnd ^ 2;

  // Plane p's conserved values from memory straight into buffer p & 1: lane l
  // of a wave moves 16 bytes to the wave's LDS base (m0) + 16 l.  In asm, since
  // the compiler would wait for the copy before the next read of any LDS
  // array; wait_loads and a barrier stand between a copy and its readers.
  auto stage = [&](int p) {
    if (t < 200) {
      const unsigned off = 16 * t;
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        const unsigned dst = __builtin_amdgcn_readfirstlane(
            (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)&cp[p & 1][v * 400] +
            16 * (t & ~63));
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :: "s"(dst), "v"(off), "s"(Uc + (size_t)v * PLANE + p * 400)
                     : "memory", "m0");
      }
    }
  };
  auto wait_loads = [] { __builtin_amdgcn_s_waitcnt(0xF70); };   // vmcnt(0)
  auto column = [&](int p, double (&q)[5]) {
#pragma unroll
    for (int v = 0; v < 5; ++v) q[v] = at_byte(Uc + (size_t)v * PLANE + p * 400, 8u * col);
  };
  // ZBC_IN_FLUX: the staged plane's z-ghost cells, 4 per row of 20.
  auto fix_z = [&](int p) {
    const int row = t >> 2, q = t & 3;
    if (t >= 80 || !(q < 2 ? zlo : zhi)) return;
    double* b = cp[p & 1] + row * 20;
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      const double x = b[v * 400 + (q < 2 ? 2 : 17)];
      b[v * 400 + (q < 2 ? q : q + 16)] = v == 3 && q < 2 ? -x : x;
    }
  };
  // A cell's primitives into ring slot s.
  auto put_prims = [&](int s, int n, const double (&q)[5]) {
    const double r = q[0];
    const DivBy dq = div_by(r);
    const double u = div_sh(dq, q[1]), v = div_sh(dq, q[2]), w = div_sh(dq, q[3]);
    const double P = (q[4] - 0.5 * r * (u * u + v * v + w * w)) * KM1;
    const int o = s * PR_PLANE + n;
    pr[0][o] = u;
    pr[1][o] = v;
    pr[2][o] = w;
    pr[3][o] = dvd(P, r * RG);
  };
  // Primitives of plane p from its staged buffer into ring slot s: the lane's
  // own cell, and on waves wbrd (sides) and wbrd ^ 1 (corners) the border.  A
  // border cell is the mean of two cells a and b, the same cell where it is no
  // edge ghost cell (0.5 (x + x) = x).  `inner` is the buffer of the interior
  // plane next to a ghost plane.
  auto fill_prims = [&](int p, int s) {
    const double* b = cp[p & 1];
    double q[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) q[v] = b[v * 400 + col];
    put_prims(s, (j - 1) * PR_ROW + (k - 1), q);
    const int w = t >> 6, l = t & 63;
    if (!(w == wbrd || (w == (wbrd ^ 1) && l < 4))) return;
    const bool corner = w != wbrd, ghost = p == 1 || p == 18;
    int jj, kk;
    if (corner) {
      jj = l & 2 ? 18 : 1;
      kk = l & 1 ? 18 : 1;
    } else {
      const int side = l >> 4, m = (l & 15) + 2;
      jj = side == 0 ? 1 : side == 1 ? 18 : m;
      kk = side == 2 ? 1 : side == 3 ? 18 : m;
    }
    int ca = jj * 20 + kk, cb = ca;
    const double* bb = b;
    bool na = false, nb = false;
    if (MODE == PUSH) {
      const int jn = jj == 1 ? 2 : 17, kn = kk == 1 ? 2 : 17;   // next interior row, column
      const bool lo = zlo && kk == 1, hi = zhi && kk == 18;      // z-BC on cells k = 1, 18
      if (ghost) {
        if (!corner) {
          ca = l < 32 ? jn * 20 + kk : jj * 20 + kn;
          bb = cp[~p & 1];
          if (l >= 32 && (lo || hi)) cb = jj * 20 + kn;
          nb = l >= 32 && lo;
        }
      } else if (corner) {
        ca = jj * 20 + kn;
        cb = jn * 20 + (lo || hi ? kn : kk);
        nb = lo;
      } else if (l >= 32 && (lo || hi)) {
        ca = cb = jj * 20 + kn;
        na = nb = lo;
      }
    }
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      const double x = b[v * 400 + ca];
      if (MODE == PUSH) {
        const double y = bb[v * 400 + cb];
        q[v] = 0.5 * ((v == 3 && na ? -x : x) + (v == 3 && nb ? -y : y));
      } else {
        q[v] = x;
      }
    }
    put_prims(s, (jj - 1) * PR_ROW + (kk - 1), q);
  };

  // ---- before the march: planes i0-1 and i0 staged, the column's registers,
  // the x-face before plane i0 ----
  double p2[5], p1[5], n2[5];   // the lane's column cells of planes i-2, i-1, i+2
  double p3[5] = {0, 0, 0, 0, 0};   // IN_PLACE: plane i-3, no longer in memory
  double cF[5], cdP;            // x-face before plane i, and the order it was formed with
  int corder;
  unsigned fb = 0;              // flags of planes i-2..i+2 equal to 1, bits 0..4
  int fo[2] = {0, 0};           // the lane's two flags of the plane to stage
  auto load_flags = [&](int p) {
    fo[0] = Fc[p * 400 + (unsigned)t];
    if (t < 400 - WG) fo[1] = Fc[p * 400 + WG + (unsigned)t];
  };
  auto store_flags = [&](int p) {
    fl[p & 1][t] = (int8_t)fo[0];
    if (t < 400 - WG) fl[p & 1][WG + t] = (int8_t)fo[1];
  };
  {
    stage(i0 - 1);
    stage(i0);
    load_flags(i0);
    double s[6][5];
#pragma unroll
    for (int m = 0; m < 6; ++m) column(max(i0 - 3 + m, 0), s[m]);   // (plane -1 is not read)
#pragma unroll
    for (int m = 0; m < 4; ++m) fb |= (Fc[(i0 - 2 + m) * 400 + (unsigned)col] == 1) << m;
    wait_loads();
    __syncthreads();
    if (zlo || zhi) {
      // (No run starts at a ghost plane, whose z-ghost cells the BCs wrote.)
      fix_z(i0);
      if (i0 > 2) fix_z(i0 - 1);
      __syncthreads();
    }
    store_flags(i0);
    fill_prims(i0 - 1, 0);
    fill_prims(i0, 1);
    const auto is = [&](int m) { return (int)(fb >> m & 1); };
    corder = order_bwd(i0, is(0), is(1), is(3));
    double L[5], R[5];
    face_states(corder, [&](int m, int v) { return s[m][v]; }, L, R);
    roe_flux<0>(L, R, e, cF, cdP);
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      if (MODE == IN_PLACE) p3[v] = s[0][v];
      p2[v] = s[1][v];
      p1[v] = s[2][v];
      n2[v] = s[5][v];
    }
    __syncthreads();
  }
  // RK 3: totals of a plane's norm and force terms (lanes 0..7; waves in order).
  auto plane_row = [&] {
    double s = red[0][t];
#pragma unroll
    for (int w = 1; w < WG / 64; ++w) s += red[w][t];
    return s;
  };
  const bool single = MODE == IN_PLACE || run.nseg == 1;   // one row per cube
  int sl0 = 0, sl1 = 1, sl2 = 2;           // ring slots of planes i-1, i, i+1

#pragma unroll 1
  for (int i = i0; i <= i1; ++i) {
    // The lane index passes through an empty asm statement, so every
    // per-lane quantity derived from it (LDS addresses, face and flag
    // indices) is computed inside the iteration that uses it rather than
    // hoisted before the loop and held across it, where it would spill.
    asm volatile("" : "+v"(t));
    j = (t >> 4) + 2;
    k = (t & 15) + 2;
    col = j * 20 + k;
    const double* __restrict__ cpi = cp[i & 1];
    const int8_t* __restrict__ fli = fl[i & 1];

    // ---- phase 1: y- and z-faces of plane i ----
    stage(i + 1);
    load_flags(i + 1);
    double n3[5];
    column(min(i + 3, 19), n3);   // (plane 20 is not read: order 3 or 1 there)
    const int f2 = Fc[(i + 2) * 400 + (unsigned)col];
    double zF[5], dPzf;
    {
      const int8_t* f = fli + col;
      double L[5], R[5], F[5], dP;
      face_states(order_fwd(j, f[-20], f[20], f[40]),
                  [&](int m, int v) { return cpi[v * 400 + col + (m - 2) * 20]; }, L, R);
      roe_flux<1>(L, R, e, F, dP);
#pragma unroll
      for (int v = 0; v < 5; ++v) fy[v][(j - 1) * 16 + (k - 2)] = F[v];
      face_states(order_fwd(k, f[-1], f[1], f[2]),
                  [&](int m, int v) { return cpi[v * 400 + col + (m - 2)]; }, L, R);
      roe_flux<2>(L, R, e, zF, dPzf);
    }
    // The 16 y-faces and 16 z-faces next to the first ghost layers.
    if ((t >> 6) == wbnd && (t & 63) < 32) {
      const bool ydir = t & 16;
      const int a = (t & 15) + 2, st = ydir ? 20 : 1;
      const int base = ydir ? 20 + a : a * 20 + 1;
      const int8_t* f = fli + base;
      double L[5], R[5], F[5], dP;
      face_states(order_bwd(2, f[-st], f[0], f[2 * st]),
                  [&](int m, int v) { return cpi[v * 400 + base + (m - 2) * st]; }, L, R);
      roe_flux<3>(L, R, e, F, dP, ydir);
      if (ydir) {
#pragma unroll
        for (int v = 0; v < 5; ++v) fy[v][a - 2] = F[v];
      } else {
#pragma unroll
        for (int v = 0; v < 5; ++v) fzb[v][a - 2] = F[v];
        fzb[5][a - 2] = dP;
      }
    }
    wait_loads();
    __syncthreads();

    // ---- phase 2: primitives of plane i+1, x-face, differences ----
    // One row of norm partials per plane, so the norms do not depend on the
    // runs; a whole cube's rows are added here, in the order k_reduce would.
    if (MODE != FLUX_ONLY && RK == 3 && i > i0 && t < 8) {
      const double s = plane_row();
      if (single)
        tot[t] = i == i0 + 1 ? s : tot[t] + s;
      else
        A.partials[((size_t)(c - 1) * PUSH_ROWS_PER_CUBE + (i - 3)) * 8 + t] = s;
    }
    store_flags(i + 1);
    fill_prims(i + 1, sl2);
    if ((zlo || zhi) && i < 17) fix_z(i + 1);
    double u[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) u[v] = cpi[v * 400 + col];
    fb |= (unsigned)(f2 == 1) << 4;
    const auto is = [&](int m) { return (int)(fb >> m & 1); };
    double Rx[5], px, pz;   // px, pz: face pressure differences
    {
      const double* cpn = cp[~i & 1];
      double n1[5];
#pragma unroll
      for (int v = 0; v < 5; ++v) n1[v] = cpn[v * 400 + col];
      auto at = [&](int m, int v) {
        return m == 0 ? p2[v] : m == 1 ? p1[v] : m == 2 ? u[v] : m == 3 ? n1[v] : m == 4 ? n2[v] : n3[v];
      };
      const int of = order_fwd(i, is(1), is(3), is(4));
      double L[5], R[5], Ff[5], dPf;
      face_states(of, at, L, R);
      roe_flux<0>(L, R, e, Ff, dPf);
      const int ob = order_bwd(i, is(0), is(1), is(3));
      if (ob != corder) {
        double q3[5];
        if (MODE == IN_PLACE) {
#pragma unroll
          for (int v = 0; v < 5; ++v) q3[v] = p3[v];
        } else {
          column(max(i - 3, 0), q3);
        }
        face_states(ob, [&](int m, int v) { return m == 0 ? q3[v] : at(m - 1, v); }, L, R);
        roe_flux<0>(L, R, e, cF, cdP);
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
    // The cell's time levels arrive while the viscous terms run.
    const size_t row = (size_t)c * CUBE_STRIDE + i * 400;
    const unsigned ob8 = 8u * col;
    auto own = [&](auto* a, int v) -> auto& { return at_byte(a + row + (size_t)v * PLANE, ob8); };
    double tu1[5], tuq[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      tu1[v] = own(A.U1, v);
      tuq[v] = own(A.U1q, v);
    }
    const int8_t* f = fli + col;
    const int IF = f[0];
    double Ry[5], Rz[5];
    {
      double Fb[5], dPu;
      const int ob = order_bwd(j, f[-40], f[-20], f[20]);
      if (j == 2 || ob == order_fwd(j - 1, f[-40], f[0], f[20])) {
#pragma unroll
        for (int v = 0; v < 5; ++v) Fb[v] = fy[v][(j - 2) * 16 + (k - 2)];
      } else {
        double L[5], R[5];
        face_states(ob, [&](int m, int v) { return cpi[v * 400 + col + (m - 3) * 20]; }, L, R);
        roe_flux<1>(L, R, e, Fb, dPu);
      }
#pragma unroll
      for (int v = 0; v < 5; ++v) Ry[v] = fy[v][(j - 1) * 16 + (k - 2)] - Fb[v];
    }
    {
      // The z-face behind comes from the lane behind in the row of 16, the
      // first lane's from LDS.
      double Fb[6];
#pragma unroll
      for (int v = 0; v < 6; ++v) {
        const double x = v < 5 ? zF[v] : dPzf, first = fzb[v][j - 2];
        Fb[v] = __hiloint2double(
            __builtin_amdgcn_update_dpp(__double2hiint(first), __double2hiint(x), 0x111, 0xf, 0xf, false),
            __builtin_amdgcn_update_dpp(__double2loint(first), __double2loint(x), 0x111, 0xf, 0xf, false));
      }
      const int ob = order_bwd(k, f[-2], f[-1], f[1]);
      if (!(k == 2 || ob == order_fwd(k - 1, f[-2], f[0], f[1]))) {
        double L[5], R[5], F[5];
        face_states(ob, [&](int m, int v) { return cpi[v * 400 + col + (m - 3)]; }, L, R);
        roe_flux<2>(L, R, e, F, Fb[5]);
#pragma unroll
        for (int v = 0; v < 5; ++v) Fb[v] = F[v];
      }
#pragma unroll
      for (int v = 0; v < 5; ++v) Rz[v] = zF[v] - Fb[v];
      pz = dPzf - Fb[5];
    }
    double Rf[5];
    if (pow2) {
#pragma unroll
      for (int v = 0; v < 5; ++v) Rf[v] = -(Rx[v] * inv + Ry[v] * inv + Rz[v] * inv);
    } else {
#pragma unroll
      for (int v = 0; v < 5; ++v) Rf[v] = -(div_sh(ddx, Rx[v]) + div_sh(ddx, Ry[v]) + div_sh(ddx, Rz[v]));
    }
    __syncthreads();

    // ---- viscous (Flux.cpp:1722-2279) from the primitive ring ----
    const double rho = u[0];
    auto Q = [&](int a, int bb, int cc, int m) -> double {
      const int s = a < 0 ? sl0 : a == 0 ? sl1 : sl2;
      return pr[m][s * PR_PLANE + (j + bb - 1) * PR_ROW + (k + cc - 1)];
    };
    Prim me;
    const DivBy drho = div_by(rho);
    me.u = Q(0, 0, 0, 0);
    me.v = Q(0, 0, 0, 1);
    me.w = Q(0, 0, 0, 2);
    const double VV = me.u * me.u + me.v * me.v + me.w * me.w;
    const double P = (u[4] - 0.5 * rho * VV) * KM1;
    const double PoR = div_sh(drho, P);   // P / rho
    me.T = dvd(PoR, RG);
    double vF[5] = {0, 0, 0, 0, 0};
    double Lb[5], Lf[5];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
#pragma unroll
      for (int side = -1; side <= 1; side += 2) {
        const int o0 = d == 0 ? side : 0, o1 = d == 1 ? side : 0, o2 = d == 2 ? side : 0;
        Prim f;
        f.u = Q(o0, o1, o2, 0);
        f.v = Q(o0, o1, o2, 1);
        f.w = Q(o0, o1, o2, 2);
        f.T = Q(o0, o1, o2, 3);
        const double Tf = 0.5 * (me.T + f.T);
        const double temp = div_sh(dT0, Tf);
        const double mu = dvd(ph.mu_L * temp * root(temp) * (ph.T0 + 110.), Tf + 110.);
        double g[3][4];
#pragma unroll
        for (int tt = 0; tt < 3; ++tt) {
          if (tt == d) {
            if (side < 0) {
              g[tt][0] = (me.u - f.u) * inv;
              g[tt][1] = (me.v - f.v) * inv;
              g[tt][2] = (me.w - f.w) * inv;
              g[tt][3] = (me.T - f.T) * inv;
            } else {
              g[tt][0] = (f.u - me.u) * inv;
              g[tt][1] = (f.v - me.v) * inv;
              g[tt][2] = (f.w - me.w) * inv;
              g[tt][3] = (f.T - me.T) * inv;
            }
          } else {
            const int p0 = tt == 0, p1 = tt == 1, p2 = tt == 2;
#pragma unroll
            for (int m = 0; m < 4; ++m)
              g[tt][m] = (Q(p0, p1, p2, m) + Q(p0 + o0, p1 + o1, p2 + o2, m) - Q(-p0, -p1, -p2, m) -
                          Q(-p0 + o0, -p1 + o1, -p2 + o2, m)) * inv4;
          }
        }
        const double uf = 0.5 * (me.u + f.u), vf = 0.5 * (me.v + f.v), wf = 0.5 * (me.w + f.w);
        const double div = g[0][0] + g[1][1] + g[2][2];
        double sg[3];
#pragma unroll
        for (int m = 0; m < 3; ++m)
          sg[m] = (m == d) ? mu * (2 * g[d][d] - 2.0 / 3.0 * div) : mu * (g[m][d] + g[d][m]);
        double* L = side < 0 ? Lb : Lf;
        L[1] = sg[0];
        L[2] = sg[1];
        L[3] = sg[2];
        L[4] = uf * sg[0] + vf * sg[1] + wf * sg[2] + dvd(mu * CVG * KG * g[d][3], PRG);
      }
#pragma unroll
      for (int v = 1; v < 5; ++v) {
        const double term = (Lf[v] - Lb[v]) * inv;
        vF[v] = d == 0 ? term : vF[v] + term;
      }
    }

    // ---- residual with the dual-time source, preconditioner, increment ----
    double Rk[5];
    Rk[0] = div_sh(d2t, -(3 * u[0] - 4 * tu1[0] + tuq[0])) + Rf[0];
#pragma unroll
    for (int v = 1; v < 5; ++v) {
      const double Rp = div_sh(d2t, -(3 * u[v] - 4 * tu1[v] + tuq[v]));
      Rk[v] = Rp + Rf[v] + vF[v];
    }
    double out[5] = {0, 0, 0, 0, 0};
    if (IF == 1) {
      const double U_ = me.u, V_ = me.v, W_ = me.w;
      const double C = div_sh(drho, KG * P);
      const double T = PoR;
      const double H = 0.5 * VV + dvd(C, KM1);
      const double beta = rmax(dvd(VV, C), e);
      const double temp = KG * T * (2 * deltaT + 3 * deltaTau) * (2 * deltaT + 3 * beta * deltaTau);
      const double temp2 = KM1 * (beta - 1) * deltaT * deltaT;
      const double temp3 = H - H * KG - VV + KG * (T + VV);
      // The reference's entries; those that differ in sign only (scaling by 4
      // and negation are exact) are formed once.
      const DivBy dT = div_by(temp);
      const double U4 = 4 * U_, V4 = 4 * V_, W4 = 4 * W_, H4 = 4 * H;
      const double d11 = div_sh(dT, (2 * deltaT * (-2 * (-KM1 * (H - VV) - temp3 * beta) * deltaT + 3 * KG * T * beta * deltaTau)));
      const double d15 = div_sh(dT, (4 * temp2));
      const double d25 = div_sh(dT, (U4 * temp2));   // -d12
      const double d35 = div_sh(dT, (V4 * temp2));   // -d13
      const double d45 = div_sh(dT, (W4 * temp2));   // -d14
      out[0] = deltaTau * (d11 * Rk[0] - d25 * Rk[1] - d35 * Rk[2] - d45 * Rk[3] + d15 * Rk[4]);
      const double d21 = div_sh(dT, (U4 * temp3 * (beta - 1) * deltaT * deltaT));
      const double d22 = div_sh(dT, (2 * deltaT * (2 * KG * (T - U_ * U_ * (beta - 1)) * deltaT + 2 * U_ * U_ * (beta - 1) * deltaT + 3 * KG * T * beta * deltaTau)));
      const double m23 = div_sh(dT, (U4 * V_ * temp2));
      const double m24 = div_sh(dT, (U4 * W_ * temp2));
      out[1] = deltaTau * (d21 * Rk[0] + d22 * Rk[1] - m23 * Rk[2] - m24 * Rk[3] + d25 * Rk[4]);
      const double d31 = div_sh(dT, (V4 * temp3 * (beta - 1) * deltaT * deltaT));
      const double d33 = div_sh(dT, (2 * deltaT * (2 * KG * (T - V_ * V_ * (beta - 1)) * deltaT + 2 * V_ * V_ * (beta - 1) * deltaT + 3 * KG * T * beta * deltaTau)));
      const double m34 = div_sh(dT, (V4 * W_ * temp2));
      out[2] = deltaTau * (d31 * Rk[0] - m23 * Rk[1] + d33 * Rk[2] - m34 * Rk[3] + d35 * Rk[4]);
      const double d41 = div_sh(dT, (W4 * temp3 * (beta - 1) * deltaT * deltaT));
      const double d44 = div_sh(dT, (2 * deltaT * (2 * KG * (T - W_ * W_ * (beta - 1)) * deltaT + 2 * W_ * W_ * (beta - 1) * deltaT + 3 * KG * T * beta * deltaTau)));
      out[3] = deltaTau * (d41 * Rk[0] - m24 * Rk[1] - m34 * Rk[2] + d44 * Rk[3] + d45 * Rk[4]);
      const double d51 = div_sh(dT, (H4 * temp3 * (beta - 1) * deltaT * deltaT));
      const double m52 = div_sh(dT, (H4 * U_ * temp2));
      const double m53 = div_sh(dT, (H4 * V_ * temp2));
      const double m54 = div_sh(dT, (H4 * W_ * temp2));
      const double d55 = div_sh(dT, (2 * deltaT * (2 * H * KM1 * (beta - 1) * deltaT + KG * T * (2 * deltaT + 3 * beta * deltaTau))));
      out[4] = deltaTau * (d51 * Rk[0] - m52 * Rk[1] - m53 * Rk[2] - m54 * Rk[3] + d55 * Rk[4]);
    }
    if (AUX && A.rku) {
#pragma unroll
      for (int v = 0; v < 5; ++v) own(A.Rku, v) = out[v];
    }
    double pn[8] = {0, 0, 0, 0, 0, 0, 0, 0};   // the cell's norm and force terms
    if (IF < 1) {
      const double fx = pow2 ? -px * inv : div_sh(ddx, -px);
      const double fz = pow2 ? -pz * inv : div_sh(ddx, -pz);
      pn[5] = -(fx + vF[1]) * dx * dx * dx;
      pn[6] = -(fz + vF[3]) * dx * dx * dx;
      if (AUX && A.rku) {
        own(A.Res, 0) = pn[5];
        own(A.Res, 1) = pn[6];
      }
    }
    if (MODE != FLUX_ONLY) {
      double nv[5];
#pragma unroll
      for (int v = 0; v < 5; ++v) nv[v] = u[v];
      if (IF == 1) {
        if (RK == 1) {
#pragma unroll
          for (int v = 0; v < 5; ++v) nv[v] = u[v] + out[v];
        } else if (RK == 2) {
#pragma unroll
          for (int v = 0; v < 5; ++v) {
            const double m = MODE == PUSH ? u[v] : own(A.U1p1, v);
            nv[v] = 0.75 * u[v] + 0.25 * m + 0.25 * out[v];
          }
        } else {
#pragma unroll
          for (int v = 0; v < 5; ++v) {
            const double m = MODE == PUSH ? u[v] : own(A.U1p2, v);
            nv[v] = 1.0 / 3.0 * u[v] + 2.0 / 3.0 * m + 2.0 / 3.0 * out[v];
          }
          const double r = nv[0];
          const DivBy dn = div_by(r);
          const double un = div_sh(dn, nv[1]), vn = div_sh(dn, nv[2]), wn = div_sh(dn, nv[3]);
          const double Pn = (nv[4] - 0.5 * r * (un * un + vn * vn + wn * wn)) * KM1;
          const double dTn = div_sh(dn, Pn) - PoR;
          pn[0] = (Pn - P) * (Pn - P);
          pn[1] = (un - me.u) * (un - me.u);
          pn[2] = (vn - me.v) * (vn - me.v);
          pn[3] = (wn - me.w) * (wn - me.w);
          pn[4] = dTn * dTn;
        }
        if (AUX && RK < 3) {
          double* m = RK == 1 ? A.U1p1 : A.U1p2;
#pragma unroll
          for (int v = 0; v < 5; ++v) own(m, v) = nv[v];
        }
      }
      if (MODE == IN_PLACE) {
        if (IF == 1) {
#pragma unroll
          for (int v = 0; v < 5; ++v) own(A.U, v) = nv[v];
        }
      } else {
        const int nx = i <= 3 ? hs.src[0] : (i >= 16 ? hs.src[1] : 0);
        const int ny = j <= 3 ? hs.src[2] : (j >= 16 ? hs.src[3] : 0);
        const int nz = k <= 3 ? hs.src[4] : (k >= 16 ? hs.src[5] : 0);
        const int o = i * 400 + col;
        const int oy = o + (j <= 3 ? 16 * 20 : -16 * 20);
        const int oz = o + (k <= 3 ? 16 : -16);
        const size_t rx = (size_t)nx * CUBE_STRIDE + (i <= 3 ? i + 16 : i - 16) * 400;
#pragma unroll
        for (int v = 0; v < 5; ++v) {
          own(A.Uout, v) = nv[v];
          if (nx > 0) at_byte(A.Uout + rx + (size_t)v * PLANE, ob8) = nv[v];
        }
        if (ny > 0) {
          double* O = A.Uout + (size_t)ny * CUBE_STRIDE + oy;
#pragma unroll
          for (int v = 0; v < 5; ++v) O[v * PLANE] = nv[v];
        }
        if (nz > 0) {
          double* O = A.Uout + (size_t)nz * CUBE_STRIDE + oz;
#pragma unroll
          for (int v = 0; v < 5; ++v) O[v * PLANE] = nv[v];
        }
      }
      if (RK == 3) {
        const double s = wave_sum8(pn);
        if ((t & 7) == 0) red[t >> 6][(t >> 3) & 7] = s;
      }
    }
    // ---- advance the column, the flags and the ring ----
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      if (MODE == IN_PLACE) p3[v] = p2[v];
      p2[v] = p1[v];
      p1[v] = u[v];
      n2[v] = n3[v];
    }
    fb >>= 1;
    const int s = sl0;
    sl0 = sl1;
    sl1 = sl2;
    sl2 = s;
  }
  if (MODE != FLUX_ONLY && RK == 3) {
    __syncthreads();
    if (t < 8) {
      const double s = plane_row();
      const size_t row = (size_t)(c - 1) * (MODE == IN_PLACE ? 1 : PUSH_ROWS_PER_CUBE);
      if (single)
        A.partials[row * 8 + t] = tot[t] + s;
      else
        A.partials[(row + i1 - 2) * 8 + t] = s;
    }
  }
}

}  // namespace

void launch_flux_march(hipStream_t s, double* U, const double* U1, const double* U1q,
                       const int8_t* fws, const double* cube_size, double* Rku, double* Res,
                       int ncube, PhysTab pt, double deltaT, double deltaTau, double e, int nseg) {
  if (ncube <= 1) return;
  const MarchArgs a{U, U1, U1q, fws, cube_size, Rku, Res, pt, deltaT, deltaTau, e, Runs{0, nseg}, 1,
                    ncube, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, {}, true};
  hipLaunchKernelGGL((k_flux_march<FLUX_ONLY, true>), run_grid(a.runs, ncube), dim3(WG), 0, s, a);
}

int launch_flux_in_place(hipStream_t s, double* U, const double* U1, const double* U1q,
                         const int8_t* fws, const double* cube_size, double* Rku, double* Res,
                         int ncube, PhysTab pt, double deltaT, double deltaTau, double e, int RK,
                         double* U1p1, double* U1p2, double* partials) {
  const int n = ncube - 1;
  if (n <= IN_PLACE_SPLIT) {
    launch_flux_march(s, U, U1, U1q, fws, cube_size, Rku, Res, ncube, pt, deltaT, deltaTau, e,
                      push_runs(n));
    launch_update(s, RK, U, U1p1, U1p2, Rku, Res, fws, ncube, pt.cube_case, partials,
                  true);
    return PUSH_ROWS_PER_CUBE;
  }
  const MarchArgs a{U, U1, U1q, fws, cube_size, Rku, Res, pt, deltaT, deltaTau, e, Runs{0, 1}, RK,
                    ncube, U1p1, U1p2, partials, nullptr, nullptr, nullptr, {}, true};
  hipLaunchKernelGGL((k_flux_march<IN_PLACE, true>), run_grid(a.runs, ncube), dim3(WG), 0, s, a);
  return 1;
}

int launch_flux_push(hipStream_t s, double* Uin, double* Uout, const HaloSrc* halo,
                      const uint8_t* cube_mask, const double* U1, const double* U1q,
                      const int8_t* fws, const double* cube_size, double* Rku, double* Res,
                      int ncube, PhysTab pt, double deltaT, double deltaTau, double e, int RK,
                      double* U1p1, double* U1p2, double* partials, PushAux aux, IbRefresh ib,
                      int nseg) {
  if (ncube <= 1) return 0;
  const MarchArgs a{Uin, U1, U1q, fws, cube_size, Rku, Res, pt, deltaT, deltaTau, e,
                    runs_for(ncube, nseg), RK, ncube, U1p1, U1p2, partials, Uout, halo, cube_mask,
                    ib, aux == PushAux::ALL || RK == 3};
  if (aux != PushAux::NONE)
    hipLaunchKernelGGL((k_flux_march<PUSH, true>), run_grid(a.runs, ncube), dim3(WG), 0, s, a);
  else
    hipLaunchKernelGGL((k_flux_march<PUSH, false>), run_grid(a.runs, ncube), dim3(WG), 0, s, a);
  return single_rows(a.runs, ncube);
}

// Runs per cube of the pushing kernel.  The chip holds 512 of its workgroups
// (two per CU), and a run costs one x-face pass and two primitive planes more,
// about two thirds of a plane.  The most runs that fit at once to 64 cubes (8
// cubes: 19 us in 16 runs, 161 in one; 64: 43 in 8, 45 in 16); a plane per run to
// 90, where 8 runs would leave a second, nearly empty wave (80: 54, 59 in 8);
// again what fits at once to 128 (100: 68 in 4, 69 in 16; 128: 73, 99 in 2); then
// the last wave's share against the prologues: 8 runs to 240 (216: 117, 127 in
// 4), 4 to 370 (294: 158, 166 in 8, 185 in 2), 2 to 560 (384: 193, 197 in 4; 512:
// 256, 262 in 4), above one run with quartered last cubes (runs_for; 576: 284,
// 299 in 2; 1,000: 479, 487 in one without them).
int push_runs(int n) {
  return n <= 48 ? 16 : n <= 64 ? 8 : n <= 90 ? 16 : n <= 128 ? 4 : n <= 240 ? 8 : n <= 370 ? 4
       : n <= 560 ? 2 : 1;
}

}  // namespace bcm
