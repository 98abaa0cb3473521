// Device data layout and kernel launch interface of the BCM engine.
//
// State arrays live in HBM as structure-of-arrays per cube:
//   [cube][var][i][j][k], 20^3 doubles per (cube, var) plane, k fastest.
// A wavefront of 64 lanes covers four 16-cell k-rows of one i-plane, so every
// stencil load is a coalesced row segment.  Flags are int8 [cube][i][j][k].
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

namespace bcm {

constexpr int PLANE = 8000;               // 20^3 cells of one variable of one cube
constexpr int CUBE_STRIDE = 5 * PLANE;    // doubles per cube in a state array

struct DevPhys {
  double rho0, U0, Uin, V0, W0, P0, T0, mu_L;
};

// Freestream conserved state of a case: (rho0, rho0 Uin, rho0 V0, rho0 W0,
// P0/(K-1) + rho0 |V|^2 / 2).  The mixed-precision path stores the inner
// iterate as its FP32 deviation from this state.
__host__ __device__ inline void ref_state(const DevPhys& ph, double (&u)[5]) {
  u[0] = ph.rho0;
  u[1] = ph.rho0 * ph.Uin;
  u[2] = ph.rho0 * ph.V0;
  u[3] = ph.rho0 * ph.W0;
  u[4] = ph.P0 / (1.4 - 1) + 0.5 * ph.rho0 * (ph.Uin * ph.Uin + ph.V0 * ph.V0 + ph.W0 * ph.W0);
}

// Edge ghost cells (layer-1/18 lines where two ghost layers meet).  The edge
// passes of an exchange (Interface.cpp:5640-5732) set each edge cell a flux
// kernel reads to the mean of two face ghost cells of the same cube: the
// corners (j, k in {1, 18}) of interior planes i = 2..17 (i-edges), and in
// the ghost planes i = 1, 18 the border cells with one of j, k in {1, 18}
// (k-edges along j = 1, 18, j-edges along k = 1, 18).  For a cell (i, j, k)
// with i, j, k in 1..18 this returns true and the two source cells (flat
// i*400 + j*20 + k) when the cell is one of those; cube corners, which no
// flux stencil reads, and all other cells return false.
__host__ __device__ inline bool edge_sources(int i, int j, int k, int& a, int& b) {
  const bool ej = j == 1 || j == 18, ek = k == 1 || k == 18;
  const int in = i == 1 ? 2 : 17, jn = j == 1 ? 2 : 17, kn = k == 1 ? 2 : 17;
  if (i != 1 && i != 18) {
    if (!(ej && ek)) return false;
    a = i * 400 + j * 20 + kn;
    b = i * 400 + jn * 20 + k;
  } else if (ej && !ek) {
    a = i * 400 + jn * 20 + k;
    b = in * 400 + j * 20 + k;
  } else if (ek && !ej) {
    a = i * 400 + j * 20 + kn;
    b = in * 400 + j * 20 + k;
  } else {
    return false;
  }
  return true;
}

// A cell where two or three ghost layers meet (edge or corner of the padded
// cube).
__host__ __device__ inline bool edge_cell(int i, int j, int k) {
  const int g = (i < 2 || i > 17) + (j < 2 || j > 17) + (k < 2 || k > 17);
  return g >= 2;
}

// Physics of every cube of a pool that holds several independent cases:
// phys[cube_case[c]] is the case constants of cube c; cube_case[c] < 0 marks
// a cube that belongs to no case (kernels skip it).
struct PhysTab {
  const DevPhys* phys;
  const int* cube_case;
};

// One resident case in the per-case norm reduction: cubes [first, first+n)
// of the pool, norm scaling cube count mpi_ncube, norm slot and physics index.
struct CaseDesc {
  int first, n, mpi_ncube, slot;
};

// One IB ghost-fill entry in level order (see the ghost schedule in the engine).
// Where the ghost cell itself is a corner its weights and slots come with that
// corner last, the others in their order: the interpolation without it is then
// the sum of the first seven.
struct alignas(16) GhostEntry {
  double w[8];
  int16_t lc[8], lg;                // LDS slots read for the corners and written
  int16_t self;                     // corner that is the ghost cell itself (8: none)
  int cube;
  int16_t gi, gj, gk, pi, pj, pk;   // ghost cell and interpolation base corner
};

// IB fill of one cube in LDS: two value slots per entry (primitives for later
// levels, conserved values for memory) and one per cell that an entry reads
// before any entry has written it; a cube needing more slots works on memory.
// 3072 slots of five doubles are 120 KB of the 160 KB of a CU; a whole body
// inside one cube needs about 1000 to 2100.
constexpr int GHOST_LDS_SLOTS = 3072;
// Largest limit the diagnostic hook accepts; it stands for no limit but the
// kernel's (a caller that lowered the limit takes that back with it).
constexpr int GHOST_LDS_HOOK_MAX = 1536;

// IB fill of one cube: its levels, entries and the cells it reads.
struct GhostCube {
  int cube;
  int lev0, nlev;     // levels lev0 .. lev0+nlev-1 (nlev 0: no fill)
  int ent0, n1, ne;   // first entry, entries of the first level, all entries
  int read0, nread;   // staged cells; nread -1: the fill works on memory
};

// Device tables of the IB fill: entries grouped per cube and level.  In LDS
// every entry writes a slot of its own (its index within the cube) and reads
// the slots of the values the sequential fill would read, so levels follow
// read-after-write dependencies only; the cells it reads as memory holds them
// are staged in the slots after the entries'.  On memory the fill is in place
// and levels also order writes after earlier reads and writes of a cell.
struct GhostTables {
  const GhostEntry* ent = nullptr;
  const GhostCube* cubes = nullptr;
  const int* level_off = nullptr;   // per level: first entry (+1 sentinel)
  const int16_t* read = nullptr;    // staged cells i*400 + j*20 + k
  const int16_t* out = nullptr;     // per LDS slot of an entry: its ghost cell
                                    // (-1: a later entry writes the cell)
  int ncubes = 0;
  int max_slots = 0;
};

// One cube's work at the opening of a stage: edge ghost cells edge0 ..
// edge0 + nedge - 1 of the list, its BCs (mask) and its IB fill.
struct OpenItem {
  int edge0, nedge, mask, slot;
  GhostCube g;
};

// Source cubes for the six face halos of a cube (0 = no equal-size neighbour).
struct HaloSrc {
  int src[6];   // -X, +X, -Y, +Y, -Z, +Z
};

// One ghost region of a face across a change of cube size (two-level grid):
// dst's two ghost layers on side hi (1 upper, 0 lower) of axis `axis` from
// the neighbour src.  restrict_ 0: dst is the small cube, each ghost cell
// copies the big cube's face cell above it (BCM_Interface.cpp:1790-2021 for
// x); restrict_ 1: dst is the big cube, the 2 x 8 x 8 ghost cells of quadrant
// `slot` (1..4) take 0.125 times the sum of the 8 small cells beneath, in the
// reference's order (:2026-2600 for x; y and z alike).
struct MlTaskDev {
  int dst, src;
  int8_t axis, hi, restrict_, slot;
};

// Boundary-cube mask bit (shifted left by 1 for z-max) marking a z-BC face
// whose BC the pushing flux kernels apply to the interior planes i = 2..17
// themselves (BCM_Z_boundary_condition.cpp:47-88 reads only the plane's cell
// k = 2, or 17, which nothing changes between a stage's BCs and its flux on
// such cubes); the stage opening then does only the ghost planes.
constexpr int ZBC_IN_FLUX = 64;

// The z-min BC's w-momentum, -x, in storage form: FP64 stores the state, FP32
// its deviation from the case's reference state (r3 = rho0 W0).
__device__ inline double zbc_neg(double x, double) { return -x; }
__device__ inline float zbc_neg(float x, double r3) { return (float)(-((double)x + r3) - r3); }

// How a marching flux kernel divides cubes 1..n among workgroups: cubes 1..whole
// (a multiple of 8) take one each, every other cube nseg runs of 16/nseg planes.
struct Runs {
  int whole, nseg;
};
struct RunOf {
  int cube, seg, nseg;
};
// Workgroups go to the 8 XCDs in turn; the runs of one cube share planes and so
// go to one XCD's L2.
__device__ inline RunOf run_of(const Runs& r, int block) {
  if (block < r.whole) return RunOf{block + 1, 0, 1};
  const int b = block - r.whole;
  return RunOf{r.whole + b / (8 * r.nseg) * 8 + b % 8 + 1, b / 8 % r.nseg, r.nseg};
}
// Whole groups of one cube per XCD.
inline dim3 run_grid(const Runs& r, int ncube) {
  return dim3(r.whole + (ncube - 1 - r.whole + 7) / 8 * 8 * r.nseg);
}
// nseg runs per cube; with one run, the last 192 of more than 560 cubes take
// four.  Workgroups of one CU fall out of step, and with whole cubes only the
// last half cube's time finds half the slots empty; quarters fill them (FP64
// 2,048 cubes 958 -> 947 us, 1,584: 779 -> 742, 800: 448 -> 386, 576: 362 -> 285;
// mixed 519 -> 492, 435 -> 396, 245 -> 220, 206 -> 154).  128 to 256 cubes are alike;
// 512 cost more prologues than they save.
inline Runs runs_for(int ncube, int nseg) {
  const int n = ncube - 1;
  return nseg == 1 && n > 560 ? Runs{(n - 192) & ~7, 4} : Runs{0, nseg};
}

// Leading cubes of the pool that one workgroup marches whole: it sums their
// planes' norm rows into one.
inline int single_rows(const Runs& r, int ncube) { return r.nseg == 1 ? ncube - 1 : r.whole; }

// Copies, with the threads of one workgroup, the ghost regions the domain BCs
// of cube c write (mask bits 1 x-min, 2 x-max, 4 y-min, 8 y-max, 16 z-min,
// 32 z-max) from Uin to Uout: x faces over j,k in [2,17], y faces over all i
// and k in [2,17], z faces over all i,j.  The regions are disjoint and no
// neighbour writes them.
template <typename T>
__device__ inline void copy_bc_regions(const T* __restrict__ Uin, T* __restrict__ Uout, int c,
                                       int m, double r3) {
  const size_t base = (size_t)c * CUBE_STRIDE;
  auto cp = [&](int cell) {
#pragma unroll
    for (int v = 0; v < 5; ++v) Uout[base + (size_t)v * PLANE + cell] = Uin[base + (size_t)v * PLANE + cell];
  };
  for (int side = 0; side < 2; ++side) {
    const int off = side ? 18 : 0;
    if (m & (1 << side))
      for (int n = threadIdx.x; n < 512; n += blockDim.x)
        cp((off + n / 256) * 400 + ((n % 256) / 16 + 2) * 20 + (n % 16 + 2));
    if (m & (4 << side))
      for (int n = threadIdx.x; n < 640; n += blockDim.x)
        cp(((n % 320) / 16) * 400 + (off + n / 320) * 20 + (n % 16 + 2));
    if (m & (16 << side)) {
      // Planes whose z-BC this stage's flux kernel applied (ZBC_IN_FLUX):
      // the BC values, from the plane's cell k = 2 (or 17).
      const bool influx = m & (ZBC_IN_FLUX << side);
      for (int n = threadIdx.x; n < 800; n += blockDim.x) {
        const int i = (n % 400) / 20, cell = i * 400 + ((n % 400) % 20) * 20 + off + n / 400;
        if (influx && i >= 2 && i <= 17) {
          const int src = cell - (off + n / 400) + (side ? 17 : 2);
#pragma unroll
          for (int v = 0; v < 5; ++v) {
            const T x = Uin[base + (size_t)v * PLANE + src];
            Uout[base + (size_t)v * PLANE + cell] = (v == 3 && !side) ? zbc_neg(x, r3) : x;
          }
        } else {
          cp(cell);
        }
      }
    }
  }
}

// IB ghost cells that lie in the source layers of a neighbour, which the
// pre-flux exchange refreshes in its face layers: cell pairs sorted by
// destination cube, (source, destination) flat cells, cube * 8000 + cell, those
// of cube c at off[c] .. off[c + 1] - 1.
struct IbRefresh {
  const int2* pairs = nullptr;
  const int* off = nullptr;
};
// The refresh of cube c by a workgroup of the pushing flux kernel, before its
// first read of the cube: in a launch of its own it took 5 us per stage, a
// tenth of a stage on 8 cubes.  Sources are interior cells, which that kernel
// writes in the other copy only; the runs of a cube store the same values.
template <typename T>
__device__ inline void refresh_cube(T* __restrict__ U, const IbRefresh& r, int c) {
  const int q0 = r.off[c], q1 = r.off[c + 1];
  if (q0 == q1) return;
  for (int q = q0 + threadIdx.x; q < q1; q += blockDim.x) {
    const int2 pr = r.pairs[q];
    const size_t so = (size_t)(pr.x / PLANE) * CUBE_STRIDE + pr.x % PLANE;
    const size_t dd = (size_t)(pr.y / PLANE) * CUBE_STRIDE + pr.y % PLANE;
    T x[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) x[v] = U[so + (size_t)v * PLANE];
#pragma unroll
    for (int v = 0; v < 5; ++v) U[dd + (size_t)v * PLANE] = x[v];
  }
  __syncthreads();
}

// Sums eight doubles over the 64 lanes of a wave in a fixed order; every lane
// returns the total of x[lane >> 3].  Halving the values kept at each exchange
// (lane halves, rows of 16, halves of a row) takes 10 additions where eight
// separate wave sums would take 48.
__device__ inline double wave_sum8(double (&x)[8]) {
  auto both = [](double a, double b, auto swap) {
    const auto lo = swap((unsigned)__double2loint(a), (unsigned)__double2loint(b));
    const auto hi = swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b));
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
  };
  auto half = [](unsigned a, unsigned b) { return __builtin_amdgcn_permlane32_swap(a, b, false, false); };
  auto row = [](unsigned a, unsigned b) { return __builtin_amdgcn_permlane16_swap(a, b, false, false); };
#pragma unroll
  for (int m = 0; m < 4; ++m) x[m] = both(x[m], x[m + 4], half);
#pragma unroll
  for (int m = 0; m < 2; ++m) x[m] = both(x[m], x[m + 2], row);
  auto moved = [](double v, auto ctrl) {
    constexpr int c = decltype(ctrl)::value;
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), c, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), c, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
  };
  const bool up = threadIdx.x & 8;
  double s = up ? x[1] : x[0];
  s += moved(up ? x[0] : x[1], std::integral_constant<int, 0x128>());   // row_ror 8
  s += moved(s, std::integral_constant<int, 0x141>());                  // row_half_mirror
  s += moved(s, std::integral_constant<int, 0xB1>());                   // quad_perm 1,0,3,2
  s += moved(s, std::integral_constant<int, 0x4E>());                   // quad_perm 2,3,0,1
  return s;
}

// Launches cover pool cubes 1..ncube-1; "ncube" is one past the last cube in use.
// The BC, IB fill and halo kernels exist for an FP64 inner iterate and for the
// FP32 one of the mixed-precision path, which holds the deviation from the
// case's freestream state (ref_state); arithmetic is FP64 on full states
// either way, copies move stored values as they are.
void launch_bc(hipStream_t s, double* U, const int* cubes, const uint8_t* masks, int n,
               PhysTab pt);
void launch_bc(hipStream_t s, float* U, const int* cubes, const uint8_t* masks, int n,
               PhysTab pt);
void launch_ghost(hipStream_t s, double* U, const GhostTables& g, PhysTab pt);
void launch_ghost(hipStream_t s, float* U, const GhostTables& g, PhysTab pt);
void launch_halo_edge(hipStream_t s, double* U, const HaloSrc* src, int ncube, const int* cube_case);
void launch_halo_edge(hipStream_t s, float* U, const HaloSrc* src, int ncube, const int* cube_case);
// Pre-flux refresh: copy (source, destination) cell pairs (cube*8000 + cell).
void launch_halo_pairs(hipStream_t s, double* U, const int2* pairs, int npairs);
void launch_halo_pairs(hipStream_t s, float* U, const int2* pairs, int npairs);
// Edge passes of the listed cubes.
void launch_edge_list(hipStream_t s, double* U, const int* list, int n);
void launch_edge_list(hipStream_t s, float* U, const int* list, int n);
// Opening of a stage after a flux kernel that wrote the face halos itself, in one
// launch: per item the listed edge cells and the domain BCs, then the IB fill.
// `before` holds the ghost regions the previous stage's BCs wrote: the other copy
// of the iterate, or U where they were carried over.
void launch_open(hipStream_t s, double* U, const double* before, const OpenItem* items, int n,
                 const int16_t* edges, const GhostTables& g, const DevPhys* phys);
void launch_open(hipStream_t s, float* U, const float* before, const OpenItem* items, int n,
                 const int16_t* edges, const GhostTables& g, const DevPhys* phys);
// Ghost regions the BCs wrote of the listed cubes, from Uin to Uout.
void launch_carry_bc(hipStream_t s, const double* Uin, double* Uout, const int* cubes, int n,
                     const uint8_t* cube_mask, PhysTab pt);
void launch_carry_bc(hipStream_t s, const float* Uin, float* Uout, const int* cubes, int n,
                     const uint8_t* cube_mask, PhysTab pt);
// Edge passes of every cube.
void launch_edge(hipStream_t s, double* U, int ncube, const int* cube_case);
void launch_edge(hipStream_t s, float* U, int ncube, const int* cube_case);
// Two-level faces: one workgroup per task.
void launch_halo_ml(hipStream_t s, double* U, const MlTaskDev* tasks, int ntask, PhysTab pt);
void launch_halo_ml(hipStream_t s, float* U, const MlTaskDev* tasks, int ntask, PhysTab pt);
void launch_flux(hipStream_t s, const double* U, const double* U1, const double* U1q,
                 const int8_t* fws, const double* cube_size, double* Rku, double* Res,
                 int ncube, PhysTab pt, double deltaT, double deltaTau, double e);
// Marching variant of the flux kernel: one workgroup per cube segment
// (nseg in {1, 2, 4, 8, 16} segments of the cube's 16 i-planes).
void launch_flux_march(hipStream_t s, double* U, const double* U1, const double* U1q,
                       const int8_t* fws, const double* cube_size, double* Rku, double* Res,
                       int ncube, PhysTab pt, double deltaT, double deltaTau, double e, int nseg);
// Flux and RK update of one stage in place, writing Rku, Res, U1p1 (RK1) and
// U1p2 (RK2).  Returns the rows of 8 norm partials per cube that RK 3 writes: 1
// from the marching kernel that updates as it goes (one run per cube, since a
// run would read planes another has updated); 16 to IN_PLACE_SPLIT cubes, where
// the flux runs in many runs and the update follows as a kernel of its own.  The
// norms are bitwise the same either way (and those of launch_flux_push).  A
// stage on 8 cubes takes 20 us split and 163 in one kernel, on 125 cubes 95 and
// 193, on 294 200 and 258, on 512 340 and 300.
int launch_flux_in_place(hipStream_t s, double* U, const double* U1, const double* U1q,
                         const int8_t* fws, const double* cube_size, double* Rku, double* Res,
                         int ncube, PhysTab pt, double deltaT, double deltaTau, double e, int RK,
                         double* U1p1, double* U1p2, double* partials);
constexpr int IN_PLACE_SPLIT = 320;
// Marching kernel with the update written to Uout, nseg (1, 2, 4, 8 or 16) runs
// of 16/nseg planes per cube, one workgroup each, bitwise the same results for
// every nseg: every interior cell, and the two layers next to each face with an
// equal-size neighbour (halo[c]) into that neighbour's ghost layers in Uout.
// With PushAux::ALL it writes Rku, Res, U1p1 (RK1) and U1p2 (RK2) bitwise as the
// in-place fused kernel does (nothing reads them back during stages), with
// STEP_END Rku and Res at RK 3 only, with NONE none of them.  At RK 3 one row
// of 8 norm partials per plane, PUSH_ROWS_PER_CUBE to a cube; the leading cubes
// marched whole, whose number it returns, have their sum in the first.
// Ghost regions the domain BCs wrote (cube_mask) stay in Uin (launch_carry_bc).
constexpr int PUSH_ROWS_PER_CUBE = 16;
enum class PushAux { NONE, STEP_END, ALL };
int launch_flux_push(hipStream_t s, double* Uin, double* Uout, const HaloSrc* halo,
                      const uint8_t* cube_mask, const double* U1, const double* U1q,
                      const int8_t* fws, const double* cube_size, double* Rku, double* Res,
                      int ncube, PhysTab pt, double deltaT, double deltaTau, double e, int RK,
                      double* U1p1, double* U1p2, double* partials, PushAux aux, IbRefresh ib,
                      int nseg);
// Runs per cube of the pushing FP64 kernel for n resident cubes.
int push_runs(int n);
void launch_copy_d(hipStream_t s, const double* src, double* dst, size_t n);
// Runs n threads of the shared-denominator division against a / b (four
// quotients each); *mismatches receives the count of differing bit patterns.
// Returns nonzero on a HIP error.
int div_selftest(unsigned long long seed, int n, unsigned long long* mismatches);
void launch_update(hipStream_t s, int RK, double* U, double* U1p1, double* U1p2,
                   const double* Rku, const double* Res, const int8_t* fws, int ncube,
                   const int* cube_case, double* partials, bool body_only = false);
// Norms er[0..7] of each case in cases[0..ncases) from partial rows, stride per
// cube (1 or 16), of which the pool's first `single` cubes use one; case d
// writes er[d.slot*8 .. d.slot*8+7].
void launch_reduce(hipStream_t s, const double* partials, int stride, int single,
                   const CaseDesc* cases, int ncases, const DevPhys* phys, double* er);
void launch_shift(hipStream_t s, const double* U, double* U1, double* U1q, int ncube,
                  const int* cube_case);
// AoS <-> SoA transposes of ncube whole cubes (cube 0 of both arrays included).
void launch_aos_to_soa(hipStream_t s, const double* aos, double* soa, int ncube);
void launch_soa_to_aos(hipStream_t s, const double* soa, double* aos, int ncube);
int update_blocks(int ncube);

// ---- Mixed-precision path (bcm_kernels_mixed.hip) ----
// Inner iterate U in FP32 SoA as the deviation from ref_state of the cube's
// case; U1, U1q (physical time levels) in FP64 as full states; Bsrc, the
// dual-time source constant 3 Uref - 4 U1 + U1q of every interior cell (FP64),
// which the stages read in place of U1 and U1q.
// One workgroup per cube: flux, residual, preconditioned increment and the RK
// update of stage RK, reading Uin and writing every interior cell to Uout
// (updated fluid cells, other cells unchanged).  Cells of the two layers
// next to a face with an equal-size neighbour (halo[c]) are also written into
// that neighbour's ghost layers in Uout: the face part of the post-update
// exchange.  nseg (1, 2, 4, 8 or 16) runs of 16/nseg planes per cube, one
// workgroup each; results are bitwise the same for every nseg.  Norm rows at
// RK 3, and the return value, as launch_flux_push has them.
constexpr int MIXED_ROWS_PER_CUBE = 16;
int launch_flux_mixed(hipStream_t s, float* Uin, float* Uout, const HaloSrc* halo,
                       const uint8_t* cube_mask, const double* Bsrc, const int8_t* fws,
                       const double* cube_size, int ncube, PhysTab pt, double deltaT,
                       double deltaTau, double e, int RK, double* partials, IbRefresh ib, int nseg);
// Runs per cube for n resident cubes.
int mixed_runs(int n);
// dst[0..n) <- src[0..n).
void launch_copy_f(hipStream_t s, const float* src, float* dst, size_t n);
// U1q <- U1, U1 <- ref_state + U and Bsrc <- 3 ref_state - 4 U1 + U1q on
// interior cells.
void launch_shift_mixed(hipStream_t s, const float* U, double* U1, double* U1q, double* Bsrc,
                        int ncube, PhysTab pt);
// Bsrc <- 3 ref_state - 4 U1 + U1q on the interior cells of cubes
// first..first+n-1 (after U1 or U1q were set from outside).
void launch_bsrc_mixed(hipStream_t s, const double* U1, const double* U1q, double* Bsrc, int first,
                       int n, PhysTab pt);
// FP64 AoS full states <-> FP32 SoA deviations from the reference state ref
// (5 doubles) of ncube whole cubes of one case.
void launch_aos_to_soa_f(hipStream_t s, const double* aos, float* soa, int ncube,
                         const double* ref5);
void launch_soa_to_aos_f(hipStream_t s, const float* soa, double* aos, int ncube,
                         const double* ref5);

}  // namespace bcm
