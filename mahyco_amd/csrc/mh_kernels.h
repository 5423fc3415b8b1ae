// mh_kernels.h -- gfx950 kernels of the Lagrange + ADI remap cycle (FP64 on the vector ALUs).
//
// Per cycle (Mahyco.config:23-36):
//   k_node_lag      SaveValuesAtN (nodes) + UpdateVelocity + ApplyBoundaryCondition +
//                   UpdatePosition (nodes): node-centric force gather in cell order
//   k_cell_lag      UpdatePosition (cells) + ComputeGeometricValues + UpdateDensity +
//                   ComputeArtificialViscosity + UpdateEnergyAndPressure, then the remap
//                   vector U (PrepareRemap.cc:94-193) or, without remap, EOS + mean pressure
//                   and the CFL candidate
//   k_sweep_cell    one ADI direction, cell part (RemapADIService.cc:119-575)
//   k_sweep_node    the same direction, dual part (DualPhaseRemap.cc:38-258)
//   k_finalize      remapVariables (RemapADIFinal.cc:21-316) + applyEOS + computePressionMoyenne
//                   + the CFL candidate of computeDeltaT
//   k_dt            computeDeltaT reduction and time-step rules (MahycoModule.cc:1739-1864)
//
// Every value is produced by one thread with the reference's operation order, so the
// results do not depend on launch shape or scheduling.
#ifndef MH_KERNELS_H
#define MH_KERNELS_H

#include <hip/hip_runtime.h>

#include <type_traits>

#include "mh_geom.h"
#include "mh_state.h"

#define MH_BLOCK 256
#define MH_FIRST_BLOCKS 256  // one block on each CU (late_halted)
#define MH_DT_BLOCK 1024

__device__ __forceinline__ bool mh_halted(const MhScalars* sc) { return sc->status != 0 || sc->stopped != 0; }
// An iteration after the end is a no-op.  The first blocks of a launch read the stop flag together with
// what they work on (a wait less for a small mesh), the later ones, whose wait is hidden, ahead of it, so
// that the iterations queued beyond a run's end read next to nothing: 256x128x128 335 -> 45 us, 97x61x83
// 73 -> 29, 512x512 33 -> 19 (with 1024 first blocks 70, 47, 32), running ones as before.
__device__ __forceinline__ bool late_halted(const MhScalars* sc) {
  return blockIdx.x >= MH_FIRST_BLOCKS && mh_halted(sc);
}

// Blocks are dispatched round-robin over the 8 XCDs, each with its own L2.  Single-mesh
// grids are a multiple of 8 blocks and block b works on block (b % 8) * (grid / 8) + b / 8,
// so each XCD sweeps one contiguous slab and the neighbours of a stencil stay in its L2.
__device__ __forceinline__ int xcd_block(int b, int nb) { return (b & 7) * (nb >> 3) + (b >> 3); }

// The value of the lane behind / ahead (a shift of the whole wavefront by one lane; the lane at the
// end gets 0): a register move, where a shuffle goes through LDS.
__device__ __forceinline__ double lane_back(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x138, 0xf, 0xf, true);  // wave_shr:1
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x138, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane_front(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x130, 0xf, 0xf, true);  // wave_shl:1
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x130, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// Arcane math::min / math::max
__device__ __forceinline__ double amin(double a, double b) { return (a < b) ? a : b; }
__device__ __forceinline__ double amax(double a, double b) { return (a < b) ? b : a; }

__device__ __forceinline__ D3 load3(double* const* a, long n) { return d3(a[0][n], a[1][n], a[2][n]); }


// The node coordinates of the cell whose node 0 is b, in Arcane's local node order.
template <int DIM>
__device__ __forceinline__ void cell_nodes(const MhDev& S, long b, double* const* xs, D3* x) {
  const long nnx = S.g.nnx, nnxy = (long)S.g.nnx * S.g.nny;
  if (DIM == 3) {
    x[0] = load3(xs, b);
    x[1] = load3(xs, b + 1);
    x[2] = load3(xs, b + 1 + nnx);
    x[3] = load3(xs, b + nnx);
    x[4] = load3(xs, b + nnxy);
    x[5] = load3(xs, b + 1 + nnxy);
    x[6] = load3(xs, b + 1 + nnx + nnxy);
    x[7] = load3(xs, b + nnx + nnxy);
  } else {
    x[0] = d3(xs[0][b], xs[1][b], 0.);
    x[1] = d3(xs[0][b + 1], xs[1][b + 1], 0.);
    x[2] = d3(xs[0][b + 1 + nnx], xs[1][b + 1 + nnx], 0.);
    x[3] = d3(xs[0][b + nnx], xs[1][b + nnx], 0.);
  }
}

// Block-wide minimum (Arcane math::min semantics on non-NaN input), written by thread 0.
// CFL minimum with the reference's sequential semantics.  computeDeltaT folds
// min = math::min(min, dx) over the cells in order (MahycoModule.cc:1777), and math::min(a,
// b) = a < b ? a : b turns NaN at a NaN candidate (an emptied cell's sound speed) and
// restarts at the next cell: the result is the minimum over the cells after the last NaN
// candidate, NaN if the last cell is one.  A run of cells therefore reduces to (nan: a NaN
// was seen, m: minimum after the last NaN, NaN if there is no value there), combined in
// cell order; (NaN, no NaN seen) is the empty run.  The reference's start value (the
// largest double) is applied once, at the end.
struct MhCflMin {
  double m;
  int nan;
};
__device__ __forceinline__ double min_skip_nan(double a, double b) { return (b < a || a != a) ? b : a; }
__device__ __forceinline__ MhCflMin cfl_leaf(double x, bool active) {
  MhCflMin r;
  r.nan = active && x != x;
  r.m = active ? x : __longlong_as_double(0x7ff8000000000000LL);  // inactive: the empty run
  return r;
}
__device__ __forceinline__ MhCflMin cfl_combine(MhCflMin l, MhCflMin r) {
  if (r.nan) return r;
  MhCflMin o;
  o.nan = l.nan;
  o.m = min_skip_nan(l.m, r.m);
  return o;
}
// in-order reduction over a wavefront (lane 0 ends with lanes 0..63 combined); without a
// NaN in the wavefront it is a plain minimum, in any order
__device__ __forceinline__ MhCflMin cfl_wave(MhCflMin v) {
  const int lane = threadIdx.x & 63;
  if (__ballot(v.nan) == 0) {
    for (int off = 32; off > 0; off >>= 1) v.m = min_skip_nan(v.m, __shfl_xor(v.m, off, 64));
    return v;
  }
  for (int off = 1; off < 64; off <<= 1) {
    MhCflMin o;
    o.m = __shfl_down(v.m, off, 64);
    o.nan = __shfl_down(v.nan, off, 64);
    if (lane + off < 64) v = cfl_combine(v, o);
  }
  return v;
}

// Per-block CFL partial of the cells of block lb, in cell order: out[2 lb] = minimum after
// the last NaN, out[2 lb + 1] = 1 if a NaN was seen.
__device__ __forceinline__ void block_min_store(double v, bool active, double* out, int lb) {
  __shared__ double rm[MH_BLOCK / 64];
  __shared__ int rn[MH_BLOCK / 64];
  MhCflMin r = cfl_wave(cfl_leaf(v, active));
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) {
    rm[wid] = r.m;
    rn[wid] = r.nan;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    MhCflMin t;
    t.m = rm[0];
    t.nan = rn[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) {
      MhCflMin o;
      o.m = rm[w];
      o.nan = rn[w];
      t = cfl_combine(t, o);
    }
    out[2 * lb] = t.m;
    out[2 * lb + 1] = t.nan ? 1. : 0.;
  }
}

// ----------------------------------------------------------------------------- nodes
// Node mass and corner forces of node (i,j,k) over its cells, in the order of a cell-order scatter
// (MahycoModule.cc:247-262 and :455-462).
// FWD: the corner vectors at this cycle's Lagrangian positions (updateVelocityForward,
// :638-690) instead of the previous cycle's.
// The 3x3(x3) nodes around are read once each; indices past the mesh are clamped and the terms of a
// cell outside it are dropped by a select, so no branch parts the loads: they are all in flight
// together (3D: those of one cell plane), where a branch per cell waited for each cell in turn: 28.5 ->
// 26 us on 1023x1021, 6.2 -> 5.4 us on 200x10, 146 -> 128 us for 64 meshes of 64^2 to 512^2.
template <int DIM, int A, int B, int DZ>  // this node's corner vector of cell (A,B,DZ) around it
__device__ __forceinline__ D3 node_corner(const D3 (*lo)[3], const D3 (*hi)[3]) {
  constexpr int L = 4 * (1 - DZ) + (B ? (A ? 0 : 1) : (A ? 3 : 2));
  if constexpr (DIM == 3) {
    const D3 x[8] = {lo[B][A], lo[B][A + 1], lo[B + 1][A + 1], lo[B + 1][A],
                     hi[B][A], hi[B][A + 1], hi[B + 1][A + 1], hi[B + 1][A]};
    return cqs_hex_corner<L>(x);
  } else {
    const D3 x[4] = {lo[B][A], lo[B][A + 1], lo[B + 1][A + 1], lo[B + 1][A]};
    return cqs_quad_corner<L & 3>(x);
  }
}
template <int DIM, int A, int B, int DZ>
__device__ __forceinline__ void node_add(const D3 (*lo)[3], const D3 (*hi)[3], double M, double p, double q, bool ok,
                                         double& mass, double& fx, double& fy, double& fz) {
  const D3 v = node_corner<DIM, A, B, DZ>(lo, hi);
  const double pr = p + q;
  mass = ok ? mass + (DIM == 3 ? 0.125 : 0.25) * M : mass;
  fx = ok ? fx + pr * v.x : fx;
  fy = ok ? fy + pr * v.y : fy;
  if (DIM == 3) fz = ok ? fz + pr * v.z : fz;
}
template <int DIM, int FWD = 0>
__device__ __forceinline__ void node_gather(const MhDev& S, int i, int j, int k, double& mass, double& fx, double& fy,
                                            double& fz) {
  double* const* X = FWD ? S.xlc : S.xlp;
  const int nx = S.g.nx, ny = S.g.ny, nz = S.g.nz;
  const long nnx = S.g.nnx, nny = S.g.nny;
  const int ni[3] = {max(i - 1, 0), i, min(i + 1, nx)}, nj[3] = {max(j - 1, 0), j, min(j + 1, ny)};
  const int ci[2] = {max(i - 1, 0), min(i, nx - 1)}, cj[2] = {max(j - 1, 0), min(j, ny - 1)};
  const bool oi[2] = {i > 0, i < nx}, oj[2] = {j > 0, j < ny};
  D3 lo[3][3], hi[3][3];
  auto plane = [&](D3 (*P)[3], int kz) {
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const long n = ni[a] + nnx * (nj[b] + nny * kz);
        P[b][a] = d3(X[0][n], X[1][n], DIM == 3 ? X[2][n] : 0.);
      }
  };
  // the four cells of cell plane kc, as members of the mesh where ok
  auto cells = [&](auto dz, int kc, bool ok) {
    constexpr int DZ = decltype(dz)::value;
    double M[4], p[4], q[4];
#pragma unroll
    for (int l = 0; l < 4; ++l) {
      const long c = ci[l & 1] + (long)nx * (cj[l >> 1] + (long)ny * kc);
      M[l] = S.M[c];
      p[l] = S.p[c];
      q[l] = S.q[c];
    }
    node_add<DIM, 0, 0, DZ>(lo, hi, M[0], p[0], q[0], ok && oi[0] && oj[0], mass, fx, fy, fz);
    node_add<DIM, 1, 0, DZ>(lo, hi, M[1], p[1], q[1], ok && oi[1] && oj[0], mass, fx, fy, fz);
    node_add<DIM, 0, 1, DZ>(lo, hi, M[2], p[2], q[2], ok && oi[0] && oj[1], mass, fx, fy, fz);
    node_add<DIM, 1, 1, DZ>(lo, hi, M[3], p[3], q[3], ok && oi[1] && oj[1], mass, fx, fy, fz);
  };
  if constexpr (DIM == 3) {
    plane(lo, max(k - 1, 0));
    plane(hi, k);
    cells(std::integral_constant<int, 0>{}, max(k - 1, 0), k > 0);
    asm volatile("" ::: "memory");  // the next plane's loads would take the registers of this one's corners
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int a = 0; a < 3; ++a) lo[b][a] = hi[b][a];
    plane(hi, min(k + 1, nz));
    cells(std::integral_constant<int, 1>{}, min(k, nz - 1), k < nz);
  } else {
    plane(lo, 0);
    cells(std::integral_constant<int, 1>{}, 0, true);
  }
}

// UpdateVelocity tail (u += dt_half / m F), ApplyBoundaryCondition (Vx/Vy/Vz on the
// XMIN..ZMAX node groups, in option order) and UpdatePosition (x += dt u) for node n.
// The node's own state, u and the position the step starts from (the Eulerian one with remap), is
// loaded by the caller ahead of the forces.
struct NodePre {
  double u[3], x[3];
};
template <int DIM>
__device__ __forceinline__ void node_pre_load(const MhDev& S, long n, int i, int j, int k, NodePre& pre) {
#pragma unroll
  for (int d = 0; d < 3; ++d) pre.u[d] = d < DIM ? S.u[d][n] : 0.;
  if (S.with_proj) {
    pre.x[0] = S.ax[i];
    pre.x[1] = S.ay[j];
    pre.x[2] = DIM == 3 ? S.az[k] : 0.;
  } else {
#pragma unroll
    for (int d = 0; d < 3; ++d) pre.x[d] = d < DIM ? S.xlp[d][n] : 0.;
  }
}
template <int DIM>
__device__ __forceinline__ void node_finish(const MhDev& S, long n, int i, int j, int k, double dt, double dth,
                                            const NodePre& pre, double mass, double fx, double fy, double fz) {
  const double s = dth / mass;
  double ux = pre.u[0], uy = pre.u[1], uz = pre.u[2];
  if (S.csts) {  // SaveValuesAtN of the velocity
    S.un[0][n] = ux;
    S.un[1][n] = uy;
    if (DIM == 3) S.un[2][n] = uz;
  }
  if (S.csts && S.with_proj) {  // updateVelocityBackward (:451-453, 574-627)
    const double sb = (-0.5 * S.sc->dt_old) / mass;
    ux = ux + sb * fx;
    uy = uy + sb * fy;
    if (DIM == 3) uz = uz + sb * fz;
  }
  ux = ux + s * fx;
  uy = uy + s * fy;
  if (DIM == 3) uz = uz + s * fz;
  for (int b = 0; b < S.nbc; ++b) {
    const int sf = S.bc_surf[b];
    bool on;
    switch (sf) {
      case MH_XMIN: on = (i == 0); break;
      case MH_XMAX: on = (i == S.g.nx); break;
      case MH_YMIN: on = (j == 0); break;
      case MH_YMAX: on = (j == S.g.ny); break;
      case MH_ZMIN: on = DIM == 3 ? (k == 0) : true; break;
      default: on = DIM == 3 ? (k == S.g.nz) : true; break;
    }
    if (on) {
      const int t = S.bc_type[b];
      if (t == MH_BC_VX) ux = S.bc_val[b];
      else if (t == MH_BC_VY) uy = S.bc_val[b];
      else if (DIM == 3) uz = S.bc_val[b];
    }
  }
  S.u[0][n] = ux;
  S.u[1][n] = uy;
  S.xlc[0][n] = pre.x[0] + dt * ux;
  S.xlc[1][n] = pre.x[1] + dt * uy;
  if (DIM == 3) {
    S.u[2][n] = uz;
    S.xlc[2][n] = pre.x[2] + dt * uz;
  }
  S.mn[n] = mass;
}


// SaveValuesAtN + UpdateVelocity (:438-562) + ApplyBoundaryCondition (:756-807) +
// UpdatePosition (:730-751) for one node.
template <int DIM>
__device__ __forceinline__ void k_node_lag_body(const MhDev& S, int lb) {
  const long n = lb * (long)blockDim.x + threadIdx.x;
  if (n >= S.g.nn) return;
  const bool halted = mh_halted(S.sc);
  const int nnx = S.g.nnx, nny = S.g.nny;
  const int i = (int)(n % nnx);
  const long r = n / nnx;
  const int j = (int)(r % nny);
  const int k = (int)(r / nny);
  const double dt = S.sc->dt;
  const double dth = 0.5 * (S.sc->dt_old + dt);
  NodePre pre;
  node_pre_load<DIM>(S, n, i, j, k, pre);
  double mass = 0., fx = 0., fy = 0., fz = 0.;
  node_gather<DIM>(S, i, j, k, mass, fx, fy, fz);
  if (halted) return;
  node_finish<DIM>(S, n, i, j, k, dt, dth, pre, mass, fx, fy, fz);
}


// The same in 3D with the cells shared out over the wavefronts: a block owns 64 nodes, each of its
// four wavefronts the two cells (one below, one above) of one quadrant around them, and the first
// one adds the eight terms from LDS in cell order.  A thread of the kernel above forms eight corner
// vectors of some 200 operations each one after the other, and waits for its two cell planes in
// turn; a mesh of a few hundred wavefronts has the processors free to do that at once: 12.6 -> 7.2 us
// on 100x5x5, one thread per node against this.
template <int A, int B>
__device__ __forceinline__ void node_quadrant(const MhDev& S, int i, int j, int k, double* out) {
  const int nx = S.g.nx, ny = S.g.ny, nz = S.g.nz;
  const long nnx = S.g.nnx, nny = S.g.nny;
  const int ni[2] = {A ? i : max(i - 1, 0), A ? min(i + 1, nx) : i}, nj[2] = {B ? j : max(j - 1, 0), B ? min(j + 1, ny) : j};
  const int nk[3] = {max(k - 1, 0), k, min(k + 1, nz)};
  D3 P[3][3][3];  // rows and columns A, A + 1 of the 3x3 neighbourhood are used
#pragma unroll
  for (int z = 0; z < 3; ++z)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int a = 0; a < 2; ++a) P[z][B + b][A + a] = load3(S.xlp, ni[a] + nnx * (nj[b] + nny * nk[z]));
  const int ci = A ? min(i, nx - 1) : max(i - 1, 0), cj = B ? min(j, ny - 1) : max(j - 1, 0);
  double M[2], p[2], q[2];
#pragma unroll
  for (int z = 0; z < 2; ++z) {
    const long c = ci + (long)nx * (cj + (long)ny * (z ? min(k, nz - 1) : max(k - 1, 0)));
    M[z] = S.M[c];
    p[z] = S.p[c];
    q[z] = S.q[c];
  }
  auto corner = [&](auto dz) {
    constexpr int DZ = decltype(dz)::value;
    const D3 v = node_corner<3, A, B, DZ>(P[DZ], P[DZ + 1]);
    const double pr = p[DZ] + q[DZ];
    double* o = out + DZ * (4 * 4 * 64);
    o[0] = 0.125 * M[DZ];
    o[64] = pr * v.x;
    o[128] = pr * v.y;
    o[192] = pr * v.z;
  };
  corner(std::integral_constant<int, 0>{});
  corner(std::integral_constant<int, 1>{});
}
__device__ __forceinline__ void k_node_lag3_split_body(const MhDev& S, int lb) {
  static_assert(MH_BLOCK == 256, "one wavefront per quadrant");
  __shared__ double part[2][4][4][64];  // cells below / above, quadrant, (mass, force), node
  const bool halted = mh_halted(S.sc);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long n = min(lb * 64L + lane, S.g.nn - 1);
  const int nnx = S.g.nnx, nny = S.g.nny;
  const int i = (int)(n % nnx);
  const long r = n / nnx;
  const int j = (int)(r % nny);
  const int k = (int)(r / nny);
  const double dt = S.sc->dt;
  const double dth = 0.5 * (S.sc->dt_old + dt);
  NodePre pre;
  if (w == 0) {
    node_pre_load<3>(S, n, i, j, k, pre);
    node_quadrant<0, 0>(S, i, j, k, &part[0][0][0][lane]);
  } else if (w == 1) {
    node_quadrant<1, 0>(S, i, j, k, &part[0][1][0][lane]);
  } else if (w == 2) {
    node_quadrant<0, 1>(S, i, j, k, &part[0][2][0][lane]);
  } else {
    node_quadrant<1, 1>(S, i, j, k, &part[0][3][0][lane]);
  }
  __syncthreads();
  if (w || halted || lb * 64L + lane >= S.g.nn) return;
  double sum[4] = {0., 0., 0., 0.};
  const bool okz[2] = {k > 0, k < S.g.nz};
  const bool okq[4] = {i > 0 && j > 0, i < S.g.nx && j > 0, i > 0 && j < S.g.ny, i < S.g.nx && j < S.g.ny};
#pragma unroll
  for (int z = 0; z < 2; ++z)
#pragma unroll
    for (int l = 0; l < 4; ++l)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const double t = sum[v] + part[z][l][v][lane];
        sum[v] = okz[z] && okq[l] ? t : sum[v];
      }
  node_finish<3>(S, n, i, j, k, dt, dth, pre, sum[0], sum[1], sum[2], sum[3]);
}

// updateVelocityForward (:638-690), before a CSTS remap: u += (dt/2) / m F with the force of
// this cycle's pressure array, pseudo-viscosity and corner vectors (no boundary condition).
template <int DIM>
__device__ __forceinline__ void k_node_fwd_body(const MhDev& S, int lb) {
  const long n = lb * (long)blockDim.x + threadIdx.x;
  if (n >= S.g.nn) return;
  if (mh_halted(S.sc)) return;
  const int nnx = S.g.nnx, nny = S.g.nny;
  const int i = (int)(n % nnx);
  const long r = n / nnx;
  const int j = (int)(r % nny);
  const int k = (int)(r / nny);
  double mass = 0., fx = 0., fy = 0., fz = 0.;
  node_gather<DIM, 1>(S, i, j, k, mass, fx, fy, fz);
  const double s = (0.5 * S.sc->dt) / S.mn[n];
  S.u[0][n] = S.u[0][n] + s * fx;
  S.u[1][n] = S.u[1][n] + s * fy;
  if (DIM == 3) S.u[2][n] = S.u[2][n] + s * fz;
}

// Advection mode (sans-lagrange), node part: updateVelocityWithoutLagrange
// (MahycoModule.cc:702-718), u = u0 (1 - r) + (r u0) cos(pi t parametre) with r = 1 under
// the reverse option, the boundary conditions, and updatePosition (:730-751), which moves
// only the nodes shared by exactly four cells.
template <int DIM>
__device__ __forceinline__ void k_node_adv_body(const MhDev& S, int lb) {
  const long n = lb * (long)blockDim.x + threadIdx.x;
  if (n >= S.g.nn) return;
  if (mh_halted(S.sc)) return;
  const int nnx = S.g.nnx, nny = S.g.nny;
  const int i = (int)(n % nnx);
  const long r = n / nnx;
  const int j = (int)(r % nny);
  const int k = (int)(r / nny);
  const double dt = S.sc->dt;
  const long it = S.sc->iteration;
  const double cs = S.rev_cos[it < S.rev_n ? it : S.rev_n - 1];
  const double opt = S.rider_reverse ? 1. : 0.;
  double u[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double a = S.u0[d][n];
    u[d] = a * (1. - opt) + opt * a * cs;
  }
  for (int b = 0; b < S.nbc; ++b) {
    const int sf = S.bc_surf[b];
    bool on;
    switch (sf) {
      case MH_XMIN: on = (i == 0); break;
      case MH_XMAX: on = (i == S.g.nx); break;
      case MH_YMIN: on = (j == 0); break;
      case MH_YMAX: on = (j == S.g.ny); break;
      case MH_ZMIN: on = DIM == 3 ? (k == 0) : true; break;
      default: on = DIM == 3 ? (k == S.g.nz) : true; break;
    }
    if (on) u[S.bc_type[b]] = S.bc_val[b];
  }
  const int cells = ((i > 0) + (i < S.g.nx)) * ((j > 0) + (j < S.g.ny)) * (DIM == 3 ? (k > 0) + (k < S.g.nz) : 1);
  const bool moves = cells == 4;
  const double x0[3] = {S.ax[i], S.ay[j], DIM == 3 ? S.az[k] : 0.};
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    S.u[d][n] = u[d];
    S.xlc[d][n] = moves ? x0[d] + dt * u[d] : x0[d];
  }
  if (DIM == 2) S.u[2][n] = u[2];
}

// 3D node kernel, z-marching tiles: a block owns MH_NTX x MH_NTY node columns over MhDev::nt_kc node
// planes, so each cell plane of the tile is (MH_NTX+1) x (MH_NTY+1) = 256 cells, one per thread.  Each
// cell plane is processed once: its corner vectors (cqs_hex, computed once per cell instead of once
// per corner) are multiplied by p+q and go to LDS with M/8.  The node threads then finish node plane k
// with the bottom corners, on top of the sums they hold of the cells below, and start the sums of
// plane k + 1 with the top corners: the 8 cells are added in cell order, as in k_node_lag, so both
// kernels give the same bits.
// Bound by FP64 issue, at two wavefronts per SIMD (the corner vectors take 240 registers), 60 % busy:
// so the geometry is formed in the units of hex_face32, and all that a plane reads (the next cell, the
// node's own velocity) is in flight before the corner vectors are formed.  267 -> 234 us on
// 256x128x128, 433 -> 361 us on 192^3, with node_tile_depth 79 -> 59 us on 128x96x64.
#ifndef MH_NTX
#define MH_NTX 31  // node columns of a tile along x
#endif
#define MH_NTY (MH_BLOCK / (MH_NTX + 1) - 1)  // along y: (MH_NTX + 1)(MH_NTY + 1) cells = MH_BLOCK
#define MH_NT_KC 8  // node planes per tile by default (MhDev::nt_kc)
#define MH_NT_CELLS ((MH_NTX + 1) * (MH_NTY + 1))  // = MH_BLOCK
// What one cell of a column needs beyond its lower face: the 4 nodes of its upper face
// (previous Lagrangian positions) and p, q, M.  The lower face is the upper face of the
// cell below, carried in registers.
struct NtCellIn {
  D3 top[4];
  double p, q, M;
};
__device__ __forceinline__ void nt_load_face(const MhDev& S, int ii, int jj, int kn, D3* f) {
  const long nnx = S.g.nnx;
  const long b = ii + nnx * (jj + (long)S.g.nny * kn);
  f[0] = load3(S.xlp, b);
  f[1] = load3(S.xlp, b + 1);
  f[2] = load3(S.xlp, b + 1 + nnx);
  f[3] = load3(S.xlp, b + nnx);
}
__device__ __forceinline__ void nt_load_cell(const MhDev& S, int ii, int jj, int kk, NtCellIn& in) {
  const long c = ii + (long)S.g.nx * (jj + (long)S.g.ny * kk);
  nt_load_face(S, ii, jj, kk + 1, in.top);
  in.p = S.p[c];
  in.q = S.q[c];
  in.M = S.M[c];
}
// corner force contributions (p + q) CQS_l and the node-mass share M/8 of one cell to slot s: lower
// corners to up, upper corners to lo
__device__ __forceinline__ void nt_cell(const D3* bot, const NtCellIn& in, double* up, double* lo, int s) {
  const D3 x[8] = {bot[0], bot[1], bot[2], bot[3], in.top[0], in.top[1], in.top[2], in.top[3]};
  const double pr = in.p + in.q;
  const double wm = 0.125 * in.M;
  cqs_hex_each(x, [&](int l, const D3& q) {
    double* P = l < 4 ? up : lo;
    P[(3 * (l & 3) + 0) * MH_NT_CELLS + s] = pr * q.x;
    P[(3 * (l & 3) + 1) * MH_NT_CELLS + s] = pr * q.y;
    P[(3 * (l & 3) + 2) * MH_NT_CELLS + s] = pr * q.z;
  });
  up[12 * MH_NT_CELLS + s] = wm;
}

__device__ __forceinline__ void nt_add(const double* P, const double* W, int s, int corner, bool ok, double& mass,
                                       double& fx, double& fy, double& fz) {
  const double m = mass + W[12 * MH_NT_CELLS + s];
  const double x = fx + P[(3 * corner + 0) * MH_NT_CELLS + s];
  const double y = fy + P[(3 * corner + 1) * MH_NT_CELLS + s];
  const double z = fz + P[(3 * corner + 2) * MH_NT_CELLS + s];
  mass = ok ? m : mass;
  fx = ok ? x : fx;
  fy = ok ? y : fy;
  fz = ok ? z : fz;
}

__device__ __forceinline__ void k_node_lag3_tiled_body(const MhDev& S, int bx, int by, int bz) {
  static_assert(MH_NT_CELLS == MH_BLOCK, "one cell of the tile plane per thread");
  __shared__ double up[13 * MH_NT_CELLS];  // bottom corners (0..3) and M/8 of the cell plane
  __shared__ double lo[12 * MH_NT_CELLS];  // its top corners (4..7)
  if (mh_halted(S.sc)) return;
  const int tid = threadIdx.x;
  const int i0 = bx * MH_NTX, j0 = by * MH_NTY, k0 = bz * S.nt_kc;
  const int nx = S.g.nx, ny = S.g.ny, nz = S.g.nz;
  const int kend = min(k0 + S.nt_kc, S.g.nnz);
  const double dt = S.sc->dt;
  const double dth = 0.5 * (S.sc->dt_old + dt);
  // this thread's cell column of the tile; a column outside the mesh reads the nearest one inside
  const int ci = min(max(i0 - 1 + tid % (MH_NTX + 1), 0), nx - 1);
  const int cj = min(max(j0 - 1 + tid / (MH_NTX + 1), 0), ny - 1);
  // this thread's node column (threads below MH_NTX * MH_NTY)
  const int tx = tid % MH_NTX, ty = tid / MH_NTX;
  const int i = i0 + tx, j = j0 + ty;
  const bool node_ok = tid < MH_NTX * MH_NTY && i < S.g.nnx && j < S.g.nny;
  const int s00 = min(ty * (MH_NTX + 1) + tx, MH_NT_CELLS - MH_NTX - 3);  // cell (i-1, j-1)
  const int in = min(i, nx), jn = min(j, ny);
  const long n0 = in + (long)S.g.nnx * jn, nplane = (long)S.g.nnx * S.g.nny;
  const bool okx0 = i >= 1, okx1 = i < nx, oky0 = j >= 1, oky1 = j < ny;
  auto add4 = [&](const double* P, double& mass, double& fx, double& fy, double& fz) {
    nt_add(P, up, s00, 2, okx0 && oky0, mass, fx, fy, fz);
    nt_add(P, up, s00 + 1, 3, okx1 && oky0, mass, fx, fy, fz);
    nt_add(P, up, s00 + MH_NTX + 1, 1, okx0 && oky1, mass, fx, fy, fz);
    nt_add(P, up, s00 + MH_NTX + 2, 0, okx1 && oky1, mass, fx, fy, fz);
  };
  // the lower face of the thread's cell is carried from plane to plane; the next cell's loads and
  // the loads of the node's own state go out one plane ahead
  D3 bot[4];
  NtCellIn cur, nxt;
  NodePre pre;
  const int kc_end = min(kend, nz);  // cell planes kb .. kc_end - 1
  const int kb = max(k0 - 1, 0);
  nt_load_face(S, ci, cj, kb, bot);
  nt_load_cell(S, ci, cj, kb, nxt);
  // sums of the node over the cells below it
  double mass = 0., fx = 0., fy = 0., fz = 0.;
  for (int k = kb; k < kend; ++k) {
    const bool cells = k < nz;  // a cell plane sits on this node plane
    node_pre_load<3>(S, n0 + nplane * k, in, jn, k, pre);
    if (cells) {
      cur = nxt;
      if (k + 1 < kc_end) nt_load_cell(S, ci, cj, k + 1, nxt);
      nt_cell(bot, cur, up, lo, tid);
      for (int l = 0; l < 4; ++l) bot[l] = cur.top[l];
    }
    __syncthreads();
    if (k >= k0) {
      if (cells) add4(up, mass, fx, fy, fz);
      if (node_ok) node_finish<3>(S, n0 + nplane * k, i, j, k, dt, dth, pre, mass, fx, fy, fz);
    }
    mass = fx = fy = fz = 0.;
    if (cells) add4(lo, mass, fx, fy, fz);
    __syncthreads();
  }
}

// ----------------------------------------------------------------------------- cells

// max over the cell's nodes of |u| (MahycoModule.cc:1771-1774).  The root is taken of the largest
// square: sqrt is monotonic and correctly rounded, so that is the largest root, and amax hands on
// the same operand of squares as of roots, NaN included.
template <int DIM>
__device__ __forceinline__ double cell_vmax2(const MhDev& S, long b) {
  const long nnx = S.g.nnx, nnxy = (long)S.g.nnx * S.g.nny;
  const long off[8] = {0, 1, 1 + nnx, nnx, nnxy, 1 + nnxy, 1 + nnx + nnxy, nnx + nnxy};
  double v = 0.;
#pragma unroll
  for (int l = 0; l < (DIM == 3 ? 8 : 4); ++l) {
    const long n = b + off[l];
    const double ux = S.u[0][n], uy = S.u[1][n];
    const double uz = DIM == 3 ? S.u[2][n] : 0.;
    v = amax(ux * ux + uy * uy + uz * uz, v);
  }
  return v;
}

// updateEnergyAndPressureforGP, MahycoModule.cc:1633-1659 (pseudo-centree off)
__device__ __forceinline__ double gp_energy(double e_n, double p, double rho, double rho_n, double q,
                                            double gamma) {
  const double dv = 1.0 / rho - 1.0 / rho_n;
  double pseudo = 0.;
  if (q * (1.0 / rho - 1.0 / rho_n) < 0.) pseudo = q;
  const double denom = 1 + 0.5 * (gamma - 1.0) * rho * dv;
  const double numer = e_n - (0.5 * p + pseudo) * dv;
  return numer / denom;
}

// Energy of one environment after the Lagrange step: updateEnergyAndPressureforGP (closed
// form above), updateEnergyAndPressurebyNewton (MahycoModule.cc:1506-1540: Newton on fvnr,
// MahycoModule.h:378-386, with the EOS of applyOneCellEOS at each iterate) or
// updateEnergyAndPressureExplicite (:1484-1502).  Newton's last pressure and sound speed are
// replaced by the EOS call that follows the update (or the remap), so only e is returned.
// What the Lagrange step takes from an environment's parameters (MhEnvParam has the same names).
struct MhEosCoef {
  double gamma, pinf, a1, a2;
  int stiffened;
};
template <class EnvP>
__device__ __forceinline__ double lag_energy(const MhDev& S, const EnvP& ep, double e_n, double p_n, double rho,
                                             double rho_n, double q) {
  if (S.p_explicit) return e_n - (p_n + q) * (1.0 / rho - 1.0 / rho_n);
  if (!S.newton) return gp_energy(e_n, p_n, rho, rho_n, q, ep.gamma);
  double pseudo = 0.;
  if (q * (1.0 / rho - 1.0 / rho_n) < 0.) pseudo = q;
  const double g = ep.gamma;
  double e = e_n, p = p_n;
  for (int i = 0; i < 50; ++i) {
    if (!(fabs(e - e_n + 0.5 * (p + p_n + 2. * pseudo) * (1. / rho - 1. / rho_n)) >= S.thr_module)) break;
    p = ep.stiffened ? ((g - 1.) * rho * e) - (g * ep.pinf) : (g - 1.) * rho * e;
    const double dpde = (g - 1.) * rho;
    const double f = e - e_n + 0.5 * (p + p_n + 2. * pseudo) * (1. / rho - 1. / rho_n);
    e = e - f / (1. + 0.5 * dpde * (1. / rho - 1. / rho_n));
  }
  return e;
}

// applyEOS (PerfectGasEOSService.cc:45-67, StiffenedGasEOSService.cc:43-63)
template <class EnvP>
__device__ __forceinline__ void eos(const EnvP& ep, double rho, double e, double& p, double& c) {
  const double g = ep.gamma;
  if (ep.stiffened) {
    p = ((g - 1.) * rho * e) - (g * ep.pinf);
    c = sqrt((g / rho) * (p + ep.pinf));
  } else {
    p = (g - 1.) * rho * e;
    c = sqrt(g * p / rho);
  }
}

// FictifEOSService::applyEOS (eos/fictif/FictifEOSService.cc:45-75): the pressure only
// depends on the time t of the iteration, the sound speed is 1 and the caller zeroes the
// internal energy.
__device__ __forceinline__ void fictif_eos(const MhEnvParam& ep, double t, double pprev, double& p, double& c) {
  p = pprev;
  if (t > ep.ft0) p = ep.fp0 + ep.fdpdt * t;
  if (t > ep.ft1) p = 0.;
  c = 1.;
}

// updateEnergyAndPressureforGP, CSTS branch (MahycoModule.cc:1661-1697): the work of the
// corner forces at n (previous cycle's corner vectors, saved velocity) and n+1 (this cycle's
// corner vectors qv, velocity at n+1/2), one set per cell ...
template <int DIM>
__device__ __forceinline__ void csts_work(const MhDev& S, long b, const D3* qv, double& cn1, double& cn, double& cdn,
                                          double& cvon) {
  constexpr int NN = DIM == 3 ? 8 : 4;
  const long nnx = S.g.nnx, nnxy = (long)S.g.nnx * S.g.nny;
  const long off[8] = {0, 1, 1 + nnx, nnx, nnxy, 1 + nnxy, 1 + nnx + nnxy, nnx + nnxy};
  D3 xp[8], qn[8];
  for (int l = 0; l < NN; ++l)
    xp[l] = d3(S.xlp[0][b + off[l]], S.xlp[1][b + off[l]], DIM == 3 ? S.xlp[2][b + off[l]] : 0.);
  if (DIM == 3) cqs_hex(xp, qn);
  else cqs_quad(xp, qn);
  const double dtn = S.sc->dt, dto = S.sc->dt_old;
  cn1 = 0.;
  cn = 0.;
  cdn = 0.;
  cvon = 0.;
  for (int l = 0; l < NN; ++l) {
    const long n = b + off[l];
    const D3 v = d3(S.u[0][n], S.u[1][n], DIM == 3 ? S.u[2][n] : 0.);
    const D3 vn = d3(S.un[0][n], S.un[1][n], DIM == 3 ? S.un[2][n] : 0.);
    const D3 dv = v - vn;
    cn1 += (v.x * qv[l].x + v.y * qv[l].y + v.z * qv[l].z) * dtn;
    cn += (v.x * qn[l].x + v.y * qn[l].y + v.z * qn[l].z) * dtn;
    cdn += (dv.x * qn[l].x + dv.y * qn[l].y + dv.z * qn[l].z) * (dtn - dto);
    cvon += (vn.x * qn[l].x + vn.y * qn[l].y + vn.z * qn[l].z) * dto;
  }
}
// ... priced per environment with its own mass, density, pressure and pseudo-viscosities
template <class EnvP>
__device__ __forceinline__ double csts_e(const EnvP& ep, double e, double M, double rho, double pn, double qn,
                                         double qnm1, double q, double cn1, double cn, double cdn, double cvon) {
  const double denom = 1 + 0.5 * (ep.gamma - 1.0) * rho * cn1 / M;
  const double numer = e - (0.5 * (pn + qn) * cn / M) - (0.5 * q * cn1 / M) + (0.25 * (pn + qn) * cdn / M) -
                       (0.5 * (qn - qnm1) * cvon / M);
  return numer / denom;
}
// q^(n-1) of environment k in cell c (m_pseudo_viscosity_nmoins1, MahycoModule.cc:347, 360),
// through Arcane's membership changes at the last remap (mask before it: mkm1): an
// environment that entered has a new partial value (0); one that was alone in the cell takes
// the cell value (qm1); one of a mixed cell keeps its partial value, the remap-before-last's
// U_q / V (qem1).  A cell alone in one environment now reads the cell value.
__device__ __forceinline__ double csts_qnm1(const MhDev& S, long c, int k, bool mixed_now) {
  const uint8_t pm = S.mkm1[c];
  const bool was = (pm >> k) & 1;
  if (__popc(pm) >= 2) return was ? S.qem1[c] : 0.;
  if (mixed_now) return was ? S.qm1[c] : 0.;
  return S.qm1[c];
}

// The characteristic lengths other than V^(1/d) (computeGeometricValues, MahycoModule.cc:
// 1195-1236): the median lengths between opposite faces (3D), or one side of the cell.
template <int DIM>
__device__ __forceinline__ double char_length_alt(int lc, const D3* x) {
  if (DIM == 3 && lc == MH_L_FACES_OPPOSEES) {
    auto quarter_sum = [](D3 a, D3 b, D3 c, D3 d) {
      const D3 s = a + b + c + d;
      return d3(0.25 * s.x, 0.25 * s.y, 0.25 * s.z);
    };
    auto norm = [](D3 v) { return sqrt(v.x * v.x + v.y * v.y + v.z * v.z); };
    const D3 f0 = quarter_sum(x[0], x[3], x[2], x[1]), f1 = quarter_sum(x[0], x[4], x[7], x[3]);
    const D3 f2 = quarter_sum(x[0], x[1], x[5], x[4]), f3 = quarter_sum(x[4], x[5], x[6], x[7]);
    const D3 f4 = quarter_sum(x[1], x[2], x[6], x[5]), f5 = quarter_sum(x[2], x[3], x[7], x[6]);
    const double d1 = norm(f0 - f3), d2 = norm(f2 - f5), d3v = norm(f1 - f4);
    return (d1 * d2 * d3v) / (d1 * d2 + d1 * d3v + d2 * d3v);
  }
  if (lc == MH_L_MONODIM_X) return fabs(x[2].x - x[0].x);
  if (lc == MH_L_MONODIM_Y) return fabs(x[2].y - x[0].y);
  return fabs(x[2].z - x[0].z);
}

// Which environments a cell's remap vector holds anything of.  Most cells of a multi-material mesh
// hold one material, and the volume, mass and energy slots of the others are zeros that every sweep
// would read, divide, limit and write.  Beside each U buffer one byte per cell (MhDev::pm, null for
// meshes whose sweeps do not use it) keeps the invariant: bit k clear => the buffer's three slots of
// environment k are 0 in that cell.  The buffers always hold those zeros, so code that ignores the
// bytes reads the same values; a writer stores a zero only where the bit was set.
__device__ __forceinline__ bool mh_finite_nonzero(double x) { return __builtin_amdgcn_class(x, 0x198); }
__device__ __forceinline__ bool mh_finite(double x) { return __builtin_amdgcn_class(x, 0x1f8); }

// A cell that no environment occupies gets no remap values from computeVariablesForRemap
// (PrepareRemap.cc:100-166 loop over environment cells): its U is 0 and its Phi is the one
// the last sweep of the previous remap left, U / sum V_k (RemapADIService.cc:493-538).
// Without pente-borne the remap vector written for such a cell holds that Phi, read by the
// first sweep with a unit denominator, and the sweep starts its own U from 0.
template <int M>
__device__ __forceinline__ void empty_cell_phi(const MhDev& S, long c, double* u_out) {
  const long nc = S.g.nc;
  const double* __restrict__ Ulast = (S.nsweep & 1) ? S.Ub : S.Ua;
  double sv = 0.;
  for (int kk = 0; kk < M; ++kk) sv += Ulast[kk * nc + c];
  for (int v = 0; v <= 3 * M; ++v) u_out[v] = Ulast[v * nc + c] / sv;
}

// The remap vector of cell c (environments mk) to the first buffer.
template <int M>
__device__ __forceinline__ void store_remap_vector(const MhDev& S, long c, unsigned mk, const double* u) {
  double* __restrict__ U = S.Ua;
  const long nc = S.g.nc;
  if (M > 1 && S.pm[0]) {
    const unsigned held = mk ? mk : (1u << M) - 1u;  // an empty cell holds a phi of every slot
    const unsigned old = S.pm[0][c];
#pragma unroll
    for (int v = 0; v < 3 * M; ++v)
      if (((held | old) >> (v % M)) & 1u) U[v * nc + c] = u[v];
    U[3 * M * nc + c] = u[3 * M];
    S.pm[0][c] = (uint8_t)held;
  } else {
#pragma unroll
    for (int v = 0; v <= 3 * M; ++v) U[v * nc + c] = u[v];
  }
}

// ComputeGeometricValues (:1097-1253) + UpdateDensity (:1267-1316) +
// ComputeArtificialViscosity (:386-426) + UpdateEnergyAndPressure (:1430-1480) for one cell.
// With remap: writes U (V_k, V_k rho_k, V_k rho_k e_k, V q; PrepareRemap.cc:100-136), V, L.
// Without: applies the EOS and the mean pressure and writes the CFL candidate.
// The cell's work once its node coordinates x (at this cycle's Lagrangian positions) are
// in registers; returns the CFL candidate of the Lagrange-only loop.
// The cell's own state read by the Lagrange step.  2D kernels are latency-bound: all loads go out
// together (33.9 -> 27.3 us on 1023x1021, 8.9 -> 7.3 us on 200x10).  3D ones are bound by the FP64 issue
// of the volume, which takes all 160 registers of three wavefronts per SIMD, so the state is read
// after it (216 -> 192 us on 256x128x128, 304 -> 257 us on 192^3, 55 -> 46 us on 128x96x64 without remap).
struct CellPre {
  uint8_t mk;
  double cs, rho_n, Mc, e_c, p_c;
  double vmax2;  // Lagrange-only loop: the square of the largest node speed, for the CFL candidate
};
__device__ __forceinline__ void cell_pre_load(const MhDev& S, long c, CellPre& pr) {
  pr.mk = S.mask[c];
  pr.cs = S.c[c];
  pr.rho_n = S.rho[c];
  pr.Mc = S.M[c];
  pr.e_c = S.e[c];
  pr.p_c = S.p[c];
}

// VGIVEN: the volume Vgiven was formed by the caller (the 3D kernels but CSTS); x is unused.
template <int DIM, int M, int CSTS = 0, int VGIVEN = 0, int REMAP = 0>
__device__ __forceinline__ double cell_lag_core(const MhDev& S, long c, long b, const D3* x, const CellPre& pre,
                                                double Vgiven = 0.) {
  // REMAP: known at compile time to be the Lagrange step of the remap loop (1: with_proj set,
  // sans_lagrange and staged not) or of the Lagrange-only loop (2), so the other branches are
  // not compiled.  Staged mode takes the
  // Lagrange-only branch (state and EOS written back) and k_prepare_remap forms U later.
  const bool with_proj = REMAP == 1 ? true : (REMAP == 2 ? false : S.with_proj != 0 && !S.staged);
  const bool sans_lagrange = REMAP ? false : (S.sans_lagrange != 0);
  constexpr int NV = 3 * M + 1;
  double dxs = 1.79769313486231570815e+308;
  {
    const uint8_t mk = pre.mk;
    const double cs = pre.cs;
    const double rho_n = pre.rho_n;
    const double Mc = pre.Mc;
    const double e_c = pre.e_c;
    const double p_c = pre.p_c;
    D3 qv[8];
    double V;
    if constexpr (VGIVEN) {
      V = Vgiven;
    } else if (DIM == 3) {
      cqs_hex(x, qv);
      V = cell_volume<8>(x, qv, 3);
    } else {
      cqs_quad(x, qv);
      V = cell_volume<4>(x, qv, 2);
    }
    if (V < 0.) S.err[0] = MH_ERR_NEG_VOLUME;
    // the other characteristic lengths come from k_cell_length, launched just before
    const double L = S.lc == MH_L_RACINE_CUBIQUE_VOLUME ? (DIM == 3 ? mh_pow_third(V) : mh_pow_half(V)) : S.L[c];
    if (sans_lagrange) {
      // advection mode: no density, pseudo or energy update (MahycoModule.cc:1271, 389,
      // 1433); the remap vector of PrepareRemap.cc:100-155 from the stored state
      const long nc = S.g.nc;
      double u_out[NV];
      for (int v = 0; v < NV; ++v) u_out[v] = 0.;
      if (__popc(mk) == 1) {
        const int ke = __ffs(mk) - 1;
        const double rho = rho_n, e = e_c;
        u_out[ke] = V;
        u_out[M + ke] = V * rho;
        u_out[2 * M + ke] = V * rho * e;
        if (S.pb) {
          S.phi0[ke * nc + c] = S.fg[c];
          S.phi0[(M + ke) * nc + c] = rho;
          S.phi0[(2 * M + ke) * nc + c] = e;
        }
      } else {
        for (int kk = 0; kk < M; ++kk) {
          if (!((mk >> kk) & 1)) continue;
          const long o = kk * nc + c;
          const double Vk = S.fk[o] * V;
          u_out[kk] = Vk;
          u_out[M + kk] = Vk * S.rhok[o];
          u_out[2 * M + kk] = Vk * S.rhok[o] * S.ek[o];
          if (S.pb) {
            S.phi0[o] = S.fk[o];
            S.phi0[(M + kk) * nc + c] = S.rhok[o];
            S.phi0[(2 * M + kk) * nc + c] = S.ek[o];
          }
        }
      }
      u_out[3 * M] = V * S.q[c];
      if (S.pb && mk) S.phi0[3 * M * nc + c] = S.q[c];
      if (!mk && !S.pb && S.nsweep > 0) empty_cell_phi<M>(S, c, u_out);
      store_remap_vector<M>(S, c, mk, u_out);
      S.Vl[c] = V;
      S.L[c] = L;
      return dxs;
    }
    const double dt = S.sc->dt;
    const double rho = Mc / V;
    const double tau = 0.5 * (1.0 / rho_n + 1.0 / rho);
    const double divu = 1.0 / dt * (1.0 / rho - 1.0 / rho_n) / tau;
    const long nc = S.g.nc;
    double u_out[NV];
    for (int v = 0; v < NV; ++v) u_out[v] = 0.;
    if (__popc(mk) == 1) {
      const int ke = __ffs(mk) - 1;
      // by selects: an index that varies over the lanes would be another load to wait for
      MhEosCoef ep{S.env[0].gamma, S.env[0].pinf, S.env[0].a1, S.env[0].a2, S.env[0].stiffened};
#pragma unroll
      for (int kk = 1; kk < M; ++kk) {
        const MhEnvParam& o = S.env[kk];
        ep.gamma = kk == ke ? o.gamma : ep.gamma;
        ep.pinf = kk == ke ? o.pinf : ep.pinf;
        ep.a1 = kk == ke ? o.a1 : ep.a1;
        ep.a2 = kk == ke ? o.a2 : ep.a2;
        ep.stiffened = kk == ke ? o.stiffened : ep.stiffened;
      }
      double q = 0.;
      if (divu < 0.0) q = 1. / tau * (-ep.a1 * L * cs * divu + ep.a2 * L * L * divu * divu);
      double e;
      if constexpr (CSTS) {
        double cn1, cn, cdn, cvon;
        csts_work<DIM>(S, b, qv, cn1, cn, cdn, cvon);
        e = csts_e(ep, e_c, Mc, rho, p_c, S.q[c], csts_qnm1(S, c, ke, false), q, cn1, cn, cdn, cvon);
      } else {
        e = lag_energy(S, ep, e_c, p_c, rho, rho_n, q);
      }
      if (with_proj) {
        for (int kk = 0; kk < M; ++kk)
          if (kk == ke) {
            u_out[kk] = V;
            u_out[M + kk] = V * rho;
            u_out[2 * M + kk] = V * rho * e;
          }
        u_out[3 * M] = V * q;
        if (S.q_frozen) S.q[c] = q;  // the Lagrangian pseudo, for the remap's unswept V q slot
        if (CSTS) {  // SaveValuesAtN of the pseudo; this cycle's for the forward velocity step
          S.qm1[c] = S.q[c];
          S.q[c] = q;
        }
        if (S.pb) {  // pente-borne phi of the first sweep (PrepareRemap.cc:138-155)
          S.phi0[ke * nc + c] = S.fg[c];
          S.phi0[(M + ke) * nc + c] = rho;
          S.phi0[(2 * M + ke) * nc + c] = e;
          S.phi0[3 * M * nc + c] = q;
        }
      } else {
        double p, cc;
        eos(ep, rho, e, p, cc);
        if (CSTS) S.qm1[c] = S.q[c];
        S.rho[c] = rho;
        S.e[c] = e;
        S.p[c] = p;
        S.c[c] = cc;
        S.q[c] = q;
        if (REMAP == 2 || !S.staged) dxs = L / (cc + sqrt(pre.vmax2));
      }
    } else {
      double fk[M], rk[M], qk[M], ek[M], Vk[M];
      double qsum = 0., esum = 0.;
      double cn1 = 0., cn = 0., cdn = 0., cvon = 0.;
      if constexpr (CSTS) csts_work<DIM>(S, b, qv, cn1, cn, cdn, cvon);
      for (int kk = 0; kk < M; ++kk) {
        if (!((mk >> kk) & 1)) continue;
        const MhEnvParam& ep = S.env[kk];
        const long o = kk * nc + c;
        fk[kk] = S.fk[o];
        Vk[kk] = fk[kk] * V;
        const double rkn = S.rhok[o];
        rk[kk] = S.Mk[o] / Vk[kk];
        const double tk = 0.5 * (1.0 / rkn + 1.0 / rk[kk]);
        qk[kk] = 0.;
        if (divu < 0.0) qk[kk] = 1. / tk * (-ep.a1 * L * cs * divu + ep.a2 * L * L * divu * divu);
        if constexpr (CSTS) {
          // with remap: the history of the remap (qe, csts_qnm1); without: the environment's own
          const double qn = with_proj ? S.qe[c] : S.qkn[o];
          const double qnm1 = with_proj ? csts_qnm1(S, c, kk, true) : S.qknm1[o];
          ek[kk] = csts_e(ep, S.ek[o], S.Mk[o], rk[kk], S.pk[o], qn, qnm1, qk[kk], cn1, cn, cdn, cvon);
          if (!with_proj) {
            S.qknm1[o] = qn;
            S.qkn[o] = qk[kk];
          }
        } else
          ek[kk] = lag_energy(S, ep, S.ek[o], S.pk[o], rk[kk], rkn, qk[kk]);
      }
      for (int kk = 0; kk < M; ++kk)
        if ((mk >> kk) & 1) qsum += qk[kk] * fk[kk];
      for (int kk = 0; kk < M; ++kk)
        if ((mk >> kk) & 1) esum += S.chik[kk * nc + c] * ek[kk];
      if (with_proj) {
        for (int kk = 0; kk < M; ++kk) {
          if (!((mk >> kk) & 1)) continue;
          u_out[kk] = Vk[kk];
          u_out[M + kk] = Vk[kk] * rk[kk];
          u_out[2 * M + kk] = Vk[kk] * rk[kk] * ek[kk];
        }
        u_out[3 * M] = V * qsum;
        if (S.q_frozen) S.q[c] = qsum;
        if (CSTS) {  // as for a single-environment cell
          S.qm1[c] = S.q[c];
          S.q[c] = qsum;
        }
        if (S.pb) {
          for (int kk = 0; kk < M; ++kk) {
            if (!((mk >> kk) & 1)) continue;
            S.phi0[kk * nc + c] = fk[kk];
            S.phi0[(M + kk) * nc + c] = rk[kk];
            S.phi0[(2 * M + kk) * nc + c] = ek[kk];
          }
          if (mk) S.phi0[3 * M * nc + c] = qsum;  // an empty cell keeps the last sweep's
        }
      } else {
        double ps = 0., cmix = 0.;
        const double opt = S.vitson_max ? 1. : 0.;
        for (int kk = 0; kk < M; ++kk) {
          if (!((mk >> kk) & 1)) continue;
          double p, cc;
          eos(S.env[kk], rk[kk], ek[kk], p, cc);
          const long o = kk * nc + c;
          S.rhok[o] = rk[kk];
          S.ek[o] = ek[kk];
          S.pk[o] = p;
          ps += fk[kk] * p;
          cmix = opt * ((cc < cmix) ? cmix : cc);  // std::max(c_k, c)
          cmix += (1. - opt) * fk[kk] * cc;
        }
        if (CSTS) S.qm1[c] = S.q[c];
        S.rho[c] = rho;
        S.e[c] = esum;
        S.p[c] = ps;
        S.c[c] = cmix;
        S.q[c] = qsum;
        if (REMAP == 2 || !S.staged) dxs = L / (cmix + sqrt(pre.vmax2));
      }
    }
    if (with_proj && !mk && !S.pb && S.nsweep > 0) empty_cell_phi<M>(S, c, u_out);
    if (with_proj) store_remap_vector<M>(S, c, mk, u_out);
    S.Vl[c] = V;
    S.L[c] = L;
  }
  return dxs;
}

template <int DIM, int M, int CSTS = 0, int REMAP = 0>
__device__ __forceinline__ void k_cell_lag_body(const MhDev& S, int lb) {
  const long c = lb * (long)blockDim.x + threadIdx.x;
  const bool halted = mh_halted(S.sc);
  const bool active = c < S.g.nc && !halted;
  double dxs = 1.79769313486231570815e+308;
  if (c < S.g.nc) {
    const int nx = S.g.nx, ny = S.g.ny;
    const int i = (int)(c % nx);
    const long r = c / nx;
    const int j = (int)(r % ny);
    const int k = (int)(r / ny);
    const long b = i + (long)S.g.nnx * (j + (long)S.g.nny * k);
    CellPre pre;
    constexpr bool VOL = DIM == 3 && !CSTS;
    double V = 0.;
    D3 x[8];
    cell_nodes<DIM>(S, b, S.xlc, x);
    if (VOL) V = hex_volume(x);
    cell_pre_load(S, c, pre);
    if (REMAP == 2 || (!REMAP && !S.with_proj)) pre.vmax2 = cell_vmax2<DIM>(S, b);
    if (active) dxs = cell_lag_core<DIM, M, CSTS, VOL, REMAP>(S, c, b, x, pre, V);
  }
  if (REMAP == 2 || (!REMAP && !S.with_proj)) block_min_store(dxs, active, S.partial, lb);
}
// computeVariablesForRemap (PrepareRemap.cc:100-155) from the stored Lagrangian state, for
// staged mode: the cell kernel wrote the state of UpdateEnergyAndPressure and the caller may
// have changed it.  U = (V_k, V_k rho_k, V_k rho_k e_k, V q) with V_k = f_k V for a cell of
// several environments and V for a single-environment cell, the pente-borne phi of the first
// sweep, and an empty cell's phi as the fused cell kernel forms them (same operations, so an
// unchanged state gives the fused kernel's bits).
template <int DIM, int M>
__device__ __forceinline__ void k_prepare_remap_body(const MhDev& S, int lb) {
  const long c = lb * (long)blockDim.x + threadIdx.x;
  if (c >= S.g.nc || mh_halted(S.sc)) return;
  constexpr int NV = 3 * M + 1;
  const long nc = S.g.nc;
  const uint8_t mk = S.mask[c];
  const double V = S.Vl[c];
  const double q = S.q[c];
  double u_out[NV];
  for (int v = 0; v < NV; ++v) u_out[v] = 0.;
  if (__popc(mk) == 1) {
    const int ke = __ffs(mk) - 1;
    const double rho = S.rho[c], e = S.e[c];
    for (int kk = 0; kk < M; ++kk)
      if (kk == ke) {
        u_out[kk] = V;
        u_out[M + kk] = V * rho;
        u_out[2 * M + kk] = V * rho * e;
      }
    if (S.pb) {
      S.phi0[ke * nc + c] = S.fg[c];
      S.phi0[(M + ke) * nc + c] = rho;
      S.phi0[(2 * M + ke) * nc + c] = e;
      S.phi0[3 * M * nc + c] = q;
    }
  } else {
    for (int kk = 0; kk < M; ++kk) {
      if (!((mk >> kk) & 1)) continue;
      const long o = kk * nc + c;
      const double Vk = S.fk[o] * V;
      u_out[kk] = Vk;
      u_out[M + kk] = Vk * S.rhok[o];
      u_out[2 * M + kk] = Vk * S.rhok[o] * S.ek[o];
      if (S.pb) {
        S.phi0[o] = S.fk[o];
        S.phi0[(M + kk) * nc + c] = S.rhok[o];
        S.phi0[(2 * M + kk) * nc + c] = S.ek[o];
      }
    }
    if (S.pb && mk) S.phi0[3 * M * nc + c] = q;
  }
  u_out[3 * M] = V * q;
  if (!mk && !S.pb && S.nsweep > 0) empty_cell_phi<M>(S, c, u_out);
  store_remap_vector<M>(S, c, mk, u_out);
}

// 3D cell kernel of the remap loop with the node neighbourhood staged in LDS: a block owns
// MH_CT_X x MH_CT_Y cells of MH_CT_K consecutive z planes and marches up in z.  The node
// coordinates of a tile plane ((MH_CT_X+1) x (MH_CT_Y+1) nodes, every node read from HBM once
// per tile instead of by each of its cells) go to a rolling set of three LDS planes: the two a
// cell plane needs, and the next one, whose global loads are issued before the cell plane's
// arithmetic and written to LDS after it.  The cell's own state is also loaded one plane ahead.
// The volume takes its nodes from LDS; everything else is cell_lag_core.
#define MH_CT_X 64
#define MH_CT_Y (MH_BLOCK / MH_CT_X)
#define MH_CT_K 8  // cell planes per tile by default (MhDev::ct_k)
#define MH_CT_NX (MH_CT_X + 1)
#define MH_CT_NP (MH_CT_NX * (MH_CT_Y + 1))  // nodes of a tile plane
#define MH_CT_PER ((MH_CT_NP + MH_BLOCK - 1) / MH_BLOCK)  // node entries loaded per thread
#ifndef MH_CT_MIN_WAVES
#define MH_CT_MIN_WAVES 2
#endif

// Volume of the cell whose node 0 is entry s of the bottom plane.
__device__ __forceinline__ double hex_volume_lds(const double* bot, const double* top, int s) {
  const int o[4] = {s, s + 1, s + 1 + MH_CT_NX, s + MH_CT_NX};
  D3 x[8];
#pragma unroll
  for (int l = 0; l < 4; ++l) {
    x[l] = d3(bot[o[l]], bot[MH_CT_NP + o[l]], bot[2 * MH_CT_NP + o[l]]);
    x[l + 4] = d3(top[o[l]], top[MH_CT_NP + o[l]], top[2 * MH_CT_NP + o[l]]);
  }
  return hex_volume(x);
}

template <int M>
__device__ __forceinline__ void k_cell_lag3_tiled_body(const MhDev& S, int bx, int by, int bz) {
  __shared__ double pl[3][3 * MH_CT_NP];
  if (mh_halted(S.sc)) return;
  const int tid = threadIdx.x, tx = tid % MH_CT_X, ty = tid / MH_CT_X;
  const int nx = S.g.nx, ny = S.g.ny, nz = S.g.nz;
  const int i0 = bx * MH_CT_X, j0 = by * MH_CT_Y, k0 = bz * S.ct_k;
  const int kend = min(k0 + S.ct_k, nz);
  const int i = i0 + tx, j = j0 + ty;
  const bool ok = i < nx && j < ny;
  const long nnx = S.g.nnx, nnxy = (long)S.g.nnx * S.g.nny;
  // the node entries of a tile plane this thread loads
  double nv[MH_CT_PER][3];
  auto fetch = [&](int kn) {
#pragma unroll
    for (int r = 0; r < MH_CT_PER; ++r) {
      const int e = tid + r * MH_BLOCK;
      const int gi = i0 + e % MH_CT_NX, gj = j0 + e / MH_CT_NX;
      if (e < MH_CT_NP && gi <= nx && gj <= ny) {
        const long n = gi + nnx * gj + nnxy * kn;
        nv[r][0] = S.xlc[0][n];
        nv[r][1] = S.xlc[1][n];
        nv[r][2] = S.xlc[2][n];
      }
    }
  };
  auto put = [&](double* P) {
#pragma unroll
    for (int r = 0; r < MH_CT_PER; ++r) {
      const int e = tid + r * MH_BLOCK;
      if (e < MH_CT_NP) {
        P[e] = nv[r][0];
        P[MH_CT_NP + e] = nv[r][1];
        P[2 * MH_CT_NP + e] = nv[r][2];
      }
    }
  };
  fetch(k0);
  put(pl[0]);
  fetch(k0 + 1);
  put(pl[1]);
  const long cplane = (long)nx * ny;
  const long c0 = i + (long)nx * j;
  CellPre cur, nxt;
  if (ok && k0 < kend) cell_pre_load(S, c0 + cplane * k0, nxt);
  __syncthreads();
  for (int k = k0; k < kend; ++k) {
    const int sl = k - k0;
    const bool more = k + 1 < kend;
    if (more) fetch(k + 2);  // node plane of the next step, into registers now
    cur = nxt;
    if (ok && more) cell_pre_load(S, c0 + cplane * (k + 1), nxt);
    if (ok) {
      const long c = c0 + cplane * k;
      const long b = i + nnx * j + nnxy * k;
      const double V = hex_volume_lds(pl[sl % 3], pl[(sl + 1) % 3], tx + MH_CT_NX * ty);
      (void)cell_lag_core<3, M, 0, 1, 1>(S, c, b, nullptr, cur, V);
    }
    if (more) put(pl[(sl + 2) % 3]);
    __syncthreads();
  }
}

// The characteristic length of the other options, written to L before the cell kernel
// (which then reads it instead of forming V^(1/d)): one thread per cell.
template <int DIM>
__device__ __forceinline__ void k_cell_length_body(const MhDev& S, int lb) {
  const long c = lb * (long)blockDim.x + threadIdx.x;
  if (c >= S.g.nc || mh_halted(S.sc)) return;
  const int nx = S.g.nx, ny = S.g.ny;
  const int i = (int)(c % nx);
  const long r = c / nx;
  const int j = (int)(r % ny);
  const int k = (int)(r / ny);
  const long b = i + (long)S.g.nnx * (j + (long)S.g.nny * k);
  D3 x[8];
  cell_nodes<DIM>(S, b, S.xlc, x);
  S.L[c] = char_length_alt<DIM>(S.lc, x);
}

// The Lagrange step of the remap loop and that of the Lagrange-only loop: an instance each, without
// one another's registers and those of staged mode and advection, which k_cell_lag keeps.
// CSTS (with remap): its own instance, so that the other cell kernels do not carry the
// corner-work registers
template <int DIM, int M>
__device__ __forceinline__ void k_cell_lag_remap_body(const MhDev& S, int lb) {
  k_cell_lag_body<DIM, M, 0, 1>(S, lb);
}
template <int DIM, int M>
__device__ __forceinline__ void k_cell_lag_only_body(const MhDev& S, int lb) {
  k_cell_lag_body<DIM, M, 0, 2>(S, lb);
}
template <int DIM, int M>
__device__ __forceinline__ void k_cell_lag_csts_body(const MhDev& S, int lb) {
  k_cell_lag_body<DIM, M, 1>(S, lb);
}

// ----------------------------------------------------------------------------- remap sweeps
// Lagrangian cell centre, direction-D component (UpdatePosition, MahycoModule.cc:743-750).
template <int DIM, int D>
__device__ __forceinline__ double cell_centre_d(const MhDev& S, long b) {
  const long nnx = S.g.nnx, nnxy = (long)S.g.nnx * S.g.nny;
  const double* xd = S.xlc[D];
  double s = 0.;
  s += xd[b];
  s += xd[b + 1];
  s += xd[b + 1 + nnx];
  s += xd[b + nnx];
  if (DIM == 3) {
    s += xd[b + nnxy];
    s += xd[b + 1 + nnxy];
    s += xd[b + 1 + nnx + nnxy];
    s += xd[b + nnx + nnxy];
    return 0.125 * s;
  }
  return 0.25 * s;
}

// Lagrangian quantities of the face of direction D whose first node is f0
// (computeFaceQuantitesForRemap, PrepareRemap.cc:18-59): projected area on D,
// centre coordinate along D, normal velocity.  Face nodes in Arcane order.
template <int DIM, int D>
__device__ __forceinline__ void face_quant(const MhDev& S, long f0, double& area, double& xf, double& vf) {
  const long nnx = S.g.nnx, nnxy = (long)S.g.nnx * S.g.nny;
  if (DIM == 3) {
    long nd[4];
    if (D == 0) { nd[0] = f0; nd[1] = f0 + nnx; nd[2] = f0 + nnx + nnxy; nd[3] = f0 + nnxy; }
    else if (D == 1) { nd[0] = f0; nd[1] = f0 + 1; nd[2] = f0 + 1 + nnxy; nd[3] = f0 + nnxy; }
    else { nd[0] = f0; nd[1] = f0 + 1; nd[2] = f0 + 1 + nnx; nd[3] = f0 + nnx; }
    // every load first: the branch below would split them into two rounds
    const double* ud = S.u[D];
    const double u0 = ud[nd[0]], u1 = ud[nd[1]], u2 = ud[nd[2]], u3 = ud[nd[3]];
    const D3 x0 = load3(S.xlc, nd[0]), x1 = load3(S.xlc, nd[1]);
    const D3 x2 = load3(S.xlc, nd[2]), x3 = load3(S.xlc, nd[3]);
    const D3 v1 = x2 - x0, v2 = x3 - x1;
    if (D == 0) area = 0.5 * fabs(v1.y * v2.z - v1.z * v2.y);
    else if (D == 1) area = 0.5 * fabs(v2.x * v1.z - v2.z * v1.x);
    else area = 0.5 * fabs(v1.x * v2.y - v1.y * v2.x);
    const double xa = D == 0 ? x0.x : D == 1 ? x0.y : x0.z;
    const double xb = D == 0 ? x1.x : D == 1 ? x1.y : x1.z;
    const double xc = D == 0 ? x2.x : D == 1 ? x2.y : x2.z;
    const double xd = D == 0 ? x3.x : D == 1 ? x3.y : x3.z;
    double s = 0.;
    s += 0.25 * xa;
    s += 0.25 * xb;
    s += 0.25 * xc;
    s += 0.25 * xd;
    xf = s;
    double us = 0.;
    if (S.csts) {  // the mean of n and n+1 (PrepareRemap.cc:236-240)
      const double* vd = S.un[D];
      us += 0.5 * (u0 + vd[nd[0]]);
      us += 0.5 * (u1 + vd[nd[1]]);
      us += 0.5 * (u2 + vd[nd[2]]);
      us += 0.5 * (u3 + vd[nd[3]]);
    } else {
      us += u0;
      us += u1;
      us += u2;
      us += u3;
    }
    vf = 0.25 * us;
  } else {
    const long n1 = D == 0 ? f0 + nnx : f0 + 1;
    const double u0 = S.u[D][f0], u1 = S.u[D][n1];
    const double dxv = S.xlc[0][n1] - S.xlc[0][f0];
    const double dyv = S.xlc[1][n1] - S.xlc[1][f0];
    area = D == 0 ? fabs(dyv) : fabs(dxv);
    const double* xd = S.xlc[D];
    double s = 0.;
    s += 0.5 * xd[f0];
    s += 0.5 * xd[n1];
    xf = s;
    double us = 0.;
    if (S.csts) {
      const double* vd = S.un[D];
      us += 0.5 * (u0 + vd[f0]);
      us += 0.5 * (u1 + vd[n1]);
    } else {
      us += u0;
      us += u1;
    }
    vf = 0.5 * us;
  }
}

// One ADI direction, cell part: computeGradPhiFace (RemapADIService.cc:119-149),
// computeGradPhiCell + computeAndLimitGradPhi (:161-267, UtilesRemap.cc:325-357),
// computeUpwindFaceQuantitiesForProjection (:279-383) and computeUremap (:395-575).
// Phi of the stencil is rebuilt from U (U / V before the first sweep, U / sum V_k after).
template <int DIM, int D, int M, int LIM>
__device__ __forceinline__ void k_sweep_cell_body(const MhDev& S, int lb, int usel, int first) {
  const double* __restrict__ Uin = usel ? S.Ub : S.Ua;
  double* __restrict__ Uout = usel ? S.Ua : S.Ub;
  double* __restrict__ dflux = S.dflux;
  constexpr int NV = 3 * M + 1;
  const long c = lb * (long)blockDim.x + threadIdx.x;
  if (c >= S.g.nc) return;
  if (mh_halted(S.sc)) return;
  const bool own = !(first && S.mask[c] == 0);  // an empty cell's U starts from 0 (its Phi is stale)
  const int nx = S.g.nx, ny = S.g.ny;
  const int i = (int)(c % nx);
  const long r = c / nx;
  const int j = (int)(r % ny);
  const int k = (int)(r / ny);
  const int a = D == 0 ? i : D == 1 ? j : k;
  const int na = D == 0 ? nx : D == 1 ? ny : S.g.nz;
  const long sD = D == 0 ? 1 : D == 1 ? (long)nx : (long)nx * ny;
  const long nD = D == 0 ? 1 : D == 1 ? (long)S.g.nnx : (long)S.g.nnx * S.g.nny;
  const long b = i + (long)S.g.nnx * (j + (long)S.g.nny * k);
  const long nc = S.g.nc;
  const double dt = S.sc->dt;
  // per stencil cell (offsets -2..2 along D): existence, Phi denominator, centre along D
  double den[5], xc[5];
  bool valid[5];
#pragma unroll
  for (int o = -2; o <= 2; ++o) {
    const int bb = a + o;
    valid[o + 2] = (bb >= 0 && bb < na);
    den[o + 2] = 1.;
    xc[o + 2] = 0.;
    if (valid[o + 2]) {
      const long cc = c + o * sD;
      if (first) {
        den[o + 2] = S.mask[cc] ? S.Vl[cc] : 1.;  // an empty cell holds Phi itself
      } else {
        double sv = 0.;
        for (int kk = 0; kk < M; ++kk) sv += Uin[kk * nc + cc];
        den[o + 2] = sv;
      }
      xc[o + 2] = cell_centre_d<DIM, D>(S, b + o * nD);
    }
  }
  // face f lies between offsets f-2 and f-1; Delta x along D (boundary faces: none)
  double dxf[4];
#pragma unroll
  for (int f = 0; f < 4; ++f) dxf[f] = (valid[f] && valid[f + 1]) ? xc[f + 1] - xc[f] : 0.;
  // the two faces of the cell along D: s = 0 back (outer normal -e_D), s = 1 front (+e_D)
  bool inner[2], upprev[2];
  double area[2], vf[2], hup[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    inner[s] = s == 0 ? (a > 0) : (a < na - 1);
    area[s] = 0.;
    vf[s] = 0.;
    hup[s] = 0.;
    upprev[s] = false;
    if (!inner[s]) continue;
    double xf;
    face_quant<DIM, D>(S, b + s * nD, area[s], xf, vf[s]);
    upprev[s] = vf[s] * dxf[s + 1] > 0.0;  // upwind cell: the one behind the face
    hup[s] = (double)S.order2 * (xf - (upprev[s] ? xc[s + 1] : xc[s + 2]));
  }
  // cell faces in Arcane local order: 3D min face first; 2D x: max face first
  const int s0 = (DIM == 2 && D == 0) ? 1 : 0, s1 = 1 - s0;
  const double od[2] = {-1., 1.};
  for (int v = 0; v < NV; ++v) {
    double phi[5];
#pragma unroll
    for (int o = 0; o < 5; ++o) phi[o] = valid[o] ? Uin[v * nc + c + (o - 2) * sD] / den[o] : 0.;
    double gface[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) gface[f] = (valid[f] && valid[f + 1]) ? (phi[f + 1] - phi[f]) / dxf[f] : 0.;
    double grad[3];
#pragma unroll
    for (int o = 0; o < 3; ++o) {
      double g = 0.;
      if (S.order2 && valid[o + 1]) {
        const double gb = gface[o], gf = gface[o + 1];
        if (gb != 0.) g += 0.5 * (mh_limiter<LIM>(S.limiter, gf / gb) * gb);
        if (gf != 0.) g += 0.5 * (mh_limiter<LIM>(S.limiter, gb / gf) * gf);
      }
      grad[o] = g;
    }
    double flux[2] = {0., 0.};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (!inner[s]) continue;
      // Phi_face = Phi_up + h grad_up, up = offset s-1 (behind) or s (ahead)
      const double pu = upprev[s] ? phi[s + 1] : phi[s + 2];
      const double gu = upprev[s] ? grad[s] : grad[s + 1];
      const double pf = pu + hup[s] * gu;
      flux[s] = od[s] * vf[s] * area[s] * dt * pf;
    }
    double ff = 0.;
    if (inner[s0]) ff += flux[s0];
    if (inner[s1]) ff += flux[s1];
    double un = (own ? Uin[v * nc + c] : 0.) - ff;
    if (v >= M && v < 2 * M) {
      double dd = 0.;
      if (inner[s0]) dd += 0.5 * flux[s0] * od[s0];
      if (inner[s1]) dd += 0.5 * flux[s1] * od[s1];
      dflux[(v - M) * nc + c] = dd;
    }
    if (v >= M && v < 3 * M && un < 0.) un = 0.;  // computeUremap clamps, :465-485
    Uout[v * nc + c] = un;
  }
  if (S.pm[0]) S.pm[usel ? 0 : 1][c] = 0xff;
}

// Segments of one line of a marching sweep: n cells or nodes split into ceil(n / len) segments whose
// lengths differ by at most one, so that no line ends in a short segment that costs a whole pass of threads.
MH_HD int march_nseg(int n, int len) { return (n + len - 1) / len; }
// Segments of `len` cells of a line of na cells.
MH_HD int seg_count(int na, int len) { return (na + len - 1) / len; }

// ----------------------------------------------------------------------------- order-3 remap
// Lagrangian centre of the face of direction D whose first node is f0, all three components,
// summed over the face nodes in Arcane order as computeFaceQuantitesForRemap does
// (PrepareRemap.cc:18-59): 0 + w x_0 + w x_1 (+ w x_2 + w x_3), w = 1 / nodes.
template <int DIM, int D>
__device__ __forceinline__ D3 face_centre(const MhDev& S, long f0) {
  const long nnx = S.g.nnx, nnxy = (long)S.g.nnx * S.g.nny;
  double r[3] = {0., 0., 0.};
  if (DIM == 3) {
    long nd[4];
    if (D == 0) { nd[0] = f0; nd[1] = f0 + nnx; nd[2] = f0 + nnx + nnxy; nd[3] = f0 + nnxy; }
    else if (D == 1) { nd[0] = f0; nd[1] = f0 + 1; nd[2] = f0 + 1 + nnxy; nd[3] = f0 + nnxy; }
    else { nd[0] = f0; nd[1] = f0 + 1; nd[2] = f0 + 1 + nnx; nd[3] = f0 + nnx; }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      double s = 0.;
#pragma unroll
      for (int l = 0; l < 4; ++l) s += 0.25 * S.xlc[q][nd[l]];
      r[q] = s;
    }
  } else {
    const long n1 = D == 0 ? f0 + nnx : f0 + 1;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      double s = 0.;
      s += 0.5 * S.xlc[q][f0];
      s += 0.5 * S.xlc[q][n1];
      r[q] = s;
    }
  }
  return d3(r[0], r[1], r[2]);
}

__device__ __forceinline__ double norm3(D3 d) { return sqrt(d.x * d.x + d.y * d.y + d.z * d.z); }

// Cell widths of the order-3 remap, every direction at once (computeGradPhiFace,
// RemapADIService.cc:119-149): h_D(c) = sum over the inner faces of c normal to D of
// |x_f - x_c|, with the Lagrangian face and cell centres (full 3-vectors).  The Lagrangian
// mesh does not move during the remap, so one launch before the first sweep serves all of them.
template <int DIM>
__device__ __forceinline__ void k_hcell_body(const MhDev& S, int lb) {
  const long c = lb * (long)blockDim.x + threadIdx.x;
  if (c >= S.g.nc) return;
  if (mh_halted(S.sc)) return;
  const int nx = S.g.nx, ny = S.g.ny;
  const int i = (int)(c % nx);
  const long r = c / nx;
  const int j = (int)(r % ny);
  const int k = (int)(r / ny);
  const long b = i + (long)S.g.nnx * (j + (long)S.g.nny * k);
  const long nnx = S.g.nnx, nnxy = (long)S.g.nnx * S.g.nny;
  const D3 xc = d3(cell_centre_d<DIM, 0>(S, b), cell_centre_d<DIM, 1>(S, b),
                   DIM == 3 ? cell_centre_d<DIM, (DIM == 3 ? 2 : 0)>(S, b) : 0.);
  const long nc = S.g.nc;
  {
    double h = 0.;
    if (i > 0) h += norm3(face_centre<DIM, 0>(S, b) - xc);
    if (i < nx - 1) h += norm3(face_centre<DIM, 0>(S, b + 1) - xc);
    S.hc[c] = h;
  }
  {
    double h = 0.;
    if (j > 0) h += norm3(face_centre<DIM, 1>(S, b) - xc);
    if (j < ny - 1) h += norm3(face_centre<DIM, 1>(S, b + nnx) - xc);
    S.hc[nc + c] = h;
  }
  if (DIM == 3) {
    double h = 0.;
    if (k > 0) h += norm3(face_centre<DIM, (DIM == 3 ? 2 : 0)>(S, b) - xc);
    if (k < S.g.nz - 1) h += norm3(face_centre<DIM, (DIM == 3 ? 2 : 0)>(S, b + nnxy) - xc);
    S.hc[2 * nc + c] = h;
  }
}

// The order-3 face values (ComputeFluxOrdre3, Remap-ordre-3.cc:16-189) on a line of cells: the
// limited parabola of each cell from the gradients evaluate_grad of the cells and the edge values
// evaluate_ystar of the faces, a non-uniform 1D stencil.  Every factor that depends on the widths
// and the velocity alone is formed once per cell or face and serves all remap slots; the products
// and sums over the values keep the reference's order, so the results have its bits.
struct O3Grad {  // cell of width h0 between hm and hp
  double c, cp, cm;
};
__device__ __forceinline__ O3Grad o3_grad_coef(double hm, double h0, double hp) {
  O3Grad g;
  g.c = h0 / (hm + h0 + hp);
  g.cp = (2. * hm + h0) / (h0 + hp);
  g.cm = (h0 + 2. * hp) / (hm + h0);
  return g;
}
__device__ __forceinline__ double o3_grad(const O3Grad& g, double ym, double y0, double yp) {
  return g.c * (g.cp * (yp - y0) + g.cm * (y0 - ym));
}
struct O3Star {  // face between cells of widths hm and hp, their outer neighbours hmm and hpp
  double t, gp, gm, f, w;
};
__device__ __forceinline__ O3Star o3_star_coef(double hmm, double hm, double hp, double hpp) {
  O3Star c;
  c.t = (2. * hp * hm) / (hm + hp) * ((hmm + hm) / (2. * hm + hp) - (hpp + hp) / (2. * hp + hm));
  c.gp = -hm * (hmm + hm) / (2. * hm + hp);
  c.gm = hp * (hp + hpp) / (hm + 2. * hp);
  c.f = hm / (hm + hp);
  c.w = 1. / (hmm + hm + hp + hpp);
  return c;
}
__device__ __forceinline__ double o3_star(const O3Star& c, double ym, double yp, double gradm, double gradp) {
  const double d = yp - ym;
  const double t1 = c.t * d;
  const double t2 = c.gp * gradp + c.gm * gradm;
  return ym + c.f * d + c.w * (t1 + t2);
}
struct O3Face {  // displacement vdt = u_face dt through a face between widths hm and hp
  double x, q, k;  // 0.5 |vdt| / h, 1 - 2/3 |vdt| / h of the upwind cell, the weight of its slope limit
  int dir;         // 1: from behind, -1: from ahead, 0: none
};
__device__ __forceinline__ O3Face o3_face_coef(double vdt, double hm, double hp) {
  O3Face c;
  c.x = c.q = c.k = 0.;
  c.dir = vdt > 0. ? 1 : vdt < 0. ? -1 : 0;
  if (vdt > 0.) {
    const double num = vdt / hm;
    c.x = 0.5 * vdt / hm;
    c.q = 1. - 2. / 3. * vdt / hm;
    c.k = (1. - num) / num;
  } else if (vdt < 0.) {
    const double nup = vdt / hp;
    c.x = 0.5 * -vdt / hp;
    c.q = 1. - 2. / 3. * -vdt / hp;
    c.k = (1. + nup) / nup;
  }
  return c;
}
// The face value from the cells around the face (ymm, ym behind, yp, ypp ahead) and the edge values
// of the face behind, the face and the face ahead, clipped to the interval the upwind cell and its
// neighbours allow (Remap-ordre-3.cc:155-189).
__device__ __forceinline__ double o3_flux(const O3Face& c, double ymm, double ym, double yp, double ypp, double ysm,
                                          double ys, double ysp) {
  if (c.dir == 0) return 0.;
  double flux, b;
  if (c.dir > 0) {
    flux = ys - c.x * ((ys - ysm) - c.q * (6. * (ym - 0.5 * (ysm + ys))));
    b = ym + c.k * (ym - ymm);
  } else {
    flux = ys + c.x * ((ysp - ys) - c.q * (6. * (yp - 0.5 * (ys + ysp))));
    b = yp - c.k * (yp - ypp);
  }
  const double yu = c.dir > 0 ? ym : yp;
  const double a0 = amin(ym, yp), a1 = amax(ym, yp);
  const double b0 = amin(yu, b), b1 = amax(yu, b);
  double lo, hi;
  if ((a1 < b0) || (b1 < a0)) {
    lo = 0.;
    hi = 0.;
  } else {
    lo = amax(a0, b0);
    hi = amin(a1, b1);
  }
  if (flux < lo) flux = lo;
  if (flux > hi) flux = hi;
  return flux;
}

// One ADI direction, cell part, order 3 (computeUpwindFaceQuantitiesForProjection,
// RemapADIService.cc:319-379, then computeUremap :395-575): the face value of each variable
// comes from the six cells around the face along D, clamped at the mesh boundary.  Across a face
// whose two cells are not pure cells of one environment, the mass and energy face values are
// rebuilt from the upwind cell's ratios.  The flags of the two cells come from the sweep input
// (volume fractions > 0, :559-573), or in the first sweep of a cycle from the flags
// remapVariables left (RemapADIFinal.cc:124-145).  Phi as in k_sweep_cell_body.
//
// Each thread holds L cells of a line along D and three halo cells on each side in registers; a
// halo cell beyond the mesh is the boundary cell again, as the reference clamps.  With one cell per
// thread the kernel was bound by FP64 instructions: every face value was formed by both its cells,
// from eight gradients and six edge values with their divisions in every slot (7000-8500
// instructions per cell).  Two cells per thread share them, and the factors of the widths are
// formed once: 145 / 164 / 164 -> 54 / 64 / 64 us for x / y / z on 128x64x64 cells and two
// environments, at two wavefronts per SIMD (256 registers), now bound by latency at that occupancy;
// one cell per thread with the same factors takes 68 / 66 / 66 us.  Slots run environment by
// environment (volume, mass, energy, then V q), so that the face values the correction needs live
// for one environment only; groups e0 .. e1-1 of the m environments and V q (a small mesh shares
// them out over gridDim.y).
#define MH_O3_L 2  // cells along D per thread
template <int DIM, int D, int M, int L>
__device__ __forceinline__ void k_sweep_cell3_body(const MhDev& S, int lb, int usel, int first, int e0, int e1) {
  constexpr int R = L + 6;
  const double* __restrict__ Uin = usel ? S.Ub : S.Ua;
  double* __restrict__ Uout = usel ? S.Ua : S.Ub;
  const int nx = S.g.nx, ny = S.g.ny, nz = S.g.nz;
  const int na = D == 0 ? nx : D == 1 ? ny : nz;
  const int nseg = seg_count(na, L);
  const long g = lb * (long)blockDim.x + threadIdx.x;
  if (g >= S.g.nc / na * nseg) return;
  if (mh_halted(S.sc)) return;
  // threads run along x first (segments of it for D = 0), then over the segments along D
  int i, j, k, a0;
  if (D == 0) {
    a0 = (int)(g % nseg) * L;
    const int r = (int)(g / nseg);
    i = 0;
    j = r % ny;
    k = r / ny;
  } else {
    i = (int)(g % nx);
    const int r = (int)(g / nx);
    a0 = (r % nseg) * L;
    j = D == 1 ? 0 : r / nseg;
    k = D == 1 ? r / nseg : 0;
  }
  const long nc = S.g.nc;
  const long sD = D == 0 ? 1 : D == 1 ? (long)nx : (long)nx * ny;
  const long nD = D == 0 ? 1 : D == 1 ? (long)S.g.nnx : (long)S.g.nnx * S.g.nny;
  const long line = i + (long)nx * (j + (long)ny * k);  // cell and node of the line at 0
  const long nline = i + (long)S.g.nnx * (j + (long)S.g.nny * k);
  const double dt = S.sc->dt;
  // row r: the cell at a0 - 3 + r, clamped; face f: between rows f-1 and f
  int cs[R];  // offset of the row from the line
  MhRecip den[R];
  double h[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    cs[r] = min(max(a0 - 3 + r, 0), na - 1) * (int)sD;
    double d;
    if (first) {
      d = S.mask[line + cs[r]] ? S.Vl[line + cs[r]] : 1.;  // an empty cell holds Phi itself
    } else {
      d = 0.;
      for (int kk = 0; kk < M; ++kk) d += Uin[kk * nc + line + cs[r]];
    }
    den[r] = mh_denom(d);
    h[r] = S.hc[D * nc + line + cs[r]];
  }
  // flags of the cells beside the faces: rows 2 .. L+3
  int code[L + 2];
  if (first) {
#pragma unroll
    for (int o = 0; o < L + 2; ++o) code[o] = S.est[line + cs[o + 2]];
  } else {
#pragma unroll
    for (int o = 0; o < L + 2; ++o) {
      int cnt = 0, pur = -1;
      for (int v = 0; v < M; ++v)
        if (mh_ratio(Uin[v * nc + line + cs[o + 2]], den[o + 2]) > 0.) {
          cnt++;
          pur = v;
        }
      code[o] = cnt > 1 ? MH_EST_MIXED : pur;
    }
  }
  O3Grad cg[R];   // rows 1 .. R-2
  O3Star cst[R];  // faces 2 .. R-2
  O3Face cf[L + 1];
  double w[L + 1];
  bool vpure[L + 1];
#pragma unroll
  for (int r = 1; r < R - 1; ++r) cg[r] = o3_grad_coef(h[r - 1], h[r], h[r + 1]);
#pragma unroll
  for (int f = 2; f < R - 1; ++f) cst[f] = o3_star_coef(h[f - 2], h[f - 1], h[f], h[f + 1]);
#pragma unroll
  for (int s = 0; s <= L; ++s) {  // face s of the segment: behind cell a0 + s
    const int a = a0 + s;
    double vdt = 0.;
    w[s] = 0.;
    vpure[s] = code[s] == code[s + 1] && code[s] != MH_EST_MIXED;
    if (a > 0 && a < na) {
      double area, xf, vf;
      face_quant<DIM, D>(S, nline + a * nD, area, xf, vf);
      vdt = vf * dt;
      w[s] = vf * area * dt;
    }
    cf[s] = o3_face_coef(vdt, h[s + 2], h[s + 3]);
  }
  unsigned ownm = 0;  // bit o: the cell's own U enters its update (an empty cell's U starts from 0)
#pragma unroll
  for (int o = 0; o < L; ++o)
    if (!(first && S.mask[line + cs[o + 3]] == 0)) ownm |= 1u << o;

  double pf[L + 1], pu[L + 1];  // face value and upwind phi of the slot
  auto slot = [&](int v, double* u) {
    double y[R], gr[R], ys[R];
    bool bad = false;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const double uv = Uin[v * nc + line + cs[r]];
      bad |= den[r].bad;
      y[r] = mh_div(uv, den[r], bad);
      if (r >= 3 && r < 3 + L) u[r - 3] = uv;
    }
    if (__builtin_expect(bad, 0))
#pragma unroll
      for (int r = 0; r < R; ++r) y[r] = Uin[v * nc + line + cs[r]] / den[r].b;
#pragma unroll
    for (int r = 1; r < R - 1; ++r) gr[r] = o3_grad(cg[r], y[r - 1], y[r], y[r + 1]);
#pragma unroll
    for (int f = 2; f < R - 1; ++f) ys[f] = o3_star(cst[f], y[f - 1], y[f], gr[f - 1], gr[f]);
#pragma unroll
    for (int s = 0; s <= L; ++s) {
      pf[s] = o3_flux(cf[s], y[s + 1], y[s + 2], y[s + 3], y[s + 4], ys[s + 2], ys[s + 3], ys[s + 4]);
      pu[s] = cf[s].dir > 0 ? y[s + 2] : y[s + 3];
    }
  };
  auto store = [&](int v, const double* u, bool mass, bool clamp) {
#pragma unroll
    for (int o = 0; o < L; ++o) {
      const int a = a0 + o;
      if (a >= na) continue;
      const bool inb = a > 0, inf = a < na - 1;
      const double Fb = -(w[o] * pf[o]), Ff = w[o + 1] * pf[o + 1];
      double ff = 0., dd = 0.;
      if (DIM == 2 && D == 0) {  // cell faces in Arcane order: 2D x has the max face first
        if (inf) ff += Ff;
        if (inb) ff += Fb;
        if (inf) dd += 0.5 * Ff * 1.;
        if (inb) dd += 0.5 * Fb * -1.;
      } else {
        if (inb) ff += Fb;
        if (inf) ff += Ff;
        if (inb) dd += 0.5 * Fb * -1.;
        if (inf) dd += 0.5 * Ff * 1.;
      }
      const long c = line + a * sD;
      double un = (((ownm >> o) & 1u) ? u[o] : 0.) - ff;
      if (mass) S.dflux[(v - M) * nc + c] = dd;
      if (clamp && un < 0.) un = 0.;  // computeUremap clamps, :465-485
      Uout[v * nc + c] = un;
    }
  };
  for (int e = e0; e < e1; ++e) {
    double u[L];
    if (e == M) {
      slot(3 * M, u);
      store(3 * M, u, false, false);
      break;
    }
    double fv[L + 1], pv[L + 1];
    bool cor[L + 1];
    slot(e, u);
    store(e, u, false, false);
#pragma unroll
    for (int s = 0; s <= L; ++s) {
      fv[s] = pf[s];
      pv[s] = pu[s];
    }
    slot(M + e, u);
#pragma unroll
    for (int s = 0; s <= L; ++s) {
      cor[s] = !vpure[s] && cf[s].dir != 0 && pv[s] != 0. && pu[s] != 0.;
      if (cor[s]) pf[s] = (pu[s] / pv[s]) * fv[s];
    }
    store(M + e, u, true, true);
#pragma unroll
    for (int s = 0; s <= L; ++s) {
      fv[s] = pf[s];
      pv[s] = pu[s];
    }
    slot(2 * M + e, u);
#pragma unroll
    for (int s = 0; s <= L; ++s)
      if (cor[s]) pf[s] = (pu[s] / pv[s]) * fv[s];
    store(2 * M + e, u, false, true);
  }
}

// ----------------------------------------------------------------------------- generalised
// limiters and pente-borne fluxes (UtilesRemap.cc), in the reference's operation order.
// std::min / std::max as the reference's host code has them.
__device__ __forceinline__ double smin(double a, double b) { return (b < a) ? b : a; }
__device__ __forceinline__ double smax(double a, double b) { return (a < b) ? b : a; }

// fluxLimiterG (UtilesRemap.cc:130-183): slope from the front / back gradients gp, gm and
// the neighbour values yp, ym for widths h0 (cell), hp / hm (front / back neighbour).
__device__ __forceinline__ double flux_limiter_g(int id, double gp, double gm, double yp, double ym, double h0,
                                                 double hp, double hm, int simple_pente) {
  double grady = 0.;
  if (gp * gm < 0.0) return 0.;
  if (id == MH_MINMOD_G) {
    grady = (yp - ym) > 0. ? smin(fabs(gp), fabs(gm)) : -smin(fabs(gp), fabs(gm));
  } else if (id == MH_SUPERBEE_G) {
    grady = (yp - ym) > 0. ? smax(fabs(gp), fabs(gm)) : -smax(fabs(gp), fabs(gm));
  } else if (id == MH_VANLEER_G) {
    const double lp = (h0 / 2. + hp) / (h0 + hp + hm);
    const double lm = (h0 / 2. + hm) / (h0 + hp + hm);
    const double den = lp * gp + lm * gm;
    grady = den != 0. ? gp * gm / den : 0.;
  } else if (id == MH_ULTRABEE_G) {
    grady = (yp - ym) / h0;
  } else if (id == MH_ARITHMETIC_G) {
    const double lp = (h0 / 2. + hp) / (h0 + hp + hm);
    const double lm = (h0 / 2. + hm) / (h0 + hp + hm);
    grady = lm * gp + lp * gm;
  }
  if (simple_pente) {
    const double gMp = gp * (h0 + hp) / h0;
    const double gMm = gm * (h0 + hm) / h0;
    const double gM = smin(fabs(gMp), fabs(gMm));
    grady = (yp - ym) > 0. ? smin(fabs(gM), fabs(grady)) : -smin(fabs(gM), fabs(grady));
  }
  return grady;
}

// computeAndLimitGradPhi (UtilesRemap.cc:325-357): classical limiters from the back / front
// face gradients gb, gf; generalised ones (id >= MH_MINMOD_G) from values and widths.
__device__ __forceinline__ double limited_grad(int id, double gb, double gf, double yp, double ym, double h0,
                                               double hp, double hm, int simple_pente) {
  if (id < MH_MINMOD_G) {
    double g = 0.;
    if (gb != 0.) g += 0.5 * (mh_flux_limiter(id, gf / gb) * gb);
    if (gf != 0.) g += 0.5 * (mh_flux_limiter(id, gb / gf) * gf);
    return g;
  }
  return flux_limiter_g(id, gf, gb, yp, ym, h0, hp, hm, simple_pente);
}

// INTY (UtilesRemap.cc:86-97): integral from x0 to X of the segment (x0, y0)-(x1, y1).
__device__ __forceinline__ double inty(double X, double x0, double y0, double x1, double y1, double thr) {
  double flux = 0.;
  if (fabs(x1 - x0) > thr) {
    const double eta = amin(amax(0., (X - x0) / (x1 - x0)), 1.);
    flux = (y0 + 0.5 * eta * (y1 - y0)) * (x1 - x0) * eta;
  }
  return flux;
}

// computeY0 (UtilesRemap.cc:194-258): monotonicity thresholds y0plus, y0moins.
__device__ __forceinline__ void compute_y0(int id, double yplus, double ymoins, double h0, double hplus, double hmoins,
                                           int simple_pente, double& y0plus, double& y0moins) {
  y0plus = 0.;
  y0moins = 0.;
  if (id == MH_MINMOD_G || id == MH_MINMOD) {
    y0plus = yplus;
    y0moins = ymoins;
  } else if (id == MH_SUPERBEE_G || id == MH_SUPERBEE) {
    y0plus = ((h0 + hmoins) * yplus + h0 * ymoins) / (2 * h0 + hmoins);
    y0moins = ((h0 + hplus) * ymoins + h0 * yplus) / (2 * h0 + hplus);
  } else if (id == MH_VANLEER_G || id == MH_VANLEER) {
    const double a = amin(yplus, ymoins);
    const double b = amax(yplus, ymoins);
    double xplus = (h0 * h0 + 3 * h0 * hmoins + 2 * hmoins * hmoins) * yplus;
    double xmoins = (h0 * h0 + 3 * h0 * hplus + 2 * hplus * hplus) * ymoins;
    xplus += (h0 * h0 - h0 * hplus - 2 * hplus * hplus + 2 * h0 * hmoins) * ymoins;
    xmoins += (h0 * h0 - h0 * hmoins - 2 * hmoins * hmoins + 2 * h0 * hplus) * yplus;
    xplus /= (2 * h0 * h0 + 5 * h0 * hmoins + 2 * hmoins * hmoins - h0 * hplus - 2 * hplus * hplus);
    xmoins /= (2 * h0 * h0 + 5 * h0 * hplus + 2 * hplus * hplus - h0 * hmoins - 2 * hmoins * hmoins);
    y0plus = amin(amax(xplus, a), b);
    y0moins = amin(amax(xmoins, a), b);
  } else if (id == MH_ULTRABEE_G) {
    y0plus = (yplus + ymoins) / 2.;
    y0moins = (yplus + ymoins) / 2.;
  } else if (id == MH_ARITHMETIC_G) {
    y0plus = ((h0 + hmoins + hplus) * yplus + h0 * ymoins) / (2 * h0 + hmoins + hplus);
    y0moins = ((h0 + hmoins + hplus) * ymoins + h0 * yplus) / (2 * h0 + hmoins + hplus);
  }
  if (simple_pente) {
    y0plus = yplus;
    y0moins = ymoins;
  }
}

// One pente-borne flux of one variable (computeFluxPP / computeFluxPPPure,
// UtilesRemap.cc:425-832): the three-piece reconstruction of computexgxd (:269-290) and
// computeygyd (:302-318) integrated over the part of the cell that leaves through its back
// (type 0) or front (type 1) face; ppv = positive part of the outgoing velocity x dt.
__device__ __forceinline__ double pb_flux(int type, double y0, double yplus, double ymoins, double h0, double hplus,
                                          double hmoins, double grady, double ppv, int limY, double thr,
                                          int simple_pente) {
  double y0plus, y0moins;
  compute_y0(limY, yplus, ymoins, h0, hplus, hmoins, simple_pente, y0plus, y0moins);
  double xplus = 1.;
  if (fabs(y0plus - yplus) > thr) xplus = (y0 - yplus) / (y0plus - yplus) - 1. / 2.;
  double xmoins = 1.;
  if (fabs(y0moins - ymoins) > thr) xmoins = (y0 - ymoins) / (y0moins - ymoins) - 1. / 2.;
  const double xd = +h0 * amin(amax(xplus, -1. / 2.), 1. / 2.);
  const double xg = -h0 * amin(amax(xmoins, -1. / 2.), 1. / 2.);
  const double xtd = y0 + h0 / 2 * grady;
  const double xtg = y0 - h0 / 2 * grady;
  const double ad = amin(yplus, 2. * y0moins - ymoins);
  const double bd = amax(yplus, 2. * y0moins - ymoins);
  const double ag = amin(ymoins, 2. * y0plus - yplus);
  const double bg = amax(ymoins, 2. * y0plus - yplus);
  const double yd = amin(amax(xtd, ad), bd);
  const double yg = amin(amax(xtg, ag), bg);
  double f1, f1m, f2, f2m, f3, f3m;
  if (type == 0) {
    f1m = inty(-h0 / 2. + ppv, -h0 / 2., ymoins, xg, yg, thr);
    f1 = inty(-h0 / 2., -h0 / 2., ymoins, xg, yg, thr);
    f2m = inty(-h0 / 2. + ppv, xg, yg, xd, yd, thr);
    f2 = inty(-h0 / 2., xg, yg, xd, yd, thr);
    f3m = inty(-h0 / 2. + ppv, xd, yd, h0 / 2., yplus, thr);
    f3 = inty(-h0 / 2., xd, yd, h0 / 2., yplus, thr);
  } else {
    f1 = inty(h0 / 2. - ppv, -h0 / 2., ymoins, xg, yg, thr);
    f1m = inty(h0 / 2., -h0 / 2., ymoins, xg, yg, thr);
    f2 = inty(h0 / 2. - ppv, xg, yg, xd, yd, thr);
    f2m = inty(h0 / 2., xg, yg, xd, yd, thr);
    f3 = inty(h0 / 2. - ppv, xd, yd, h0 / 2., yplus, thr);
    f3m = inty(h0 / 2., xd, yd, h0 / 2., yplus, thr);
  }
  double F = smax(((f1m - f1) + (f2m - f2) + (f3m - f3)), 0.);
  if (((yplus - y0) * (ymoins - y0)) >= 0.) F = y0 * ppv;  // formula 16
  return F;
}

// One ADI direction, cell part, for the remap variants at order <= 2: runtime classical or
// generalised limiters (the limiter of a pure neighbourhood when projection-limiteur-pure-id
// is 1, RemapADIService.cc:205-209), and pente-borne fluxes (:213-264, :312-317, :424-428,
// :441-463, :493-538): phi is (volume fraction, density, specific energy, pseudo), each
// face carries the flux leaving the cell behind it minus the flux leaving the cell ahead,
// each computed from that cell and its two neighbours, then adjusted by the debar fix
// (UtilesRemap.cc:577-623, :782-826).  Boundary cells are their own missing neighbour.
//
// One thread per face: the fluxes of all 3m+1 slots through the back face of its cell, left in LDS,
// then the update of its cell from its own face and the next one.  A flux leaves through a face
// from one side only, so a face forms the slope and the flux of its upwind cell alone (of both
// cells where the face velocity is not a number).  A block takes MH_BLOCK faces: 255 cells in
// memory order for D = x, 32 x 7 cells of a plane for y and z  Bound by the FP64 instructions and
// the latency of one face's chain of slots, whose loads run one slot ahead; with a thread per cell,
// four fluxes per slot and all slots in registers (354: one wavefront per SIMD) it took 76 / 74 us for
// y / x on 420x180 cells and three environments, now 25 / 29.
// (GenTile: tiles of fewer columns and more rows on meshes narrower than 32 cells).
template <int DIM, int D, int M>
__device__ __forceinline__ void k_sweep_cell_gen_body(const MhDev& S, int lb, int usel, int first) {
  constexpr int NV = 3 * M + 1;
  __shared__ double F[NV][MH_BLOCK];  // of the face behind the thread's cell, in the direction +D
  __shared__ double Fv[M][MH_BLOCK];  // volume fluxes of the side being formed, for the debar fix
  const double* __restrict__ Uin = usel ? S.Ub : S.Ua;
  double* __restrict__ Uout = usel ? S.Ua : S.Ub;
  if (mh_halted(S.sc)) return;
  const int nx = S.g.nx, ny = S.g.ny, nz = S.g.nz;
  const int na = D == 0 ? nx : D == 1 ? ny : nz;
  const long nc = S.g.nc;
  const int tid = threadIdx.x;
  // the thread's cell (i, j, k), and whether it has one (a face only: the last row of the tile)
  int i, j, k;
  bool face, cell;
  int next = 1;  // thread of the face ahead
  if (D == 0) {
    const long c = (long)lb * (MH_BLOCK - 1) + tid;
    face = c < nc;
    cell = face && tid < MH_BLOCK - 1;
    i = (int)(c % nx);
    const long r = c / nx;
    j = (int)(r % ny);
    k = (int)(r / ny);
  } else {
    const GenTile tile(nx, D == 1 ? nz : ny, na);
    int ad, t;
    face = tile.face(lb, tid, i, t, ad);
    cell = face && tile.cell(tid);
    next = 1 << tile.lx;
    j = D == 1 ? ad : t;
    k = D == 1 ? t : ad;
  }
  const int a = D == 0 ? i : D == 1 ? j : k;
  const long c = i + (long)nx * (j + (long)ny * k);
  const long sD = D == 0 ? 1 : D == 1 ? (long)nx : (long)nx * ny;
  const bool pb = S.pb != 0;
  const double thr = S.thr_remap;
  if (face && a > 0) {
    const long nD = D == 0 ? 1 : D == 1 ? (long)S.g.nnx : (long)S.g.nnx * S.g.nny;
    const long b = i + (long)S.g.nnx * (j + (long)S.g.nny * k);
    const double dt = S.sc->dt;
    const int sp = S.simple_pente;
    const bool order2 = S.order2 != 0;
    const int debar = S.debar;
    // cells at offsets -2 .. 1 (index o + 2), clamped to the mesh: the two beside the face and one
    // more on each side
    long cs[4];
    bool valid[4];
    double den[4], xc[4], hs[4];
#pragma unroll
    for (int o = 0; o < 4; ++o) {
      const int bb = a + o - 2;
      valid[o] = bb >= 0 && bb < na;
      const int ao = min(max(bb, 0), na - 1);
      cs[o] = c + (ao - a) * sD;
      hs[o] = S.hc[D * nc + cs[o]];
      xc[o] = valid[o] ? cell_centre_d<DIM, D>(S, b + (o - 2) * nD) : 0.;
      if (first && !pb) {
        den[o] = S.mask[cs[o]] ? S.Vl[cs[o]] : 1.;  // an empty cell holds Phi itself
      } else {
        double sv = 0.;
        if (!first)
          for (int kk = 0; kk < M; ++kk) sv += Uin[kk * nc + cs[o]];
        den[o] = sv;
      }
    }
    double area, xf, vf;
    face_quant<DIM, D>(S, b, area, xf, vf);
    // pure neighbourhoods of the cells behind and ahead of the face
    bool vpure[2] = {false, false};
    if (S.pb_mixte) {
      int code[4];
#pragma unroll
      for (int o = 0; o < 4; ++o) {
        if (first) {
          code[o] = S.est[cs[o]];
        } else {
          int cnt = 0, pu = -1;
          for (int kk = 0; kk < M; ++kk)
            if (Uin[kk * nc + cs[o]] / den[o] > 0.) {
              cnt++;
              pu = kk;
            }
          code[o] = cnt > 1 ? MH_EST_MIXED : pu;
        }
      }
#pragma unroll
      for (int x = 0; x < 2; ++x)
        vpure[x] = code[x + 1] != MH_EST_MIXED && code[x] != MH_EST_MIXED && code[x + 2] != MH_EST_MIXED &&
                   code[x + 1] == code[x + 2] && code[x + 1] == code[x];
    }
    // slots in the order volumes, then mass and energy of each environment, then V q: the debar
    // fix and the zero test need the sum of the volume fluxes
    auto slot_of = [](int t) {
      if (t < M) return t;
      if (t == 3 * M) return 3 * M;
      const int e = (t - M) >> 1;
      return ((t - M) & 1) ? 2 * M + e : M + e;
    };
    const double ppA = 0.5 * (vf + fabs(vf)) * dt, ppB = 0.5 * (-vf + fabs(-vf)) * dt;  // leaving the cell behind, ahead
    int side = pb ? (ppA != 0. ? 0 : 1) : (vf * (xc[2] - xc[1]) > 0.0 ? 0 : 1);  // 0: upwind cell behind the face
    for (int v = 0; v < NV; ++v) F[v][tid] = 0.;
    for (;;) {
      const double pp = side ? ppB : ppA;
      if ((!pb || order2) && !(pb && pp == 0.)) {
        const bool sd = side != 0;
        const long cc[3] = {sd ? cs[1] : cs[0], sd ? cs[2] : cs[1], sd ? cs[3] : cs[2]};
        const double dn[3] = {sd ? den[1] : den[0], sd ? den[2] : den[1], sd ? den[3] : den[2]};
        const double hm = sd ? hs[1] : hs[0], h0 = sd ? hs[2] : hs[1], hp = sd ? hs[3] : hs[2];
        const double xm = sd ? xc[1] : xc[0], x0 = sd ? xc[2] : xc[1], xp = sd ? xc[3] : xc[2];
        const bool okb = sd ? valid[1] : valid[0], okf = sd ? valid[3] : valid[2];  // the upwind cell exists
        const bool vp = sd ? vpure[1] : vpure[0];
        const int lim = (S.lim_pure == 1 && vp) ? S.lim_pure : S.limiter;
        const int limY = vp ? S.lim_pure : S.limiter;
        const double hup = (double)S.order2 * (xf - x0);
        const double dxb = okb ? x0 - xm : 0., dxf = okf ? xp - x0 : 0.;
        // phi of a slot: numerators and denominators, loaded one slot ahead
        auto fetch = [&](int v, double* n, double* d) {
          const bool ratio = pb && !first && v >= M && v < 3 * M;
          const double* src = pb && (first || v == 3 * M) ? S.phi0 : Uin;
#pragma unroll
          for (int o = 0; o < 3; ++o) {
            n[o] = src[v * nc + cc[o]];
            if (ratio) d[o] = Uin[(v - M) * nc + cc[o]];
          }
        };
        double n1[3], d1[3] = {1., 1., 1.};
        fetch(slot_of(0), n1, d1);
        double sfv = 0., Fm = 0.;
#pragma unroll 1
        for (int t = 0; t < NV; ++t) {
          const int v = slot_of(t);
          double y[3];
          if (pb && (first || v == 3 * M)) {
#pragma unroll
            for (int o = 0; o < 3; ++o) y[o] = n1[o];
          } else if (!pb || v < M) {
#pragma unroll
            for (int o = 0; o < 3; ++o) y[o] = n1[o] / dn[o];
          } else {
#pragma unroll
            for (int o = 0; o < 3; ++o) y[o] = d1[o] != 0. ? n1[o] / d1[o] : 0.;
          }
          if (t + 1 < NV) fetch(slot_of(t + 1), n1, d1);
          double g = 0.;
          if (order2) {
            const double gb = okb ? (y[1] - y[0]) / dxb : 0.;
            const double gf = okf ? (y[2] - y[1]) / dxf : 0.;
            g = limited_grad(lim, gb, gf, y[2], y[0], h0, hp, hm, sp);
          }
          double f;
          if (!pb) {
            f = y[1] + hup * g;
          } else {
            f = pb_flux(side == 0 ? 1 : 0, y[1], y[2], y[0], h0, hp, hm, g, pp, limY, thr, sp);
            if (v >= M && v < 3 * M) {
              const bool energy = v >= 2 * M;
              const double Fr = energy ? Fm : Fv[v - M][tid];  // the volume or the mass flux
              if (energy || !vp) {
                if (debar == 1) f = (f / sfv) * Fr;
                else if (debar == 2) f = y[1] * Fr;
              }
              if (!energy) Fm = f;
            }
          }
          auto add = [&](int q, double x) { F[q][tid] = pb && side ? F[q][tid] - x : x; };
          if (t >= M) {
            add(v, f);
          } else {
            sfv += f;
            Fv[v][tid] = f;
            if (t == M - 1) {
              if (pb && debar == 1 && !(fabs(sfv) > thr)) break;  // nothing leaves from this side
              for (int q = 0; q < M; ++q) add(q, Fv[q][tid]);
            }
          }
        }
      }
      if (!(pb && side == 0 && ppB != 0.)) break;
      side = 1;
    }
    const double w = pb ? area : vf * area * dt;
    for (int v = 0; v < NV; ++v) F[v][tid] = w * F[v][tid];
  }
  __syncthreads();
  if (!cell) return;
  const bool inb = a > 0, inf = a < na - 1;
  const bool own = !(first && S.mask[c] == 0);  // an empty cell's U starts from 0 (its Phi is stale)
  auto update = [&](int v, bool mass) {
    const double Fb = inb ? -F[v][tid] : 0., Ff = inf ? F[v][tid + next] : 0.;
    double ff = 0., dd = 0.;
    if (DIM == 2 && D == 0) {  // cell faces in Arcane order: 2D x has the max face first
      if (inf) ff += Ff;
      if (inb) ff += Fb;
      if (inf) dd += 0.5 * Ff * 1.;
      if (inb) dd += 0.5 * Fb * -1.;
    } else {
      if (inb) ff += Fb;
      if (inf) ff += Ff;
      if (inb) dd += 0.5 * Fb * -1.;
      if (inf) dd += 0.5 * Ff * 1.;
    }
    if (mass) S.dflux[(v - M) * nc + c] = dd;
    return (own ? Uin[v * nc + c] : 0.) - ff;
  };
#pragma unroll
  for (int e = 0; e < M; ++e) {
    double un[3] = {update(e, false), update(M + e, true), update(2 * M + e, false)};
    if (pb && !S.sans_lagrange) {  // with the dual phase, tiny partial volumes, masses or energies drop the environment (:441-463)
      if (un[0] < 1. * thr) un[0] = un[1] = un[2] = 0.;
      if (un[1] < 1. * thr) un[0] = un[1] = un[2] = 0.;
      if (un[2] < 1. * thr) un[0] = un[1] = un[2] = 0.;
    }
    if (un[1] < 0.) un[1] = 0.;  // computeUremap clamps, :465-485
    if (un[2] < 0.) un[2] = 0.;
#pragma unroll
    for (int q = 0; q < 3; ++q) Uout[(q * M + e) * nc + c] = un[q];
  }
  Uout[3 * M * nc + c] = update(3 * M, false);
}

// The x sweep with one wavefront per row segment: lane l holds cell i = 60 s - 2 + l of a
// row, so the stencil neighbours along x are the neighbouring lanes.  Phi, the gradient of
// the back face, the limited slope and the flux of the back face are formed once per cell
// and passed to the neighbour with a lane shuffle (the front-face value of cell i is the
// back-face value of cell i+1).  Lanes 2..61 write their cell; the two lanes at each end
// only feed the stencil.  Same formulas in the same order as k_sweep_cell_body.
#define MH_ROW_OUT 60
// Order of the cell rows (j, k) of the x sweep: slabs of MH_ROW_KT cell planes, k fastest
// inside a slab, so the four cell rows around a node row (j-1..j, k-1..k) run within
// 2 MH_ROW_KT rows of each other and find that row's coordinates and velocity in L2.
#ifndef MH_ROW_KT
#define MH_ROW_KT 4
#endif
__device__ __forceinline__ void row_jk(const MhGrid& g, long r, int& j, int& k) {
  const long slab = (long)g.ny * MH_ROW_KT;
  const int kt = (int)(r / slab);
  const int h = min(MH_ROW_KT, g.nz - kt * MH_ROW_KT);  // planes of this slab (1 in 2D)
  const long rem = r - kt * slab;
  j = (int)(rem / h);
  k = kt * MH_ROW_KT + (int)(rem % h);
}
template <int DIM, int M, int LIM>
__device__ __forceinline__ void k_sweep_cell_row_body(const MhDev& S, int lb, int usel, int first, int v0 = 0,
                                                      int v1 = 3 * M + 1) {  // slots v0 .. v1-1
  constexpr int NV = 3 * M + 1;
  const int nx = S.g.nx;
  const long rows = (long)S.g.ny * S.g.nz;
  const int wpr = (nx + MH_ROW_OUT - 1) / MH_ROW_OUT;
  const int lane = threadIdx.x & 63;
  const long gw = (long)lb * (MH_BLOCK / 64) + (threadIdx.x >> 6);
  if (gw >= rows * wpr) return;  // whole wavefront
  const double* __restrict__ Uin = usel ? S.Ub : S.Ua;
  double* __restrict__ Uout = usel ? S.Ua : S.Ub;
  double* __restrict__ dflux = S.dflux;
  int j, k;
  row_jk(S.g, gw / wpr, j, k);
  const long row = j + (long)S.g.ny * k;
  const int i = (int)(gw % wpr) * MH_ROW_OUT - 2 + lane;
  const bool valid = i >= 0 && i < nx;
  const bool validp = i - 1 >= 0 && i - 1 < nx;
  const bool out = valid && lane >= 2 && lane < 2 + MH_ROW_OUT;
  const bool inb = valid && i > 0;       // back face (node column i): inner when 0 < i < nx
  const bool inf = valid && i < nx - 1;
  const long nc = S.g.nc;
  // lanes beyond the row load its end cell again (unused), so that no branch parts the loads
  const int ic = min(max(i, 0), nx - 1);
  const long c = row * nx + ic;
  const long b = ic + (long)S.g.nnx * (j + (long)S.g.nny * k);
  const bool sparse = M > 1 && S.pm[0] != nullptr;
  unsigned slots = ((1u << v1) - 1u) & ~((1u << v0) - 1u);  // the slots to run
  // every load that depends on the kernel arguments alone goes out before anything waits (the stop
  // flag included): a wavefront's time here is that of its load rounds
  const unsigned here = sparse ? S.pm[usel ? 1 : 0][c] : 0u;
  const unsigned old = sparse ? S.pm[usel ? 0 : 1][c] : ~0u;
  const uint8_t mk = first ? S.mask[c] : (uint8_t)1;
  double den = first ? S.Vl[c] : 1.;
  double u[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const bool now = !sparse || v == 3 * M || (v < M && !first);
    u[v] = now && (((slots >> v) & 1u) || (v < M && !first)) ? Uin[v * nc + c] : 0.;
  }
  const double dt = S.sc->dt;
  const bool halted = mh_halted(S.sc);
  const double xc = cell_centre_d<DIM, 0>(S, b);
  double area, xf, vf;
  face_quant<DIM, 0>(S, b, area, xf, vf);
  if (halted) return;
  const bool own = mk != 0;  // an empty cell's U starts from 0
  if (first) {
    if (!own) den = 1.;  // an empty cell holds Phi itself
  } else {
    double sv = 0.;
#pragma unroll
    for (int kk = 0; kk < M; ++kk) sv += u[kk];
    den = sv;
  }
  const double xcp = lane_back(xc);
  const double dxb = (valid && validp) ? xc - xcp : 0.;
  const bool upprev = vf * dxb > 0.0;
  const double hb = (double)S.order2 * (xf - (upprev ? xcp : xc));
  const double w = 1. * vf * area * dt;
  // with presence bytes the slots to run are those of the environments some cell of the wavefront
  // holds, and V q.  Where no cell of a stencil holds an environment its slots stay 0, unless a
  // factor is zero, infinite or not a number, and then they all run.
  unsigned held = 0;
  if (sparse) {
    const bool irregular = valid && (!mh_finite_nonzero(den) || (validp && lane > 0 && !mh_finite_nonzero(dxb)) ||
                                     (inb && (!mh_finite(w) || !mh_finite(hb))));
    const unsigned in = irregular ? (1u << M) - 1u : valid ? here : 0u;
#pragma unroll
    for (int e = 0; e < M; ++e)
      if (__ballot((in >> e) & 1u) == 0) slots &= ~((1u << e) | (1u << (M + e)) | (1u << (2 * M + e)));
#pragma unroll
    for (int v = 0; v < 3 * M; ++v)
      if (((slots >> v) & 1u) && (v >= M || first)) u[v] = Uin[v * nc + c];
    if (out) {
#pragma unroll
      for (int e = 0; e < M; ++e)
        if (!((slots >> e) & 1u)) {  // zeros, stored where the buffer holds anything else
          dflux[e * nc + c] = 0.;
          if ((old >> e) & 1u) Uout[e * nc + c] = Uout[(M + e) * nc + c] = Uout[(2 * M + e) * nc + c] = 0.;
        }
    }
  }
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    if (!((slots >> v) & 1u)) continue;
    const double phi = valid ? u[v] / den : 0.;
    const double phip = lane_back(phi);
    const double gb = (valid && validp) ? (phi - phip) / dxb : 0.;
    const double gf = lane_front(gb);
    double g = 0.;
    if (S.order2 && valid) {
      if (gb != 0.) g += 0.5 * (mh_limiter<LIM>(S.limiter, gf / gb) * gb);
      if (gf != 0.) g += 0.5 * (mh_limiter<LIM>(S.limiter, gb / gf) * gf);
    }
    const double gp = lane_back(g);
    double F = 0.;  // flux of the back face with outer normal +e_x (for cell i-1)
    if (inb) {
      const double pf = (upprev ? phip : phi) + hb * (upprev ? gp : g);
      F = w * pf;
    }
    const double Ff = lane_front(F);
    const double fb = -F;  // the back face seen from cell i (outer normal -e_x)
    double ff = 0.;
    double dd = 0.;
    if (DIM == 2) {  // 2D: the max-x face comes first in the cell's face order
      if (inf) ff += Ff;
      if (inb) ff += fb;
      if (inf) dd += 0.5 * Ff * 1.;
      if (inb) dd += 0.5 * fb * -1.;
    } else {
      if (inb) ff += fb;
      if (inf) ff += Ff;
      if (inb) dd += 0.5 * fb * -1.;
      if (inf) dd += 0.5 * Ff * 1.;
    }
    if (out) {
      double un = (own ? u[v] : 0.) - ff;
      if (v >= M && v < 2 * M) dflux[(v - M) * nc + c] = dd;
      if (v >= M && v < 3 * M && un < 0.) un = 0.;
      if (M > 1 && v < 3 * M) {
        if (un != 0.) held |= 1u << (v % M);
        if (un != 0. || ((old >> (v % M)) & 1u)) Uout[v * nc + c] = un;
      } else {
        Uout[v * nc + c] = un;
      }
    }
  }
  if (sparse && out) S.pm[usel ? 0 : 1][c] = (uint8_t)held;
}

// Mass flux through the dual faces between node position a and a+1 along D: the sum, in
// the order of k_sweep_node_body, of the cell mass fluxes of the 2^(d-1) cells at
// position a around the node line (it1, it2) -- the "front" flux of node a and the "back"
// flux of node a+1 (DualPhaseRemap.cc:75-108).  0 when position a holds no cells.
template <int DIM, int D, int M>
__device__ __forceinline__ double dual_edge_flux(const MhDev& S, int a, int it1, int it2) {
  const int na = D == 0 ? S.g.nx : D == 1 ? S.g.ny : S.g.nz;
  const double w = DIM == 3 ? 0.25 : 0.5;
  const long nc = S.g.nc;
  const int n1 = D == 0 ? S.g.ny : S.g.nx;
  const int n2 = D == 2 ? S.g.ny : S.g.nz;
  const long st1 = D == 0 ? (long)S.g.nx : 1;
  const long st2 = D == 2 ? (long)S.g.nx : (long)S.g.nx * S.g.ny;
  const int ac = min(max(a, 0), na - 1);
  const long cbase = D == 0 ? (long)ac : D == 1 ? (long)ac * S.g.nx : (long)ac * S.g.nx * S.g.ny;
  constexpr int N2 = DIM == 3 ? 2 : 1;
  // all cells are loaded before the first is added: a cell beyond the mesh is its neighbour again,
  // left out of the sum (one wait instead of one per cell and environment)
  double d[N2][2][M];
#pragma unroll
  for (int q2 = 0; q2 < N2; ++q2)
#pragma unroll
    for (int q1 = 0; q1 < 2; ++q1) {
      const int p1 = min(max(it1 - 1 + q1, 0), n1 - 1), p2 = DIM == 3 ? min(max(it2 - 1 + q2, 0), n2 - 1) : 0;
      const long cf = cbase + p1 * st1 + (DIM == 3 ? p2 * st2 : 0);
#pragma unroll
      for (int kk = 0; kk < M; ++kk) d[q2][q1][kk] = S.dflux[kk * nc + cf];
    }
  double f = 0.;
#pragma unroll
  for (int q2 = 0; q2 < N2; ++q2)
#pragma unroll
    for (int q1 = 0; q1 < 2; ++q1) {
      const int p1 = it1 - 1 + q1, p2 = it2 - 1 + q2;
      const bool in = p1 >= 0 && p1 < n1 && (DIM == 2 || (p2 >= 0 && p2 < n2));
#pragma unroll
      for (int kk = 0; kk < M; ++kk) f = in ? f + w * d[q2][q1][kk] : f;
    }
  return a < 0 || a >= na ? 0. : f;
}

// The dual state of a node between two sweeps is four words, v and m, read from one buffer and
// written to the other (psel, as the cells' U): A = Ud, B = Pa for v and Pb for m; the first sweep
// reads v = u and m = the node mass.  phi is not stored: a node updated by an earlier sweep holds
// v = U (momentum), and phi = U / m is formed where it is read, from the operands the reference
// divides (DualPhaseRemap.cc:251-257); a node that every earlier sweep kept (a boundary node of
// each direction swept so far, hence every node in the first sweep) holds v = phi, which is still
// u, and U = m u (PrepareRemap.cc:169-178).  prev is the bit mask of the directions already swept.
// The sweeps are bound by HBM: storing phi besides U moved 6 of 17 words per node and sweep, and
// the last sweep wrote 7 words that nothing reads.  Without them, per launch: x 157 -> 119 us, y
// and z 192 -> 168 us on the 256x128x128 tube; 230 -> 169 and 247 -> 204 us on the 192^3 blast.
struct DualBuf {
  const double* v[3];
  const double* m;
};
template <int DIM>
__device__ __forceinline__ DualBuf dual_in(const MhDev& S, int psel, int prev) {
  DualBuf b;
  const double* base = psel ? S.Ud : S.Pa;
#pragma unroll
  for (int cc = 0; cc < 3; ++cc) b.v[cc] = prev ? base + cc * S.g.nn : S.u[cc];
  b.m = prev ? (psel ? S.Ud + DIM * S.g.nn : S.Pb) : S.mn;
  return b;
}
__device__ __forceinline__ double* dual_out_v(const MhDev& S, int psel) { return psel ? S.Pa : S.Ud; }
template <int DIM>
__device__ __forceinline__ double* dual_out_m(const MhDev& S, int psel) {
  return psel ? S.Pb : S.Ud + DIM * S.g.nn;
}
// Whether every sweep so far kept node (i, j, k).
template <int DIM>
__device__ __forceinline__ bool dual_kept(const MhDev& S, int prev, int i, int j, int k) {
  bool kept = true;
  if (prev & 1) kept = kept && (i == 0 || i == S.g.nx);
  if (prev & 2) kept = kept && (j == 0 || j == S.g.ny);
  if (DIM == 3 && (prev & 4)) kept = kept && (k == 0 || k == S.g.nz);
  return kept;
}

// Limited nodal gradient from the edge gradients behind (gb) and ahead (gf)
// (computeAndLimitGradPhiDual, UtilesRemap.cc:369-400), in the order of k_sweep_node_body.
template <int LIM>
__device__ __forceinline__ double dual_limited(const MhDev& S, double gb, double gf) {
  return mh_limited_gradient<LIM, true>(S.limiter, gb, gf);
}

// Writes the dual state (v, U[DIM]) of node n, or on the last sweep the velocity U / m
// (RemapADIFinal.cc:286-297); the mass is still read after it by conservation-energie-totale.
// A node with no neighbour along D keeps its state: v and m are written as they were read.
template <int DIM>
__device__ __forceinline__ void dual_store(const MhDev& S, long n, const double* U, const double* v, int psel,
                                           int last) {
  const long nn = S.g.nn;
  if (!last) {
    double* __restrict__ V = dual_out_v(S, psel);
#pragma unroll
    for (int cc = 0; cc < DIM; ++cc) V[cc * nn + n] = v[cc];
  }
  if (!last || S.dec) dual_out_m<DIM>(S, psel)[n] = U[DIM];
  if (last && U[DIM] != 0.) {
    const MhRecip rm = mh_denom(U[DIM]);
#pragma unroll
    for (int cc = 0; cc < DIM; ++cc) S.u[cc][n] = mh_quot(U[cc], rm);
  }
}

// Dual update of one node from its neighbourhood along D (DualPhaseRemap.cc:110-257):
// Pm/P0/Pp, Xm/X0/Xp, Gm/G0/Gp are phi, coordinate and limited gradient of the nodes a-1,
// a, a+1; back/front the dual mass fluxes.  Writes the dual state or, on the last sweep, u.
template <int DIM, int D>
__device__ __forceinline__ void dual_node_update(const MhDev& S, long n, double* U, const double* Pm,
                                                 const double* P0, const double* Pp, double Xm, double X0,
                                                 double Xp, const double* Gm, const double* G0,
                                                 const double* Gp, double back, double front, int psel,
                                                 int last) {
  constexpr int NC = DIM;
  const double dt = S.sc->dt;
  U[NC] += back - front;
  const double o2 = (double)S.order2;
  const double ufront = 0.5 * (P0[D] + Pp[D]);
  const int sf = ufront > 0 ? 1 : -1;
  const bool fo = front < 0.;
  const double uback = 0.5 * (Pm[D] + P0[D]);
  const int sb = uback > 0 ? 1 : -1;
  const bool bo = back > 0.;
#pragma unroll
  for (int cc = 0; cc < NC; ++cc) {
    const double FU = (fo ? Pp[cc] : P0[cc]) + o2 * (0.5 * (fo ? Gp[cc] : G0[cc]) * (sf * (Xp - X0) - dt * ufront));
    const double BU = (bo ? Pm[cc] : P0[cc]) + o2 * (0.5 * (bo ? Gm[cc] : G0[cc]) * (sb * (X0 - Xm) - dt * uback));
    U[cc] += back * BU - front * FU;
  }
#pragma unroll
  for (int cc = 0; cc < NC; ++cc)
    if (fabs(U[cc]) < 1.e-300) U[cc] = 0.;
  dual_store<DIM>(S, n, U, U, psel, last);
}

// Dual x sweep with one wavefront per 60 nodes of a node row (lane shuffles carry the
// neighbours' phi, coordinates, edge gradients and limited gradients; the front flux of
// node i is the back flux of node i+1).  Lanes 2..61 write their node.
template <int DIM, int M, int LIM>
__device__ __forceinline__ void k_sweep_node_row_body(const MhDev& S, int lb, int psel, int prev, int last) {
  constexpr int NC = DIM;
  const int nnx = S.g.nnx, na = S.g.nx;
  const long rows = (long)S.g.nny * S.g.nnz;
  const int wpr = (nnx + MH_ROW_OUT - 1) / MH_ROW_OUT;
  const int lane = threadIdx.x & 63;
  const long gw = (long)lb * (MH_BLOCK / 64) + (threadIdx.x >> 6);
  if (gw >= rows * wpr) return;  // whole wavefront
  const DualBuf in = dual_in<DIM>(S, psel, prev);
  const long row = gw / wpr;
  const int i = (int)(gw % wpr) * MH_ROW_OUT - 2 + lane;
  const bool valid = i >= 0 && i <= na;
  const bool validp = i - 1 >= 0 && i - 1 <= na;
  const bool out = valid && lane >= 2 && lane < 2 + MH_ROW_OUT;
  const int j = (int)(row % S.g.nny);
  const int k = (int)(row / S.g.nny);
  // lanes beyond the row load its end node again (unused); one round of loads, the stop flag included
  const long n = row * nnx + min(max(i, 0), na);
  double v[NC], P[NC];
#pragma unroll
  for (int cc = 0; cc < NC; ++cc) v[cc] = in.v[cc][n];
  const double m = in.m[n];
  const double X = S.xlc[0][n];
  const double flux = dual_edge_flux<DIM, 0, M>(S, i, j, k);
  if (mh_halted(S.sc)) return;
  const double front = valid ? flux : 0.;
  const bool kept = dual_kept<DIM>(S, prev, i, j, k);
#pragma unroll
  for (int cc = 0; cc < NC; ++cc) P[cc] = valid ? v[cc] : 0.;
  if (!kept && valid) {
    const MhRecip rm = mh_denom(m);
#pragma unroll
    for (int cc = 0; cc < NC; ++cc) P[cc] = mh_ratio(v[cc], rm);
  }
  const bool inner = valid && i >= 1 && i <= na - 1;
  const double Xm = lane_back(X), Xp = lane_front(X);
  double Pm[NC], Pp[NC], G0[NC], Gm[NC], Gp[NC];
  const MhRecip rX = mh_denom(X - Xm);
#pragma unroll
  for (int cc = 0; cc < NC; ++cc) {
    Pm[cc] = lane_back(P[cc]);
    Pp[cc] = lane_front(P[cc]);
    const double eb = (valid && validp) ? mh_ratio(P[cc] - Pm[cc], rX) : 0.;  // edge i-1/2
    const double ef = lane_front(eb);                                        // edge i+1/2
    G0[cc] = (S.order2 && inner) ? dual_limited<LIM>(S, eb, ef) : 0.;
    Gm[cc] = lane_back(G0[cc]);
    Gp[cc] = lane_front(G0[cc]);
  }
  const double back = lane_back(front);
  if (!out) return;
  double U[NC + 1];
#pragma unroll
  for (int cc = 0; cc < NC; ++cc) U[cc] = kept ? m * v[cc] : v[cc];
  U[NC] = m;
  if (!inner) {
    dual_store<DIM>(S, n, U, v, psel, last);
    return;
  }
  dual_node_update<DIM, 0>(S, n, U, Pm, P, Pp, Xm, X, Xp, Gm, G0, Gp, back, front, psel, last);
}

// The same sweep for D = y or z, LDS tiles: a block of 64 x 4 threads owns 64 cells along
// x by MH_TILE_L cells along D (plus two halo cells on each side).  Every cell's Phi, every
// face gradient, every limited slope and every face flux of the tile is formed once, by
// the thread owning that row, and shared through LDS (four barriers per remap slot).
// Wavefront w holds rows w, w+4, ... of the tile, 64 consecutive cells in x, so every
// global access is coalesced.  Same formulas in the same order as k_sweep_cell_body.
#ifndef MH_TILE_L
#define MH_TILE_L 16  // cells along the sweep direction written per tile (a multiple of 4)
#endif
#define MH_TILE_R (MH_TILE_L + 4)  // rows held, halos included
#define MH_TILE_Q (MH_TILE_R / 4)  // rows per thread
#ifndef MH_TILE_MIN_WAVES
#define MH_TILE_MIN_WAVES 4  // waves per SIMD the register allocation must allow
#endif
template <int DIM, int D, int M, int LIM>
__device__ __forceinline__ void k_sweep_cell_tile_body(const MhDev& S, int lb_, int usel, int first) {
  constexpr int NV = 3 * M + 1;
  __shared__ double sphi[MH_TILE_R][64];
  __shared__ double sgf[MH_TILE_R][64];  // face gradients, then face fluxes
  __shared__ double ssl[MH_TILE_R][64];  // cell centres, then limited slopes
  const int nx = S.g.nx, ny = S.g.ny, nz = S.g.nz;
  const int na = D == 1 ? ny : nz;
  const int nt = (D == 1) ? (DIM == 3 ? nz : 1) : ny;
  const int tilesx = (nx + 63) / 64;
  const long ntiles = (long)tilesx * nt * ((na + MH_TILE_L - 1) / MH_TILE_L);
  const long lb = lb_;
  if (lb >= ntiles) return;  // whole block
  if (mh_halted(S.sc)) return;
  const double* __restrict__ Uin = usel ? S.Ub : S.Ua;
  double* __restrict__ Uout = usel ? S.Ua : S.Ub;
  double* __restrict__ dflux = S.dflux;
  const int lx = threadIdx.x & 63, ly = threadIdx.x >> 6;
  // tiles along D vary fastest: the tiles sharing a halo run side by side on one XCD
  const int ntd = (na + MH_TILE_L - 1) / MH_TILE_L;
  const int abase = (int)(lb % ntd) * MH_TILE_L - 2;  // cell along D of tile row 0
  const long rest = lb / ntd;
  const int i = (int)(rest % tilesx) * 64 + lx;
  const int t = (int)(rest / tilesx);
  const long nc = S.g.nc;
  const long nnx = S.g.nnx, nny = S.g.nny;
  const long sD = D == 1 ? (long)nx : (long)nx * ny;
  const long c_base = D == 1 ? i + (long)nx * ny * t : i + (long)nx * t;
  const long nD = D == 1 ? nnx : nnx * nny;
  const long n_base = D == 1 ? i + nnx * nny * t : i + nnx * t;
  const double dt = S.sc->dt;
  const double o2 = (double)S.order2;
  // rows r = ly + 4q of this thread: cell validity, Phi denominator, Delta x of face r
  // (between rows r-1 and r) and the upwind data of that face
  bool val[MH_TILE_Q], inner[MH_TILE_Q], up[MH_TILE_Q];
  double den[MH_TILE_Q], dx[MH_TILE_Q], w[MH_TILE_Q], hh[MH_TILE_Q], xcq[MH_TILE_Q];
  unsigned ownm = 0;  // bit q: the cell's own U enters its update
#pragma unroll
  for (int q = 0; q < MH_TILE_Q; ++q) {
    const int a = abase + ly + 4 * q;
    val[q] = i < nx && a >= 0 && a < na;
    den[q] = 1.;
    xcq[q] = 0.;
    if (val[q]) {
      const long cc = c_base + a * sD;
      if (first) {
        const bool empty = !S.mask[cc];  // an empty cell holds Phi itself and its U starts from 0
        den[q] = empty ? 1. : S.Vl[cc];
        if (!empty) ownm |= 1u << q;
      } else {
        ownm |= 1u << q;
        double sv = 0.;
        for (int k = 0; k < M; ++k) sv += Uin[k * nc + cc];
        den[q] = sv;
      }
      xcq[q] = cell_centre_d<DIM, D>(S, n_base + a * nD);
    }
    ssl[ly + 4 * q][lx] = xcq[q];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < MH_TILE_Q; ++q) {
    const int r = ly + 4 * q, a = abase + r;
    const bool valp = r >= 1 && i < nx && a - 1 >= 0 && a - 1 < na;
    const double xcp = r >= 1 ? ssl[r - 1][lx] : 0.;
    dx[q] = (val[q] && valp) ? xcq[q] - xcp : 0.;
    inner[q] = val[q] && valp;  // face between cells a-1 and a
    up[q] = false;
    w[q] = 0.;
    hh[q] = 0.;
    if (inner[q] && r >= 2 && r <= MH_TILE_R - 2) {
      double area, xf, vf;
      face_quant<DIM, D>(S, n_base + a * nD, area, xf, vf);
      up[q] = vf * dx[q] > 0.0;
      hh[q] = o2 * (xf - (up[q] ? xcp : xcq[q]));
      w[q] = 1. * vf * area * dt;
    }
  }
  // the slots to run, as in k_sweep_cell_row_body: those of the environments some cell of the tile
  // holds, and V q
  const bool sparse = M > 1 && S.pm[0] != nullptr;
  unsigned slots = (1u << NV) - 1u, held = 0, olds = ~0u;  // held, olds: M bits per row q
  if (sparse) {
    static_assert(MH_TILE_Q * M <= 32, "the presence bits of a thread's rows fit a word");
    unsigned in = 0;
    olds = 0;
#pragma unroll
    for (int q = 0; q < MH_TILE_Q; ++q) {
      const int r = ly + 4 * q;
      if (!val[q]) continue;
      const long c = c_base + (abase + r) * sD;
      const bool irregular = !mh_finite_nonzero(den[q]) ||
                             (inner[q] && (!mh_finite_nonzero(dx[q]) || !mh_finite(w[q]) || !mh_finite(hh[q])));
      in |= irregular ? (1u << M) - 1u : (unsigned)S.pm[usel ? 1 : 0][c];
      if (r >= 2 && r < 2 + MH_TILE_L) olds |= (S.pm[usel ? 0 : 1][c] & ((1u << M) - 1u)) << (M * q);
    }
#pragma unroll
    for (int e = 0; e < M; ++e)
      if (!__syncthreads_or((in >> e) & 1u)) slots &= ~((1u << e) | (1u << (M + e)) | (1u << (2 * M + e)));
#pragma unroll
    for (int q = 0; q < MH_TILE_Q; ++q) {
      const int r = ly + 4 * q;
      if (!val[q] || r < 2 || r >= 2 + MH_TILE_L) continue;
      const long c = c_base + (abase + r) * sD;
#pragma unroll
      for (int e = 0; e < M; ++e)
        if (!((slots >> e) & 1u)) {
          dflux[e * nc + c] = 0.;
          if ((olds >> (M * q + e)) & 1u) Uout[e * nc + c] = Uout[(M + e) * nc + c] = Uout[(2 * M + e) * nc + c] = 0.;
        }
    }
  }
  double un_next[MH_TILE_Q];  // slot loads run one slot ahead
#pragma unroll
  for (int q = 0; q < MH_TILE_Q; ++q)
    un_next[q] = val[q] ? Uin[(__ffs(slots) - 1) * nc + c_base + (abase + ly + 4 * q) * sD] : 0.;
  while (slots) {
    const int v = __ffs(slots) - 1;
    slots &= slots - 1;
    // barriers: the previous slot read sphi and ssl before its last barrier, and reads
    // sgf (fluxes) before the first barrier of this slot
    double uq[MH_TILE_Q];
#pragma unroll
    for (int q = 0; q < MH_TILE_Q; ++q) {
      const int a = abase + ly + 4 * q;
      uq[q] = un_next[q];
      if (slots) un_next[q] = val[q] ? Uin[(__ffs(slots) - 1) * nc + c_base + a * sD] : 0.;
      sphi[ly + 4 * q][lx] = val[q] ? uq[q] / den[q] : 0.;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < MH_TILE_Q; ++q) {
      const int r = ly + 4 * q;
      sgf[r][lx] = (r >= 1 && inner[q]) ? (sphi[r][lx] - sphi[r - 1][lx]) / dx[q] : 0.;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < MH_TILE_Q; ++q) {
      const int r = ly + 4 * q;
      double g = 0.;
      if (S.order2 && val[q] && r >= 1 && r <= MH_TILE_R - 2) {
        const double gb = sgf[r][lx], gf = sgf[r + 1][lx];
        if (gb != 0.) g += 0.5 * (mh_limiter<LIM>(S.limiter, gf / gb) * gb);
        if (gf != 0.) g += 0.5 * (mh_limiter<LIM>(S.limiter, gb / gf) * gf);
      }
      ssl[r][lx] = g;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < MH_TILE_Q; ++q) {  // the gradients were all read before the barrier
      const int r = ly + 4 * q;
      double f = 0.;
      if (inner[q] && r >= 2 && r <= MH_TILE_R - 2) {
        const double pf = up[q] ? sphi[r - 1][lx] + hh[q] * ssl[r - 1][lx] : sphi[r][lx] + hh[q] * ssl[r][lx];
        f = w[q] * pf;
      }
      sgf[r][lx] = f;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < MH_TILE_Q; ++q) {
      const int r = ly + 4 * q, a = abase + r;
      if (!val[q] || r < 2 || r >= 2 + MH_TILE_L) continue;
      const bool inb = a > 0, inf = a < na - 1;
      const double fb = -sgf[r][lx];
      const double Ff = sgf[r + 1][lx];
      double ff = 0.;
      if (inb) ff += fb;
      if (inf) ff += Ff;
      const long c = c_base + a * sD;
      double un = (((ownm >> q) & 1u) ? uq[q] : 0.) - ff;
      if (v >= M && v < 2 * M) {
        double dd = 0.;
        if (inb) dd += 0.5 * fb * -1.;
        if (inf) dd += 0.5 * Ff * 1.;
        dflux[(v - M) * nc + c] = dd;
      }
      if (v >= M && v < 3 * M && un < 0.) un = 0.;
      if (M > 1 && v < 3 * M) {
        const int e = v < M ? v : v < 2 * M ? v - M : v - 2 * M;
        if (un != 0.) held |= 1u << (M * q + e);
        if (un != 0. || ((olds >> (M * q + e)) & 1u)) Uout[v * nc + c] = un;
      } else {
        Uout[v * nc + c] = un;
      }
    }
  }
  if (sparse) {
#pragma unroll
    for (int q = 0; q < MH_TILE_Q; ++q) {
      const int r = ly + 4 * q;
      if (val[q] && r >= 2 && r < 2 + MH_TILE_L)
        S.pm[usel ? 0 : 1][c_base + (abase + r) * sD] = (uint8_t)((held >> (M * q)) & ((1u << M) - 1u));
    }
  }
}

// The same sweep for D = y or z on large meshes, of one environment or (2D) two: each thread marches
// along D over a segment.  A row's phi, face gradient, limited slope, face flux and centre are formed
// once and carried to the next rows in registers (the flux and the U of two rows in LDS, so that 3
// wavefronts fit a SIMD in 3D and in 2D of one environment 4), without a barrier; a row's U, membership
// and upper face nodes are in flight while the row before is worked on.  An environment's slots are
// skipped where no lane holds it in the rows a-3 .. a that the update of row a-2 reaches.  What
// bounds it is memory: 193 us on the 192^3 blast is 4.6 TB/s of its traffic (two halo rows on each
// side are read again), and 46 us on 1023x1021; the tiles take 215 and 53 us.  Segments of 8, 24
// cells: 201, 191 us in 3D, 46 and 80 us in 2D, which runs out of threads.  Two environments in 3D
// hold 220 registers (187 us on the 256x128x128 tube, tiles 182; with 168 they spill: 690 us), so
// they and more environments keep the tiles.  Same formulas in the same order as k_sweep_cell_body.
#define MH_CM_L(DIM) ((DIM) == 3 ? 16 : 8)  // cells along D per segment, about (cell_march_len: 2 on small meshes)
#define MH_CM_HAS(DIM, M) ((M) == 1 || ((DIM) == 2 && (M) == 2))
#define MH_CM_NODES (1L << 29)  // meshes of fewer nodes: 32-bit byte offsets
template <int DIM, int D, int M, int LIM>
__device__ __forceinline__ void k_sweep_cell_march_body(const MhDev& S, int lb, int usel, int first) {
  constexpr int NV = 3 * M + 1, FN = DIM == 3 ? 4 : 2;
  const int nx = S.g.nx, ny = S.g.ny, nz = S.g.nz;
  const int na = D == 1 ? ny : nz;
  const int nt = D == 1 ? (DIM == 3 ? nz : 1) : ny;
  const int nseg = march_nseg(na, S.cm_len);
  const long g = lb * (long)blockDim.x + threadIdx.x;
  if (g >= (long)nx * nseg * nt) return;
  if (mh_halted(S.sc)) return;
  const int i = (int)(g % nx);
  const int rest = (int)(g / nx);
  const int seg = rest % nseg, t = rest / nseg;
  const int a0 = (int)((long)seg * na / nseg), a1 = (int)((long)(seg + 1) * na / nseg);  // cells a0 .. a1-1
  const int steps = (na + nseg - 1) / nseg + 4;  // the longest segment and two halo rows on each side
  const double* __restrict__ Uin = usel ? S.Ub : S.Ua;
  double* __restrict__ Uout = usel ? S.Ua : S.Ub;
  double* __restrict__ dflux = S.dflux;
  const long nc = S.g.nc;
  const unsigned nnx = S.g.nnx, nny = S.g.nny;
  // cells and nodes as 32-bit offsets, so that an access is one base in scalar registers and one
  // offset (the launch sees to it that 8 bytes per node stay below 4 GB)
  const unsigned sD = D == 1 ? nx : nx * ny, c0 = D == 1 ? i + nx * ny * t : i + nx * t;
  const unsigned nD = D == 1 ? nnx : nnx * nny, n0 = D == 1 ? i + nnx * nny * t : i + nnx * t;
  const unsigned fN = D == 1 ? nnx * nny : nnx;  // from a face's first two nodes to the others
  auto at = [](const double* p, unsigned o) { return *(const double*)((const char*)p + 8u * o); };
  auto put = [](double* p, unsigned o, double v) { *(double*)((char*)p + 8u * o) = v; };
  auto node = [&](const double* p, unsigned f, int l) {  // node l of the face whose first node is f
    const unsigned o = f + (l >= 2 ? fN : 0u);
    return *(const double*)((const char*)p + 8u * o + (l == 1 || l == 2 ? 8 : 0));
  };
  const double dt = S.sc->dt;
  const double o2 = (double)S.order2;
  const bool sparse = M > 1 && S.pm[0] != nullptr;
  const uint8_t* __restrict__ pin = S.pm[usel ? 1 : 0];
  uint8_t* __restrict__ pout = S.pm[usel ? 0 : 1];
  auto crow = [&](int a) { return c0 + (unsigned)min(max(a, 0), na - 1) * sD; };
  auto face = [&](int a) { return n0 + (unsigned)min(max(a, 0), na) * nD; };
  auto presence = [&](int a) { return sparse ? (unsigned)pin[crow(a)] : 0u; };
  auto anyof = [&](unsigned b) {  // the environments some lane of the wavefront holds
    unsigned m = (1u << M) - 1u;
    if (sparse) {
#pragma unroll
      for (int e = 0; e < M; ++e)
        if (__ballot((b >> e) & 1u) == 0) m &= ~(1u << e);
    }
    return m;
  };
  // the row in flight: U, membership and volume, and the nodes of its upper face
  double Un[NV], vl = 1., x[FN][DIM], ux[FN];
  unsigned mk = 1, held = 0;
  auto load = [&](int a) {
    const unsigned c = crow(a);
#pragma unroll
    for (int e = 0; e < M; ++e) {
      Un[e] = Un[M + e] = Un[2 * M + e] = 0.;
      if ((held >> e) & 1u) {
        Un[e] = at(Uin + e * nc, c);
        Un[M + e] = at(Uin + (M + e) * nc, c);
        Un[2 * M + e] = at(Uin + (2 * M + e) * nc, c);
      }
    }
    Un[3 * M] = at(Uin + 3 * M * nc, c);
    if (first) {
      mk = S.mask[c];
      vl = at(S.Vl, c);
    }
    const unsigned f = face(a + 1);
#pragma unroll
    for (int l = 0; l < FN; ++l) {
#pragma unroll
      for (int d = 0; d < DIM; ++d) x[l][d] = node(S.xlc[d], f, l);
      ux[l] = node(S.u[D], f, l);
    }
  };
  // carried values of the slots: row a-1's phi, the gradient of face a-1, the upwind value of face a-1
  // where it comes from row a-2; in LDS, U of rows a-1 and a-2 (in turn in 0 and 1) and the flux of face a-2
  double phiP[NV], gP[NV], pfb[NV];
  __shared__ double keep[3 * NV][MH_BLOCK];
  auto kept = [&](int v, int q) -> double& { return keep[3 * v + q][threadIdx.x]; };
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    phiP[v] = gP[v] = pfb[v] = 0.;
    kept(v, 0) = kept(v, 1) = kept(v, 2) = 0.;
  }
  unsigned hist[M];
#pragma unroll
  for (int e = 0; e < M; ++e) hist[e] = 0;
  bool innA = false, upA = false, own1 = false, own2 = false;
  double wA = 0., hhA = 0., xcP = 0., xfP = 0., vfP = 0., wP = 0., lo[FN];
#pragma unroll
  for (int l = 0; l < FN; ++l) lo[l] = node(S.xlc[D], face(a0 - 2), l);
  unsigned pnext = presence(a0 - 2), old1 = 0, old2 = 0;
  held = anyof(pnext);
  load(a0 - 2);
  pnext = presence(a0 - 1);
  for (int st = 0; st < steps; ++st) {
    const int a = a0 - 2 + st;
    const bool val = a >= 0 && a < na, valp = a - 1 >= 0 && a - 1 < na;
    const bool inn = val && valp && st > 0;  // face a
    // row a: U, denominator and centre; the face above it
    double U[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) U[v] = val ? Un[v] : 0.;
    double den = 1.;
    bool own = false;
    if (val) {
      if (first) {
        own = mk != 0;  // an empty cell holds Phi itself and its U starts from 0
        den = own ? vl : 1.;
      } else {
        own = true;
        den = 0.;
#pragma unroll
        for (int k = 0; k < M; ++k) den += Un[k];
      }
    }
    double hi[FN];
#pragma unroll
    for (int l = 0; l < FN; ++l) hi[l] = x[l][D];
    double xc = 0.;
    if constexpr (DIM == 3 && D == 2) {
      xc += lo[0]; xc += lo[1]; xc += lo[2]; xc += lo[3];
      xc += hi[0]; xc += hi[1]; xc += hi[2]; xc += hi[3];
      xc = 0.125 * xc;
    } else if constexpr (DIM == 3) {
      xc += lo[0]; xc += lo[1]; xc += hi[1]; xc += hi[0];
      xc += lo[3]; xc += lo[2]; xc += hi[2]; xc += hi[3];
      xc = 0.125 * xc;
    } else {
      xc += lo[0]; xc += lo[1]; xc += hi[1]; xc += hi[0];
      xc = 0.25 * xc;
    }
#pragma unroll
    for (int l = 0; l < FN; ++l) lo[l] = hi[l];
    double area, xfn = 0., us = 0.;
    if constexpr (DIM == 3) {
      const D3 x0 = d3(x[0][0], x[0][1], x[0][2]), x1 = d3(x[1][0], x[1][1], x[1][2]);
      const D3 x2 = d3(x[2][0], x[2][1], x[2][2]), x3 = d3(x[3][0], x[3][1], x[3][2]);
      const D3 v1 = x2 - x0, v2 = x3 - x1;
      if (D == 1) area = 0.5 * fabs(v2.x * v1.z - v2.z * v1.x);
      else area = 0.5 * fabs(v1.x * v2.y - v1.y * v2.x);
    } else {
      area = fabs(x[1][0] - x[0][0]);
    }
    const double wf = DIM == 3 ? 0.25 : 0.5;
#pragma unroll
    for (int l = 0; l < FN; ++l) xfn += wf * hi[l];
    if (S.csts) {  // the mean of n and n+1 (PrepareRemap.cc:236-240)
#pragma unroll
      for (int l = 0; l < FN; ++l) us += 0.5 * (ux[l] + node(S.un[D], face(a + 1), l));
    } else {
#pragma unroll
      for (int l = 0; l < FN; ++l) us += ux[l];
    }
    const double vfn = wf * us, wn = 1. * vfn * area * dt;
    const unsigned heldc = held;
    old2 = old1;
    if (st + 1 < steps) {  // the next row's loads
      held = anyof(pnext);
      load(a + 1);
      pnext = presence(a + 2);
      if (sparse) old1 = pout[crow(a - 1)];
    }
    const double dxr = inn ? xc - xcP : 1.;
    const bool up = inn && vfP * dxr > 0.0;
    const double hh = inn ? o2 * (xfP - (up ? xcP : xc)) : 0.;
    const double w = inn ? wP : 0.;
    const bool irregular = val && (!mh_finite_nonzero(den) || (inn && (!mh_finite_nonzero(dxr) || !mh_finite(w) || !mh_finite(hh))));
    const unsigned here = sparse && __ballot(irregular) == 0 ? heldc : (1u << M) - 1u;
    const MhRecip rden = mh_denom(den), rdx = mh_denom(dxr);
    const bool out = a - 2 >= a0 && a - 2 < a1;
    const bool inb = a - 2 > 0, inf = a - 2 < na - 1;
    const unsigned c = crow(a - 2);
    unsigned holds = 0;
    auto slot = [&](int v) {
      const double phi = mh_ratio(U[v], rden);
      const double gf = inn ? mh_ratio(phi - phiP[v], rdx) : 0.;
      const double sl = S.order2 && valp ? mh_limited_gradient<LIM>(S.limiter, gP[v], gf) : 0.;
      const double F = innA ? wA * (upA ? pfb[v] : phiP[v] + hhA * sl) : 0.;
      const double fb = -kept(v, 2), U2 = kept(v, st & 1);
      if (out) {
        double ff = 0.;
        if (inb) ff += fb;
        if (inf) ff += F;
        double un = (own2 ? U2 : 0.) - ff;
        if (v >= M && v < 2 * M) {
          double dd = 0.;
          if (inb) dd += 0.5 * fb * -1.;
          if (inf) dd += 0.5 * F * 1.;
          put(dflux + (v - M) * nc, c, dd);
        }
        if (v >= M && v < 3 * M && un < 0.) un = 0.;
        if (M > 1 && v < 3 * M) {
          const int e = v < M ? v : v < 2 * M ? v - M : v - 2 * M;
          if (un != 0.) holds |= 1u << e;
          if (!sparse || un != 0. || ((old2 >> e) & 1u)) put(Uout + v * nc, c, un);
        } else {
          put(Uout + v * nc, c, un);
        }
      }
      pfb[v] = phiP[v] + hh * sl;
      kept(v, 2) = F;
      kept(v, st & 1) = U[v];
      phiP[v] = phi;
      gP[v] = gf;
    };
#pragma unroll
    for (int e = 0; e < M; ++e) {
      hist[e] = ((hist[e] << 1) | ((here >> e) & 1u)) & 15u;
      if (hist[e]) {
        slot(e);
        slot(M + e);
        slot(2 * M + e);
      } else if (out) {
        put(dflux + e * nc, c, 0.);
        if ((old2 >> e) & 1u) {
          put(Uout + e * nc, c, 0.);
          put(Uout + (M + e) * nc, c, 0.);
          put(Uout + (2 * M + e) * nc, c, 0.);
        }
      }
    }
    slot(3 * M);
    if (sparse && out) pout[c] = (uint8_t)holds;
    xfP = xfn;
    vfP = vfn;
    wP = wn;
    innA = inn;
    upA = up;
    wA = w;
    hhA = hh;
    xcP = xc;
    own2 = own1;
    own1 = own;
  }
}

// The same sweep for D = y or z on meshes that do not fill the chip with tiles: each thread holds
// L cells of a column along D (and two halo cells on each side) in registers.  Per remap slot every
// phi, face gradient, limited slope and face flux of the segment is formed once, without LDS or
// barriers, and the chains of the L + 4 rows are independent of one another.  What bounds it is the
// latency of one wavefront (about 2000 instructions and four rounds of loads for seven slots), so
// the slots are shared out too (v0 .. v1-1 here).  Threads are consecutive along x, then over the
// segments of a column, then over the columns, so any nx fills the wavefronts and consecutive
// segments share their halo cells in L2.  Against the tiles, two environments: 15 -> 8 us on
// 100x5x5 cells, 27 -> 10 us on 181x181, 29 -> 21 us on 512x512x1, 44 -> 39 us on 97x61x83; longer
// segments are slower there (four cells: 10, 14, 24, 37 us).  In 2D no branch parts the loads of the
// prologue (y sweep with its events 12.2 -> 11.1 us on 181x181, 21.7 -> 20.4 on 512x512, 41.4 -> 39.9
// on 850x850); in 3D those loads take 214 registers instead of 126: no gain on 16^3 to 64^3, and 33 ->
// 39 us on 80^3.  Same formulas in the same order as k_sweep_cell_body.
#ifndef MH_SEG_L
#define MH_SEG_L 2  // cells along D per thread
#endif
template <int DIM, int D, int M, int LIM, int L>
__device__ __forceinline__ void k_sweep_cell_seg_body(const MhDev& S, int lb, int usel, int first, int v0, int v1) {
  constexpr int R = L + 4;
  constexpr bool FEW = DIM == 2;  // all loads of the prologue in flight together
  const int nx = S.g.nx, ny = S.g.ny, nz = S.g.nz;
  const int na = D == 1 ? ny : nz;
  const int nt = D == 1 ? (DIM == 3 ? nz : 1) : ny;
  const int nseg = seg_count(na, L);
  const long g = lb * (long)blockDim.x + threadIdx.x;
  if (g >= (long)nx * nseg * nt) return;
  const bool halted = mh_halted(S.sc);
  if (!FEW && halted) return;
  const int i = (int)(g % nx);
  const int rest = (int)(g / nx);
  const int abase = (rest % nseg) * L - 2;  // cell along D of row 0
  const int t = rest / nseg;
  const double* __restrict__ Uin = usel ? S.Ub : S.Ua;
  double* __restrict__ Uout = usel ? S.Ua : S.Ub;
  double* __restrict__ dflux = S.dflux;
  const long nc = S.g.nc;
  const long nnx = S.g.nnx, nny = S.g.nny;
  const long sD = D == 1 ? (long)nx : (long)nx * ny;
  const long cl = D == 1 ? i + (long)nx * ny * t : i + (long)nx * t;  // the column's cell and node at 0
  const long c0 = cl + abase * sD;
  const long nD = D == 1 ? nnx : nnx * nny;
  const long nl = D == 1 ? i + nnx * nny * t : i + nnx * t;
  const double dt = S.sc->dt;
  const double o2 = (double)S.order2;
  auto valid = [&](int r) { return abase + r >= 0 && abase + r < na; };
  auto inner = [&](int f) { return valid(f - 1) && valid(f); };  // face f: between rows f-1 and f
  // FEW: a row beyond the mesh is its end row again (unused), so that no branch parts the loads
  auto row = [&](int r) { return min(max(abase + r, 0), na - 1); };
  auto slot_of = [&](int v, int r) {
    if (FEW) return Uin[v * nc + cl + row(r) * sD];
    return valid(r) ? Uin[v * nc + c0 + r * sD] : 0.;
  };
  double u[R], un[R];  // slot loads run one slot ahead
#pragma unroll
  for (int r = 0; r < R; ++r) un[r] = slot_of(v0, r);
  unsigned ownm = 0;  // bit r: the cell's own U enters its update
  MhRecip den[R], dx[R];
  double xc[R], w[R], hh[R], d[R], area[R], xf[R], vf[R];
  unsigned upm = 0;  // bit f: the upwind cell of face f is the one behind it
#pragma unroll
  for (int r = 0; r < R; ++r) {
    d[r] = 1.;
    xc[r] = 0.;
    if (FEW || valid(r)) {
      const long c = cl + row(r) * sD;
      if (first) {
        const bool empty = !S.mask[c];  // an empty cell holds Phi itself and its U starts from 0
        d[r] = empty ? 1. : S.Vl[c];
        if (!empty) ownm |= 1u << r;
      } else {
        ownm |= 1u << r;
        double sv = 0.;
#pragma unroll
        for (int k = 0; k < M; ++k) sv += Uin[k * nc + c];
        d[r] = sv;
      }
      xc[r] = cell_centre_d<DIM, D>(S, nl + row(r) * nD);
    }
  }
#pragma unroll
  for (int f = 2; f <= R - 2; ++f)
    if (FEW || inner(f)) face_quant<DIM, D>(S, nl + row(f) * nD, area[f], xf[f], vf[f]);
  if (FEW && halted) return;
#pragma unroll
  for (int r = 0; r < R; ++r) den[r] = mh_denom(valid(r) ? d[r] : 1.);
#pragma unroll
  for (int f = 1; f < R; ++f) {
    const double dxf = inner(f) ? xc[f] - xc[f - 1] : 1.;
    dx[f] = mh_denom(dxf);
    w[f] = 0.;
    hh[f] = 0.;
    if (f >= 2 && f <= R - 2 && inner(f)) {
      const bool up = vf[f] * dxf > 0.0;
      if (up) upm |= 1u << f;
      hh[f] = o2 * (xf[f] - (up ? xc[f - 1] : xc[f]));
      w[f] = 1. * vf[f] * area[f] * dt;
    }
  }
  for (int v = v0; v < v1; ++v) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      u[r] = un[r];
      if (v + 1 < v1) un[r] = slot_of(v + 1, r);
    }
    double phi[R], gr[R];
    bool bad = false;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      bad |= den[r].bad;
      phi[r] = mh_div(u[r], den[r], bad);
    }
    if (__builtin_expect(bad, 0))
#pragma unroll
      for (int r = 0; r < R; ++r) phi[r] = u[r] / den[r].b;
    bad = false;
#pragma unroll
    for (int f = 1; f < R; ++f) {
      bad |= dx[f].bad;
      gr[f] = mh_div(phi[f] - phi[f - 1], dx[f], bad);
    }
    if (__builtin_expect(bad, 0))
#pragma unroll
      for (int f = 1; f < R; ++f) gr[f] = (phi[f] - phi[f - 1]) / dx[f].b;
#pragma unroll
    for (int f = 1; f < R; ++f)
      if (!inner(f)) gr[f] = 0.;
#pragma unroll
    for (int r = 1; r < R - 1; ++r)  // limited slope of row r in place of its back gradient
      gr[r] = S.order2 && valid(r) ? mh_limited_gradient<LIM>(S.limiter, gr[r], gr[r + 1]) : 0.;
    double F[R];
#pragma unroll
    for (int f = 2; f <= R - 2; ++f) {
      const bool up = (upm >> f) & 1u;
      const double pf = (up ? phi[f - 1] : phi[f]) + hh[f] * (up ? gr[f - 1] : gr[f]);
      F[f] = inner(f) ? w[f] * pf : 0.;
    }
#pragma unroll
    for (int r = 2; r < R - 2; ++r) {
      if (!valid(r)) continue;
      const double fb = -F[r], Ff = F[r + 1];
      double ff = 0.;
      if (inner(r)) ff += fb;
      if (inner(r + 1)) ff += Ff;
      const long c = c0 + r * sD;
      double uo = (((ownm >> r) & 1u) ? u[r] : 0.) - ff;
      if (v >= M && v < 2 * M) {
        double dd = 0.;
        if (inner(r)) dd += 0.5 * fb * -1.;
        if (inner(r + 1)) dd += 0.5 * Ff * 1.;
        dflux[(v - M) * nc + c] = dd;
      }
      if (v >= M && v < 3 * M && uo < 0.) uo = 0.;
      Uout[v * nc + c] = uo;
    }
  }
}

// One ADI direction, dual part for one node: limited nodal velocity gradients
// (computeDualGradPhi UtilesRemap.cc:19-72, computeAndLimitGradPhiDual :369-400), back/front
// mass fluxes gathered from the cells behind/ahead in face order, env order
// (DualPhaseRemap.cc:75-108), upwind momentum update (:110-239), filter and phi (:241-257).
// Nodes with no neighbour along D keep their values.  On the last sweep the node velocity
// u = mu / m is formed for every node (RemapADIFinal.cc:286-297).
// The mass fluxes through an inner node's back and front dual faces along D
// (DualPhaseRemap.cc:75-108): 1/2 (2D) or 1/4 (3D) of the dual mass fluxes of the cells
// behind / ahead of the node, over those cells in face order and the environments in order.
template <int DIM, int D, int M>
__device__ __forceinline__ void dual_mass_fluxes(const MhDev& S, int i, int j, int k, int a, double& back,
                                                 double& front) {
  const int it1 = D == 0 ? j : i, it2 = D == 2 ? j : k;
  back = dual_edge_flux<DIM, D, M>(S, a - 1, it1, it2);
  front = dual_edge_flux<DIM, D, M>(S, a, it1, it2);
}

template <int DIM, int D, int M, int LIM>
__device__ __forceinline__ void k_sweep_node_at(const MhDev& S, long n, int psel, int prev, int last) {
  constexpr int NC = DIM;  // velocity components carried
  const DualBuf din = dual_in<DIM>(S, psel, prev);
  const int nnx = S.g.nnx, nny = S.g.nny;
  const int i = (int)(n % nnx);
  const long r = n / nnx;
  const int j = (int)(r % nny);
  const int k = (int)(r / nny);
  const int a = D == 0 ? i : D == 1 ? j : k;
  const int na = D == 0 ? S.g.nx : D == 1 ? S.g.ny : S.g.nz;
  const long nD = D == 0 ? 1 : D == 1 ? (long)nnx : (long)nnx * nny;
  // earlier sweeps ran along other directions: the nodes of one line along D were all kept by
  // them or none was
  const bool kept = dual_kept<DIM>(S, prev, i, j, k);
  const bool inner = a >= 1 && a <= na - 1;
  // one round of loads, the stop flag included: a node beyond the mesh is its end node again (unused)
  double P[5][NC], X[5], mm[5], fl[2];
#pragma unroll
  for (int o = -2; o <= 2; ++o) {
    const long m2 = n + (min(max(a + o, 0), na) - a) * nD;
#pragma unroll
    for (int cc = 0; cc < NC; ++cc) P[o + 2][cc] = din.v[cc][m2];
    mm[o + 2] = din.m[m2];
    X[o + 2] = S.xlc[D][m2];
  }
  dual_mass_fluxes<DIM, D, M>(S, i, j, k, a, fl[0], fl[1]);
  if (mh_halted(S.sc)) return;
  double U[NC + 1], v0[NC];
  U[NC] = mm[2];
#pragma unroll
  for (int cc = 0; cc < NC; ++cc) {
    v0[cc] = P[2][cc];
    U[cc] = kept ? U[NC] * v0[cc] : v0[cc];
  }
  if (!inner) {
    dual_store<DIM>(S, n, U, v0, psel, last);
    return;
  }
  const double dt = S.sc->dt;
#pragma unroll
  for (int o = -2; o <= 2; ++o) {
    const int bb = a + o;
    if (!kept) {
      const MhRecip rm = mh_denom(mm[o + 2]);
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) P[o + 2][cc] = mh_ratio(P[o + 2][cc], rm);
    }
    if (bb < 0 || bb > na) {
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) P[o + 2][cc] = 0.;
      X[o + 2] = 0.;
    }
  }
  double G[3][NC];
  // coordinates two and three nodes away, for the dual widths of generalised limiters
  double Xmm = 0., Xpp = 0.;
  if (LIM == MH_LIM_ANY) {
    if (a - 3 >= 0) Xmm = S.xlc[D][n - 3 * nD];
    if (a + 3 <= na) Xpp = S.xlc[D][n + 3 * nD];
  }
#pragma unroll
  for (int o = -1; o <= 1; ++o) {
    const int bb = a + o;
    const bool in = S.order2 && bb >= 1 && bb <= na - 1;
    double h0 = 0., hm = 0., hp = 0.;
    if (LIM == MH_LIM_ANY && in) {  // dual cell widths (UtilesRemap.cc:50-61)
      const double xbb = o == -1 ? Xmm : X[o], xff = o == 1 ? Xpp : X[o + 4];
      h0 = 0.5 * (X[o + 3] - X[o + 1]);
      if (bb - 2 < 0) {
        if (bb + 2 <= na) hp = 0.5 * (xff - X[o + 2]);
      } else if (bb + 2 > na) {
        hm = 0.5 * (X[o + 2] - xbb);
      } else {
        hm = 0.5 * (X[o + 2] - xbb);
        hp = 0.5 * (xff - X[o + 2]);
      }
    }
    for (int cc = 0; cc < NC; ++cc) {
      double g = 0.;
      if (in) {
        const double gf = (P[o + 3][cc] - P[o + 2][cc]) / (X[o + 3] - X[o + 2]);
        const double gb = (P[o + 2][cc] - P[o + 1][cc]) / (X[o + 2] - X[o + 1]);
        if (LIM == MH_LIM_ANY && S.limiter >= MH_MINMOD_G) {
          g = flux_limiter_g(S.limiter, gf, gb, P[o + 3][cc], P[o + 1][cc], h0, hp, hm, S.simple_pente);
        } else {
          g = mh_limited_gradient<LIM, true>(S.limiter, gb, gf);
        }
      }
      G[o + 1][cc] = g;
    }
  }
  const double back = fl[0], front = fl[1];
  U[NC] += back - front;
  const double o2 = (double)S.order2;
  const double ufront = 0.5 * (P[2][D] + P[3][D]);
  const int sf = ufront > 0 ? 1 : -1;
  const int fo = (front < 0.) ? 1 : 0;
  const double uback = 0.5 * (P[1][D] + P[2][D]);
  const int sb = uback > 0 ? 1 : -1;
  const int bo = (back > 0.) ? -1 : 0;
  for (int cc = 0; cc < NC; ++cc) {
    const double FU = P[fo + 2][cc] + o2 * (0.5 * G[fo + 1][cc] * (sf * (X[3] - X[2]) - dt * ufront));
    const double BU = P[bo + 2][cc] + o2 * (0.5 * G[bo + 1][cc] * (sb * (X[2] - X[1]) - dt * uback));
    U[cc] += back * BU - front * FU;
  }
  for (int cc = 0; cc < NC; ++cc)
    if (fabs(U[cc]) < 1.e-300) U[cc] = 0.;
  dual_store<DIM>(S, n, U, U, psel, last);
}

template <int DIM, int D, int M, int LIM>
__device__ __forceinline__ void k_sweep_node_body(const MhDev& S, int lb, int psel, int prev, int last) {
  const long n = lb * (long)blockDim.x + threadIdx.x;
  if (n >= S.g.nn) return;
  k_sweep_node_at<DIM, D, M, LIM>(S, n, psel, prev, last);
}

// The y or z dual sweep of one mesh with each thread marching along D over a segment of
// nm_len nodes: the window of phi and coordinates, the edge gradients, the limited gradients
// and the mass flux through the node's front dual face are carried to the next node (they are
// its back-side values), so each is formed once per node instead of by each of the three nodes
// whose update reads it.  Threads of a wave are consecutive along x.  Same formulas and orders
// as k_sweep_node_at (classical limiters; the generalised ones keep k_sweep_node).  What bounds it
// is the latency of a node's loads at 3 waves per SIMD: with the next node's loads issued together
// ahead of this node's arithmetic, y / z take 116 / 114 us on the 256x128x128 tube (2.9 TB/s of the
// bytes it cannot do without) and 166 / 161 us on the 192^3 blast; with one load round per cell of
// a mass flux, waited for where it is added, 165 / 162 and 201 / 198 us at 4 waves.  The segment
// length is per case (the autotuner tries 4-12 nodes): 10 by default on large meshes, 4 on smaller
// ones, which need the threads, and below MH_MARCH_NODES one thread per node (k_sweep_node).
#ifndef MH_NM_L
#define MH_NM_L 10  // default target segment length (MhDev::nm_len; variant march code 0, kMarchLen[0])
#endif
#ifndef MH_NM_MIN_WAVES
#define MH_NM_MIN_WAVES 1
#endif
template <int DIM, int D, int M, int LIM>
__device__ __forceinline__ void k_sweep_node_march_body(const MhDev& S, int lb, int psel, int prev, int last) {
  constexpr int NC = DIM;
  const int nnx = S.g.nnx, nny = S.g.nny;
  const int na = D == 1 ? S.g.ny : S.g.nz;
  const int nt2 = D == 1 ? S.g.nnz : nny;  // the other transverse node count
  const long cols = (long)nnx * nt2;
  const long g = lb * (long)blockDim.x + threadIdx.x;
  const int nseg = march_nseg(na + 1, S.nm_len);  // na + 1 nodes along D
  if (g >= cols * nseg) return;
  const int seg = (int)(g / cols);
  const long rem = g - seg * cols;
  const int i = (int)(rem % nnx), t2 = (int)(rem / nnx);
  const int a0 = (int)((long)seg * (na + 1) / nseg), a1 = (int)((long)(seg + 1) * (na + 1) / nseg);  // nodes a0 .. a1-1
  const long nD = D == 1 ? (long)nnx : (long)nnx * nny;
  const long base = D == 1 ? i + (long)nnx * nny * t2 : i + (long)nnx * t2;  // node at a = 0
  const DualBuf din = dual_in<DIM>(S, psel, prev);
  // one line along D was kept by the earlier sweeps as a whole or not at all
  const bool kept = dual_kept<DIM>(S, prev, i, D == 1 ? 0 : t2, D == 1 ? t2 : 0);
  const double* __restrict__ Xd = S.xlc[D];
  const double dt = S.sc->dt;
  const double o2 = (double)S.order2;
  // a node of the line (beyond its ends the end node again, then set to 0)
  auto fetch = [&](int b, double* v, double& m, double& X) {
    const long m2 = base + min(max(b, 0), na) * nD;
#pragma unroll
    for (int cc = 0; cc < NC; ++cc) v[cc] = din.v[cc][m2];
    m = din.m[m2];
    X = Xd[m2];
  };
  auto phi = [&](int b, const double* v, double m, double* P, double& X) {
#pragma unroll
    for (int cc = 0; cc < NC; ++cc) P[cc] = v[cc];
    if (!kept) {
      const MhRecip rm = mh_denom(m);
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) P[cc] = mh_ratio(v[cc], rm);
    }
    if (b < 0 || b > na) {
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) P[cc] = 0.;
      X = 0.;
    }
  };
  // limited gradient of node b from the edge gradients behind (gb) and ahead (gf)
  auto limited = [&](int b, const double* gb, const double* gf, double* G) {
    const bool in = S.order2 && b >= 1 && b <= na - 1;
#pragma unroll
    for (int cc = 0; cc < NC; ++cc) {
      G[cc] = in ? dual_limited<LIM>(S, gb[cc], gf[cc]) : 0.;
    }
  };
  // edge gradient between nodes b and b+1 (formed only where a limited gradient reads it)
  auto edge = [&](int b, const double* P0, double X0, const double* P1, double X1, double* E) {
    const bool used = S.order2 && b >= 0 && b + 1 <= na && (b >= 1 || b + 1 <= na - 1);
    const MhRecip rX = mh_denom(X1 - X0);
#pragma unroll
    for (int cc = 0; cc < NC; ++cc) E[cc] = used ? mh_ratio(P1[cc] - P0[cc], rX) : 0.;
  };
  // window: P and X of nodes a-1 .. a+2 (slots 0..3), edges (a-1/2, a+1/2, a+3/2), G of a-1, a, a+1
  double P[4][NC], X[4], E[3][NC], G[3][NC];
  double U1[NC + 1], back, front;  // U of the next node, and the fluxes through its dual faces
  const int j0 = D == 1 ? 0 : t2, k0 = D == 1 ? t2 : 0;  // transverse node position (the D one is a)
  const int it1 = i, it2 = D == 1 ? k0 : j0;  // transverse cells: x, and z or y
  {
    double v[5][NC], m[5], Xs[5];
#pragma unroll
    for (int o = 0; o < 5; ++o) fetch(a0 - 2 + o, v[o], m[o], Xs[o]);
    back = dual_edge_flux<DIM, D, M>(S, a0 - 1, it1, it2);
    front = dual_edge_flux<DIM, D, M>(S, a0, it1, it2);
    if (mh_halted(S.sc)) return;
    double Pm2[NC];
    phi(a0 - 2, v[0], m[0], Pm2, Xs[0]);
#pragma unroll
    for (int o = 0; o < 4; ++o) {
      X[o] = Xs[o + 1];
      phi(a0 - 1 + o, v[o + 1], m[o + 1], P[o], X[o]);
    }
#pragma unroll
    for (int cc = 0; cc < NC; ++cc) U1[cc] = v[2][cc];
    U1[NC] = m[2];
    double Em[NC];  // edge a0 - 3/2
    edge(a0 - 2, Pm2, Xs[0], P[0], X[0], Em);
#pragma unroll
    for (int o = 0; o < 3; ++o) edge(a0 - 1 + o, P[o], X[o], P[o + 1], X[o + 1], E[o]);
    limited(a0 - 1, Em, E[0], G[0]);
    limited(a0, E[0], E[1], G[1]);
    limited(a0 + 1, E[1], E[2], G[2]);
  }
  for (int a = a0; a < a1; ++a) {
    const long n = base + a * nD;
    // the next node's loads go out before this one's arithmetic: its U and front flux, and the node
    // three ahead that enters the window (the state of node a + 1 is read a second time, from L2:
    // carrying it costs a wave per SIMD)
    const bool more = a + 1 < a1;
    double U2[NC + 1], v3[NC], m3 = 0., X3 = 0., front2 = 0.;
    if (more) {
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) U2[cc] = din.v[cc][n + nD];
      U2[NC] = din.m[n + nD];
      fetch(a + 3, v3, m3, X3);
      front2 = dual_edge_flux<DIM, D, M>(S, a + 1, it1, it2);
    }
    double U[NC + 1], v0[NC];
    U[NC] = U1[NC];
#pragma unroll
    for (int cc = 0; cc < NC; ++cc) {
      v0[cc] = U1[cc];
      U[cc] = kept ? U[NC] * v0[cc] : v0[cc];
    }
    if (!(a >= 1 && a <= na - 1)) {
      dual_store<DIM>(S, n, U, v0, psel, last);
    } else {
      U[NC] += back - front;
      const double ufront = 0.5 * (P[1][D] + P[2][D]);
      const int sf = ufront > 0 ? 1 : -1;
      const bool fo = front < 0.;
      const double uback = 0.5 * (P[0][D] + P[1][D]);
      const int sb = uback > 0 ? 1 : -1;
      const bool bo = back > 0.;
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) {
        const double FU = (fo ? P[2][cc] : P[1][cc]) + o2 * (0.5 * (fo ? G[2][cc] : G[1][cc]) * (sf * (X[2] - X[1]) - dt * ufront));
        const double BU = (bo ? P[0][cc] : P[1][cc]) + o2 * (0.5 * (bo ? G[0][cc] : G[1][cc]) * (sb * (X[1] - X[0]) - dt * uback));
        U[cc] += back * BU - front * FU;
      }
#pragma unroll
      for (int cc = 0; cc < NC; ++cc)
        if (fabs(U[cc]) < 1.e-300) U[cc] = 0.;
      dual_store<DIM>(S, n, U, U, psel, last);
    }
    if (more) {  // slide the window one node along D
#pragma unroll
      for (int o = 0; o < 3; ++o) {
        X[o] = X[o + 1];
#pragma unroll
        for (int cc = 0; cc < NC; ++cc) P[o][cc] = P[o + 1][cc];
      }
      X[3] = X3;
      phi(a + 3, v3, m3, P[3], X[3]);
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) {
        E[0][cc] = E[1][cc];
        E[1][cc] = E[2][cc];
        G[0][cc] = G[1][cc];
        G[1][cc] = G[2][cc];
      }
      edge(a + 2, P[2], X[2], P[3], X[3], E[2]);
      limited(a + 2, E[1], E[2], G[2]);
#pragma unroll
      for (int cc = 0; cc <= NC; ++cc) U1[cc] = U2[cc];
      back = front;
      front = front2;
    }
  }
}


// u = mu / m for every node with a non-zero projected mass (RemapADIFinal.cc:286-297), for
// cycles whose remap has a single sweep (the sweep kernel still reads u; prev is its direction)
// or none (prev 0: u and the node mass).
template <int DIM>
__device__ __forceinline__ void k_node_velocity_body(const MhDev& S, int lb, int prev) {
  const long n = lb * (long)blockDim.x + threadIdx.x;
  if (n >= S.g.nn) return;
  if (mh_halted(S.sc)) return;
  const DualBuf din = dual_in<DIM>(S, 1, prev);  // the first sweep writes buffer A
  const int i = (int)(n % S.g.nnx);
  const long r = n / S.g.nnx;
  const bool kept = dual_kept<DIM>(S, prev, i, (int)(r % S.g.nny), (int)(r / S.g.nny));
  const double m = din.m[n];
  if (m != 0.)
    for (int cc = 0; cc < DIM; ++cc) {
      const double v = din.v[cc][n];
      S.u[cc][n] = (kept ? m * v : v) / m;
    }
}

// ------------------------------------------------- conservation-energie-totale (RemapADI.axl:178)
// The dual kinetic energy of one sweep along D, run after the node sweep of that direction:
// dual U = 1/2 m |u|^2 and phi = 1/2 |u|^2 at the first sweep (PrepareRemap.cc:179-190), then
// for inner nodes the upwind phi through the back and front dual faces with the node sweep's
// mass fluxes and upwind choices (DualPhaseRemap.cc:132-238).  Its limited gradient is never
// formed (UtilesRemap.cc:369-400 covers the velocity only), so the slope term multiplies 0.
// phi = U / the node mass the node sweep has just written (:251-257).
template <int DIM, int D, int M>
__device__ __forceinline__ void k_sweep_ke_body(const MhDev& S, int lb, int psel, int prev) {
  const long n = lb * (long)blockDim.x + threadIdx.x;
  if (n >= S.g.nn) return;
  if (mh_halted(S.sc)) return;
  const int first = prev == 0;
  const DualBuf din = dual_in<DIM>(S, psel, prev);
  const double* __restrict__ Kin = psel ? S.ke_Pa : S.ke_Pb;
  double* __restrict__ Kout = psel ? S.ke_Pb : S.ke_Pa;
  const int nnx = S.g.nnx, nny = S.g.nny;
  const int i = (int)(n % nnx);
  const long r = n / nnx;
  const int j = (int)(r % nny);
  const int k = (int)(r / nny);
  const int a = D == 0 ? i : D == 1 ? j : k;
  const int na = D == 0 ? S.g.nx : D == 1 ? S.g.ny : S.g.nz;
  const long nD = D == 0 ? 1 : D == 1 ? (long)nnx : (long)nnx * nny;
  auto sq = [&](long m2) {
    const double ux = S.u[0][m2], uy = S.u[1][m2];
    double v = ux * ux + uy * uy;
    if (DIM == 3) v = v + S.u[2][m2] * S.u[2][m2];
    return v;
  };
  auto phi = [&](long m2) { return first ? 0.5 * sq(m2) : Kin[m2]; };
  double U = first ? 0.5 * S.mn[n] * sq(n) : S.ke_U[n];
  if (!(a >= 1 && a <= na - 1)) {
    S.ke_U[n] = U;
    Kout[n] = phi(n);
    return;
  }
  double back, front;
  dual_mass_fluxes<DIM, D, M>(S, i, j, k, a, back, front);
  const double dt = S.sc->dt;
  const double o2 = (double)S.order2;
  const double zero_slope = 0.;
  const bool kept = dual_kept<DIM>(S, prev, i, j, k);  // of the whole line along D
  auto vel = [&](long m2) { return kept ? din.v[D][m2] : din.v[D][m2] / din.m[m2]; };
  const double xb = S.xlc[D][n - nD], xn = S.xlc[D][n], xf = S.xlc[D][n + nD];
  const double ufront = 0.5 * (vel(n) + vel(n + nD));
  const int sf = ufront > 0 ? 1 : -1;
  const double FE = phi(front < 0. ? n + nD : n) + o2 * (0.5 * zero_slope * (sf * (xf - xn) - dt * ufront));
  const double uback = 0.5 * (vel(n - nD) + vel(n));
  const int sb = uback > 0 ? 1 : -1;
  const double BE = phi(back > 0. ? n - nD : n) + o2 * (0.5 * zero_slope * (sb * (xn - xb) - dt * uback));
  U += back * BE - front * FE;
  S.ke_U[n] = U;
  Kout[n] = U / dual_out_m<DIM>(S, psel)[n];
}

// The dual state of a remap with no sweep (every direction one cell wide): the mass and the
// kinetic energy 1/2 m |u|^2, untouched by any sweep (PrepareRemap.cc:169-190).
template <int DIM>
__device__ __forceinline__ void k_dual_init_body(const MhDev& S, int lb) {
  const long n = lb * (long)blockDim.x + threadIdx.x;
  if (n >= S.g.nn) return;
  if (mh_halted(S.sc)) return;
  const long nn = S.g.nn;
  const double mass = S.mn[n];
  double v = 0.;
  for (int cc = 0; cc < DIM; ++cc) {
    const double uc = S.u[cc][n];
    v = cc == 0 ? uc * uc : v + uc * uc;
  }
  S.Ud[DIM * nn + n] = mass;
  S.ke_U[n] = 0.5 * mass * v;
}

// The kinetic energy each cell gets back (RemapADIFinal.cc:318-339), once the node velocity
// is final: over the cell's nodes in cell order, 0.25 (also in 3D) times the projected
// minus the reconstructed kinetic energy per unit mass, for nodes with a non-zero projected
// mass; kept if positive (std::max(0., .)).  k_finalize adds it to the internal energies.
template <int DIM>
__device__ __forceinline__ void k_cons_ec_body(const MhDev& S, int lb, int psel) {
  const long c = lb * (long)blockDim.x + threadIdx.x;
  if (c >= S.g.nc) return;
  if (mh_halted(S.sc)) return;
  const double* __restrict__ mass = dual_out_m<DIM>(S, psel);  // as the last sweep left it
  const int i = (int)(c % S.g.nx);
  const long r = c / S.g.nx;
  const int j = (int)(r % S.g.ny);
  const int k = (int)(r / S.g.ny);
  const long nnx = S.g.nnx, nnxy = (long)S.g.nnx * S.g.nny;
  const long b = i + nnx * (j + (long)S.g.nny * k);
  const long off[8] = {0, 1, 1 + nnx, nnx, nnxy, 1 + nnxy, 1 + nnx + nnxy, nnx + nnxy};
  double d = 0.;
#pragma unroll
  for (int l = 0; l < (DIM == 3 ? 8 : 4); ++l) {
    const long n = b + off[l];
    const double mp = mass[n];
    if (mp != 0.) {
      const double ux = S.u[0][n], uy = S.u[1][n];
      double v = ux * ux + uy * uy;
      if (DIM == 3) v = v + S.u[2][n] * S.u[2][n];
      const double ec_proj = S.ke_U[n] / mp;
      const double ec_reconst = 0.5 * v;
      d += 0.25 * (ec_proj - ec_reconst);
    }
  }
  S.dec[c] = (0. < d) ? d : 0.;
}

// ----------------------------------------------------------------------------- finalize
// remapVariables (RemapADIFinal.cc:21-316), the remap tail (PrepareRemap.cc:220-249:
// applyEOS per environment, computePressionMoyenne) and the per-cell CFL candidate of
// computeDeltaT (MahycoModule.cc:1763-1779).  Pure cells write through the global arrays
// only (their environment value is the global value).
template <int DIM, int M>
__device__ __forceinline__ void k_finalize_body(const MhDev& S, int lb, int usel) {
  const double* __restrict__ Uin = usel ? S.Ub : S.Ua;
  const long c = lb * (long)blockDim.x + threadIdx.x;
  const bool halted = mh_halted(S.sc);
  const bool active = c < S.g.nc && !halted;
  double dxs = 1.79769313486231570815e+308;
  if (c < S.g.nc) {
    // everything the cell reads goes out together: the node velocities and L of the CFL candidate,
    // the membership and VE, then the slots, which wait for the presence byte (35.5 -> 32.6 us on
    // 1023x1021, 165 -> 147 us for 64 meshes of 64^2 to 512^2; large 3D meshes are as before)
    const long nc = S.g.nc;
    const double thr = S.thr_remap;
    double U[3 * M + 1];
    const unsigned held = M > 1 && S.pm[0] ? S.pm[usel ? 1 : 0][c] : ~0u;
    const double VE = S.VE[c];
    const uint8_t om = S.mask[c];
    const double Lc = S.L[c];
    U[3 * M] = Uin[3 * M * nc + c];
    const int ci = (int)(c % S.g.nx), cj = (int)(c / S.g.nx % S.g.ny), ck = (int)(c / S.g.nx / S.g.ny);
    const double vmax2 = cell_vmax2<DIM>(S, ci + (long)S.g.nnx * (cj + (long)S.g.nny * ck));
    for (int v = 0; v < 3 * M; ++v) U[v] = ((held >> (v % M)) & 1u) ? Uin[v * nc + c] : 0.;
    if (active) {
    if (S.pb && S.nsweep > 0) {  // phi the last sweep left (RemapADIService.cc:493-538): what the
                                  // next cycle's first sweep sees for non-member environments
      double sv = 0.;
      for (int kk = 0; kk < M; ++kk) sv += U[kk];
      for (int kk = 0; kk < M; ++kk) {
        S.phi0[kk * nc + c] = U[kk] / sv;
        S.phi0[(M + kk) * nc + c] = U[kk] != 0. ? U[M + kk] / U[kk] : 0.;
      }
      for (int kk = 0; kk < M; ++kk) S.phi0[(2 * M + kk) * nc + c] = U[M + kk] != 0. ? U[2 * M + kk] / U[M + kk] : 0.;
    }
    // environment membership (:29-78)
    uint8_t nm = om;
    for (int kk = 0; kk < M; ++kk) {
      const bool was = (om >> kk) & 1;
      if (((U[kk] / VE) < thr || (U[M + kk] == 0. && !S.sans_lagrange)) && was) {
        nm &= (uint8_t)~(1u << kk);
      } else if ((U[kk] / VE) > thr && !was) {
        double volt = 0.;
        for (int k2 = 0; k2 < M; ++k2) volt += U[k2];
        const double vol_ev = U[kk] * VE / volt;
        if ((vol_ev / VE) > thr && U[M + kk] != 0.) nm |= (uint8_t)(1u << kk);
      }
    }
    const bool pure = __popc(nm) == 1;
    // (:85-216)
    const double vol = VE;
    double volt = 0., masset = 0., vn1[M];
    for (int kk = 0; kk < M; ++kk) {
      vn1[kk] = U[kk];
      volt += vn1[kk];
      masset += U[M + kk];
    }
    const double unsurvolt = 1. / volt;
    for (int kk = 0; kk < M; ++kk) vn1[kk] *= vol * unsurvolt;
    double f[M], chi[M], dk[M], ek[M], pk[M], ck[M];
    double somme_frac = 0.;
    const double unsurvol = 1. / vol;
    for (int kk = 0; kk < M; ++kk) {
      f[kk] = 0.;
      if (!((nm >> kk) & 1)) continue;
      f[kk] = vn1[kk] * unsurvol;
      if (f[kk] < thr) f[kk] = 0.;
      somme_frac += f[kk];
    }
    double unsursomme = 0.;
    if (somme_frac != 0.) unsursomme = 1. / somme_frac;
    for (int kk = 0; kk < M; ++kk)
      if ((nm >> kk) & 1) f[kk] *= unsursomme;
    if (S.est) {  // mixed-cell flag for the order-3 remap of the next cycle (:124-145)
      int cnt = 0, pu = -1;
      for (int kk = 0; kk < M; ++kk)
        if (f[kk] > 0.) {
          cnt++;
          pu = kk;
        }
      S.est[c] = (int8_t)(cnt > 1 ? MH_EST_MIXED : pu);
    }
    if (masset > thr * thr) {
      const double unsurmasset = 1. / masset;
      double fm = 0.;
      for (int kk = 0; kk < M; ++kk) {
        chi[kk] = 0.;
        if (!((nm >> kk) & 1)) continue;
        chi[kk] = U[M + kk] * unsurmasset;
        if (f[kk] < thr) chi[kk] = 0.;
        fm += chi[kk];
      }
      if (fm != 0.) {
        const double unsurfm = 1. / fm;
        for (int kk = 0; kk < M; ++kk)
          if ((nm >> kk) & 1) chi[kk] *= unsurfm;
      }
    } else {
      // (near-)empty cell: the reference keeps the mass fractions it holds after the
      // membership change -- the global value for a single-environment cell (taken from
      // the remaining environment's partial value when the cell was mixed), the partial
      // values for a mixed cell (0 for environments that have just entered; all partial
      // values restart from 0 and the global value when a pure cell turns mixed)
      const int on = __popc(om), nnb = __popc(nm);
      for (int kk = 0; kk < M; ++kk) {
        chi[kk] = 0.;
        if (!((nm >> kk) & 1)) continue;
        if (nnb == 1) chi[kk] = on == 1 ? S.chig[c] : S.chik[kk * nc + c];
        else if (on == 1) chi[kk] = ((om >> kk) & 1) ? S.chig[c] : 0.;
        else chi[kk] = ((om >> kk) & 1) ? S.chik[kk * nc + c] : 0.;
      }
    }
    double density = 0.;
    for (int kk = 0; kk < M; ++kk) {
      dk[kk] = 0.;
      if (!((nm >> kk) & 1)) continue;
      if (f[kk] > thr && vn1[kk] != 0.) dk[kk] = U[M + kk] / vn1[kk];
      density += f[kk] * dk[kk];
    }
    for (int kk = 0; kk < M; ++kk) {
      ek[kk] = 0.;
      if (!((nm >> kk) & 1)) continue;
      if (f[kk] > thr && U[M + kk] != 0.) ek[kk] = U[2 * M + kk] / U[M + kk];
    }
    // writes, with the aliasing of single-environment cells (:221-253)
    double rho_g = density;
    double M_g = VE * density;
    double e_g, q_g;
    double Mk[M], qk[M];
    double energie = 0., pseudo = 0.;
    for (int kk = 0; kk < M; ++kk) {
      if (!((nm >> kk) & 1)) continue;
      Mk[kk] = chi[kk] * M_g;
      if (pure) M_g = Mk[kk];
      qk[kk] = (S.q_frozen ? S.Vl[c] * S.q[c] : U[3 * M]) * unsurvol;
      if (pure) rho_g = dk[kk];
      energie += chi[kk] * ek[kk];
      pseudo += f[kk] * qk[kk];
    }
    e_g = energie;
    q_g = pseudo;
    for (int kk = 0; kk < M; ++kk) {
      if (!((nm >> kk) & 1)) continue;
      if (pure) ek[kk] = e_g;  // the cell value overwrites the aliased environment value
      if (dk[kk] < 0. || ek[kk] < 0.) {
        ek[kk] = 0.;
        dk[kk] = 0.;
        f[kk] = 0.;
        chi[kk] = 0.;
        if (pure) {
          e_g = 0.;
          rho_g = 0.;
        }
      }
      if (dk[kk] != dk[kk] || ek[kk] != ek[kk]) S.err[0] = MH_ERR_NAN_REMAP;
    }
    if (S.dec) {  // conservation-energie-totale (RemapADIFinal.cc:340-344): the energy k_cons_ec
                  // found, to each environment by its mass fraction (for a single-environment
                  // cell that is the cell value) and to the value of any other cell
      const double dec = S.dec[c];
      for (int kk = 0; kk < M; ++kk) {
        if (!((nm >> kk) & 1)) continue;
        if (pure) {
          e_g += chi[kk] * dec;
          ek[kk] = e_g;
        } else {
          ek[kk] += chi[kk] * dec;
        }
      }
      if (!pure) e_g += dec;
    }
    // applyEOS per environment, computePressionMoyenne (MahycoModule.cc:1708-1735)
    double p_g = 0., c_g = 0.;
    const double opt = S.vitson_max ? 1. : 0.;
    const double tnow = S.sc->t + S.sc->dt;  // m_global_time of this iteration
    for (int kk = 0; kk < M; ++kk) {
      if (!((nm >> kk) & 1)) continue;
      if (S.env[kk].fictif) {
        fictif_eos(S.env[kk], tnow, pure ? S.p[c] : S.pk[kk * nc + c], pk[kk], ck[kk]);
        ek[kk] = 0.;
        if (pure) e_g = 0.;
      } else {
        eos(S.env[kk], pure ? rho_g : dk[kk], ek[kk], pk[kk], ck[kk]);
      }
      if (pure) {
        p_g = pk[kk];
        c_g = ck[kk];
      }
    }
    if (!pure && S.sans_lagrange) {  // computePressionMoyenne returns at once (:1711)
      p_g = S.p[c];
      c_g = S.c[c];
    } else if (!pure) {
      p_g = 0.;
      c_g = 0.;
      for (int kk = 0; kk < M; ++kk) {
        if (!((nm >> kk) & 1)) continue;
        p_g += f[kk] * pk[kk];
        c_g = opt * ((ck[kk] < c_g) ? c_g : ck[kk]);
        c_g += (1. - opt) * f[kk] * ck[kk];
      }
    }
    if (!pure) {
      for (int kk = 0; kk < M; ++kk) {
        if (!((nm >> kk) & 1)) continue;
        const long o = kk * nc + c;
        S.fk[o] = f[kk];
        S.chik[o] = chi[kk];
        S.rhok[o] = dk[kk];
        S.ek[o] = ek[kk];
        S.pk[o] = pk[kk];
        S.Mk[o] = Mk[kk];
      }
    }
    // the global volume and mass fractions are the environment values of a
    // single-environment cell; a mixed cell keeps the global values it had (Arcane leaves
    // them untouched).  Partial mass fractions follow Arcane's membership change: all
    // restart from 0 when a pure cell turns mixed, and the environment that replaces the
    // only one of a pure cell starts from 0
    if (pure) {
      double fg = 0., cg = 0.;
      for (int kk = 0; kk < M; ++kk)
        if ((nm >> kk) & 1) {
          fg = f[kk];
          cg = chi[kk];
        }
      S.fg[c] = fg;
      S.chig[c] = cg;
    }
    if (nm != om && __popc(om) == 1) {  // a mixed cell's old partial values are kept
      for (int kk = 0; kk < M; ++kk) {
        const bool now = (nm >> kk) & 1, was = (om >> kk) & 1;
        if (now && !pure) continue;  // written below with the cell's partial values
        if (pure ? (now && !was) : !now) S.chik[kk * nc + c] = 0.;
      }
    }
    S.mask[c] = nm;
    if (S.csts) {  // CSTS history: mixed cells' partial pseudo-viscosity, the mask before this remap
      S.qem1[c] = S.qe[c];
      S.qe[c] = (S.q_frozen ? S.Vl[c] * S.q[c] : U[3 * M]) * unsurvol;
      S.mkm1[c] = om;
    }
    S.rho[c] = rho_g;
    S.e[c] = e_g;
    S.p[c] = p_g;
    S.c[c] = c_g;
    S.q[c] = q_g;
    S.M[c] = M_g;
    dxs = Lc / (c_g + sqrt(vmax2));
    }
  }
  block_min_store(dxs, active, S.partial, lb);
}

// applyEOS of one environment on its member cells (PerfectGasEOSService.cc:45-67,
// StiffenedGasEOSService.cc:43-63), as a standalone call.
__device__ __forceinline__ void apply_eos_at(const MhDev& S, int env, long c) {
  const uint8_t mk = S.mask[c];
  if (!((mk >> env) & 1)) return;
  const double tnow = S.sc->t;  // between iterations: m_global_time of the last one
  if (__popc(mk) == 1) {
    double p, cs;
    if (S.env[env].fictif) {
      fictif_eos(S.env[env], tnow, S.p[c], p, cs);
      S.e[c] = 0.;
    } else {
      eos(S.env[env], S.rho[c], S.e[c], p, cs);
    }
    S.p[c] = p;
    S.c[c] = cs;
  } else {
    const long o = env * S.g.nc + c;
    double p, cs;
    if (S.env[env].fictif) {
      fictif_eos(S.env[env], tnow, S.pk[o], p, cs);
      S.ek[o] = 0.;
    } else {
      eos(S.env[env], S.rhok[o], S.ek[o], p, cs);
    }
    S.pk[o] = p;
  }
}
template <int U = 0>
__global__ __launch_bounds__(MH_BLOCK) void k_apply_eos(MhDev S, int env) {
  const long c = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (c >= S.g.nc) return;
  apply_eos_at(S, env, c);
}
// applyOneCellEOS (IEquationOfState.h:50-52): the same for one cell
template <int U = 0>
__global__ __launch_bounds__(64) void k_apply_eos_cell(MhDev S, int env, long c) {
  if (threadIdx.x == 0) apply_eos_at(S, env, c);
}

// computePressionMoyenne (MahycoModule.cc:1708-1735) on multi-environment cells; the
// environment sound speeds are those applyEOS stores for the stored density and energy
// (1 for a Fictif environment, FictifEOSService.cc:62).  Advection mode returns at once
// (:1711): the host launches nothing then.
template <int M>
__global__ __launch_bounds__(MH_BLOCK) void k_pression_moyenne(MhDev S) {
  const long c = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (c >= S.g.nc || S.sans_lagrange) return;
  const uint8_t mk = S.mask[c];
  if (__popc(mk) == 1) return;
  const double opt = S.vitson_max ? 1. : 0.;
  double ps = 0., cm = 0.;
  for (int kk = 0; kk < M; ++kk) {
    if (!((mk >> kk) & 1)) continue;
    const long o = kk * S.g.nc + c;
    double p, cs = 1.;
    if (!S.env[kk].fictif) eos(S.env[kk], S.rhok[o], S.ek[o], p, cs);
    ps += S.fk[o] * S.pk[o];
    cm = opt * ((cs < cm) ? cm : cs);
    cm += (1. - opt) * S.fk[o] * cs;
  }
  S.p[c] = ps;
  S.c[c] = cm;
}

// The CFL minimum of computeDeltaT (MahycoModule.cc:1767-1792) from the per-block minima
// partial[2b] (and NaN flags partial[2b+1]) of nblocks blocks, in cell order.  Called by every
// thread of a one-block launch; returns true on thread 0 only, with the minimum in *mn.
__device__ __forceinline__ bool cfl_fold(const double* __restrict__ partial, int nblocks, double* mn) {
  __shared__ double rm[MH_DT_BLOCK / 64];
  __shared__ int rn[MH_DT_BLOCK / 64];
  const int nw = (int)(blockDim.x >> 6), lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  __shared__ int any_nan;
  // without a NaN candidate anywhere the fold is a plain minimum, in any order
  if (threadIdx.x == 0) any_nan = 0;
  __syncthreads();
  // eight partials in flight per thread, the last one again where there are fewer (the minimum of
  // non-NaN values depends neither on the order nor on a repetition)
  double pm = __longlong_as_double(0x7ff8000000000000LL);
  int pn = 0;
  const int bd = (int)blockDim.x;
  for (int b = threadIdx.x; b < nblocks; b += 8 * bd) {
    double m[8], f[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int o = min(b + u * bd, nblocks - 1);
      m[u] = partial[2 * o];
      f[u] = partial[2 * o + 1];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      pm = min_skip_nan(pm, m[u]);
      pn |= f[u] != 0.;
    }
  }
  for (int off = 32; off > 0; off >>= 1) pm = min_skip_nan(pm, __shfl_xor(pm, off, 64));
  if (__ballot(pn) != 0 && lane == 0) any_nan = 1;
  if (lane == 0) rm[wid] = pm;
  __syncthreads();
  MhCflMin tot;
  if (!any_nan) {
    if (threadIdx.x != 0) return false;
    tot.nan = 0;
    tot.m = rm[0];
    for (int w = 1; w < nw; ++w) tot.m = min_skip_nan(tot.m, rm[w]);
  } else {
    // block partials in block (= cell) order: wavefront w folds a contiguous run of them,
    // 64 at a time, then the wavefronts are combined in order
    __syncthreads();
    const int chunk = ((nblocks + nw - 1) / nw + 63) / 64 * 64;
    const int bbeg = wid * chunk, bend = min(nblocks, bbeg + chunk);
    MhCflMin acc = cfl_leaf(0., false);
    for (int b0 = bbeg; b0 < bend; b0 += 64) {
      const int b = b0 + lane;
      MhCflMin o = cfl_leaf(0., false);
      if (b < bend) {
        o.m = partial[2 * b];
        o.nan = partial[2 * b + 1] != 0.;
      }
      o = cfl_wave(o);
      acc = cfl_combine(acc, o);  // lane 0 holds the run's value; other lanes are ignored
    }
    if (lane == 0) {
      rm[wid] = acc.m;
      rn[wid] = acc.nan;
    }
    __syncthreads();
    if (threadIdx.x != 0) return false;
    tot.m = rm[0];
    tot.nan = rn[0];
    for (int w = 1; w < nw; ++w) {
      MhCflMin o;
      o.m = rm[w];
      o.nan = rn[w];
      tot = cfl_combine(tot, o);
    }
  }
  *mn = tot.nan ? tot.m : amin(1.79769313486231570815e+308, tot.m);
  return true;
}

// computeDeltaT (MahycoModule.cc:1739-1864) on the block minima, plus the time increment
// of the iteration and the final-time stop rule.  One block.
__device__ __forceinline__ void k_dt_body(const MhDev& S) {
  MhScalars* sc = S.sc;
  // the scalars are read ahead of the fold: one round of loads instead of three
  const bool halted = mh_halted(sc);
  const double dt = sc->dt, t0 = sc->t;
  const int it = sc->iteration + 1;
  int status = S.err[0];
  double mn;
  if (!cfl_fold(S.partial, S.nblk_c, &mn) || halted) return;
  const double t = t0 + dt;
  double new_dt = S.cfl * mn;
  new_dt = amin(new_dt, 1.05 * dt);
  new_dt = amin(new_dt, S.dtmax);
  if (S.sans_lagrange) new_dt = S.dt_init;  // advection mode keeps deltat-init (:1751-1753)
  else if (status == 0 && new_dt < S.dtmin) status = MH_ERR_DT_MIN;
  sc->t = t;
  sc->iteration = it;
  sc->dxmin = mn;
  if (status != 0) {
    sc->status = status;
    return;
  }
  sc->dt_old = dt;
  sc->dt = new_dt;
  const double T = S.tfinal;
  if ((t < T && t + new_dt > T) || t > T) sc->stopped = 1;
  if (S.max_iter > 0 && it >= S.max_iter) sc->stopped = 1;
}


// ----------------------------------------------------------------------------- time history
// EnvSummationService::write (time_history/EnvSummationService.cc:77-169) every hist_period
// iterations: per environment the plain mean of M_k and p_k over its cells, the
// volume-weighted density and the mass-weighted internal energy.  Runs after k_dt; both
// kernels do nothing unless the iteration just completed is a new multiple of the period.
__device__ __forceinline__ bool hist_due(const MhDev& S) {
  const MhScalars* sc = S.sc;
  return S.hist_period > 0 && sc->status == 0 && sc->iteration > 0 &&
         (sc->iteration % S.hist_period) == 0 && sc->iteration != sc->hist_last && sc->hist_rows < S.hist_max;
}

template <int M>
__device__ __forceinline__ void k_hist_part_body(const MhDev& S, int lb) {
  __shared__ double red[6 * M][MH_BLOCK / 64];
  if (!hist_due(S)) return;
  const long c = lb * (long)blockDim.x + threadIdx.x;
  double acc[6 * M];
  for (int v = 0; v < 6 * M; ++v) acc[v] = 0.;
  if (c < S.g.nc) {
    const uint8_t mk = S.mask[c];
    const bool pure = __popc(mk) == 1;
    const double V = S.with_proj ? S.VE[c] : S.Vl[c];
    const long nc = S.g.nc;
    for (int k = 0; k < M; ++k) {
      if (!((mk >> k) & 1)) continue;
      const long o = k * nc + c;
      const double Mk = pure ? S.M[c] : S.Mk[o];
      const double pk = pure ? S.p[c] : S.pk[o];
      const double rk = pure ? S.rho[c] : S.rhok[o];
      const double ek = pure ? S.e[c] : S.ek[o];
      const double Vk = pure ? V : S.fk[o] * V;
      acc[6 * k + 0] = 1.;
      acc[6 * k + 1] = Mk;
      acc[6 * k + 2] = pk;
      acc[6 * k + 3] = rk * Vk;
      acc[6 * k + 4] = Vk;
      acc[6 * k + 5] = ek * Mk;
    }
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  for (int v = 0; v < 6 * M; ++v) {
    double x = acc[v];
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
    if (lane == 0) red[v][wid] = x;
  }
  __syncthreads();
  if (threadIdx.x < 6 * M) {
    double x = 0.;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) x += red[threadIdx.x][w];
    S.hist_part[(long)lb * 6 * M + threadIdx.x] = x;
  }
}

template <int M>
__device__ __forceinline__ void k_hist_final_body(const MhDev& S) {
  if (!hist_due(S)) return;
  MhScalars* sc = S.sc;
  const int v = threadIdx.x;
  __shared__ double tot[6 * M];
  if (v < 6 * M) {
    double x = 0.;
    for (int b = 0; b < S.nblk_c; ++b) x += S.hist_part[(long)b * 6 * M + v];
    tot[v] = x;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  double* row = S.hist + (long)sc->hist_rows * (1 + 5 * M);
  row[0] = sc->t;
  for (int k = 0; k < M; ++k) {
    const double cnt = tot[6 * k + 0];
    row[1 + 5 * k + 0] = cnt > 0. ? tot[6 * k + 1] / cnt : 0.;
    row[1 + 5 * k + 1] = cnt > 0. ? tot[6 * k + 2] / cnt : 0.;
    row[1 + 5 * k + 2] = cnt > 0. ? tot[6 * k + 3] / tot[6 * k + 4] : 0.;
    row[1 + 5 * k + 3] = cnt > 0. ? tot[6 * k + 5] / tot[6 * k + 1] : 0.;
    row[1 + 5 * k + 4] = cnt;
  }
  sc->hist_rows = sc->hist_rows + 1;
  sc->hist_last = sc->iteration;
}

template <int M>
__global__ __launch_bounds__(MH_BLOCK) void k_hist_part(MhDev S) { k_hist_part_body<M>(S, (int)blockIdx.x); }
template <int M>
__global__ __launch_bounds__(MH_BLOCK) void k_hist_final(MhDev S) { k_hist_final_body<M>(S); }

// ----------------------------------------------------------------------------- wrappers
// Single mesh: the state travels by value in the kernel arguments.  Batch: one launch
// covers many meshes; block b works on mesh bmap[b].x, local block bmap[b].y, whose state
// is tab[bmap[b].x] (meshes of one launch share DIM, M and the sweep direction).
// Single-mesh grids use the XCD-contiguous block order of xcd_block.

#ifndef MH_NODE_FLAT_MIN_WAVES
#define MH_NODE_FLAT_MIN_WAVES 2  // register budget of k_node_lag, in waves per SIMD
#endif
#ifndef MH_CELL_MIN_WAVES
#define MH_CELL_MIN_WAVES 3  // register budget of k_cell_lag, in waves per SIMD
#endif
#ifndef MH_NODE_MIN_WAVES
#define MH_NODE_MIN_WAVES 1  // register budget of k_node_lag3_tiled, in waves per SIMD
#endif
// Batched variants are persistent: a fixed grid walks the work list bmap[0 .. *nwork) (one
// entry per (case, block) of every case of a batch group) with a grid stride, so the list and
// its length can change between launches of a captured graph without re-capture.  An entry of a mesh
// whose run has ended is passed over: 32 meshes of 200^2 with half of them ended take 231 us an iteration
// instead of 266, with all of them 25 instead of 107, at the same 366 us with none.  (With the first entries
// let through as in late_halted, 241, 36 and 378 us.)
#define MH_WRAP(NAME, WAVES, TPL, TARGS, PARAMS, ARGS)                                      \
  TPL __global__ __launch_bounds__(MH_BLOCK, WAVES) void NAME(MhDev S PARAMS) {              \
    if (late_halted(S.sc)) return;                                                           \
    NAME##_body TARGS(S, xcd_block((int)blockIdx.x, (int)gridDim.x) ARGS);                   \
  }                                                                                          \
  TPL __global__ __launch_bounds__(MH_BLOCK, WAVES) void NAME##_batch(                        \
      const MhDev* __restrict__ tab, const int2* __restrict__ bmap, const int* __restrict__ nwork PARAMS) { \
    const int n = *nwork;                                                                    \
    for (int w = (int)blockIdx.x; w < n; w += (int)gridDim.x) {                              \
      const int2 bm = bmap[w];                                                               \
      if (!mh_halted(tab[bm.x].sc)) NAME##_body TARGS(tab[bm.x], bm.y ARGS);                 \
      __syncthreads();                                                                       \
    }                                                                                        \
  }
#define MH_COMMA ,
MH_WRAP(k_node_lag, MH_NODE_FLAT_MIN_WAVES, template <int DIM>, <DIM>, , )
MH_WRAP(k_cell_lag, MH_CELL_MIN_WAVES, template <int DIM MH_COMMA int M>, <DIM MH_COMMA M>, , )
MH_WRAP(k_cell_lag_remap, MH_CELL_MIN_WAVES, template <int DIM MH_COMMA int M>, <DIM MH_COMMA M>, , )
// (Single meshes only.  LATE: blocks ask for the stop flag ahead, as above; in a few rounds of blocks at 3
// waves per SIMD that wait shows, 46 -> 48 us on 128x96x64, so the launch asks for it from 8192 blocks on.)
template <int DIM, int M, bool LATE>
__global__ __launch_bounds__(MH_BLOCK, MH_CELL_MIN_WAVES) void k_cell_lag_only(MhDev S) {
  if (LATE && late_halted(S.sc)) return;
  k_cell_lag_only_body<DIM, M>(S, xcd_block((int)blockIdx.x, (int)gridDim.x));
}
MH_WRAP(k_cell_lag_csts, 1, template <int DIM MH_COMMA int M>, <DIM MH_COMMA M>, , )
MH_WRAP(k_cell_length, 1, template <int DIM>, <DIM>, , )
MH_WRAP(k_sweep_cell, 1, template <int DIM MH_COMMA int D MH_COMMA int M MH_COMMA int LIM>, <DIM MH_COMMA D MH_COMMA M MH_COMMA LIM>,
        MH_COMMA int usel MH_COMMA int first, MH_COMMA usel MH_COMMA first)
MH_WRAP(k_sweep_node, 1, template <int DIM MH_COMMA int D MH_COMMA int M MH_COMMA int LIM>,
        <DIM MH_COMMA D MH_COMMA M MH_COMMA LIM>,
        MH_COMMA int psel MH_COMMA int prev MH_COMMA int last, MH_COMMA psel MH_COMMA prev MH_COMMA last)
MH_WRAP(k_node_velocity, 1, template <int DIM>, <DIM>, MH_COMMA int prev, MH_COMMA prev)
MH_WRAP(k_finalize, 1, template <int DIM MH_COMMA int M>, <DIM MH_COMMA M>, MH_COMMA int usel, MH_COMMA usel)
MH_WRAP(k_sweep_cell_row, 1, template <int DIM MH_COMMA int M MH_COMMA int LIM>, <DIM MH_COMMA M MH_COMMA LIM>,
        MH_COMMA int usel MH_COMMA int first, MH_COMMA usel MH_COMMA first)
MH_WRAP(k_sweep_cell_tile, MH_TILE_MIN_WAVES,
        template <int DIM MH_COMMA int D MH_COMMA int M MH_COMMA int LIM>, <DIM MH_COMMA D MH_COMMA M MH_COMMA LIM>,
        MH_COMMA int usel MH_COMMA int first, MH_COMMA usel MH_COMMA first)
MH_WRAP(k_sweep_cell_march, 1, template <int DIM MH_COMMA int D MH_COMMA int M MH_COMMA int LIM>,
        <DIM MH_COMMA D MH_COMMA M MH_COMMA LIM>, MH_COMMA int usel MH_COMMA int first, MH_COMMA usel MH_COMMA first)
MH_WRAP(k_sweep_node_row, 1, template <int DIM MH_COMMA int M MH_COMMA int LIM>, <DIM MH_COMMA M MH_COMMA LIM>,
        MH_COMMA int psel MH_COMMA int prev MH_COMMA int last, MH_COMMA psel MH_COMMA prev MH_COMMA last)
MH_WRAP(k_hcell, 1, template <int DIM>, <DIM>, , )
MH_WRAP(k_node_adv, 1, template <int DIM>, <DIM>, , )
MH_WRAP(k_node_fwd, 1, template <int DIM>, <DIM>, , )
MH_WRAP(k_sweep_cell_gen, 1, template <int DIM MH_COMMA int D MH_COMMA int M>, <DIM MH_COMMA D MH_COMMA M>,
        MH_COMMA int usel MH_COMMA int first, MH_COMMA usel MH_COMMA first)
MH_WRAP(k_sweep_ke, 1, template <int DIM MH_COMMA int D MH_COMMA int M>, <DIM MH_COMMA D MH_COMMA M>, MH_COMMA int psel MH_COMMA int prev,
        MH_COMMA psel MH_COMMA prev)
MH_WRAP(k_dual_init, 1, template <int DIM>, <DIM>, , )
MH_WRAP(k_cons_ec, 1, template <int DIM>, <DIM>, MH_COMMA int psel, MH_COMMA psel)
MH_WRAP(k_prepare_remap, 1, template <int DIM MH_COMMA int M>, <DIM MH_COMMA M>, , )
MH_WRAP(k_sweep_node_march, MH_NM_MIN_WAVES, template <int DIM MH_COMMA int D MH_COMMA int M MH_COMMA int LIM>,
        <DIM MH_COMMA D MH_COMMA M MH_COMMA LIM>,
        MH_COMMA int psel MH_COMMA int prev MH_COMMA int last, MH_COMMA psel MH_COMMA prev MH_COMMA last)

// Small meshes: the remap slots of a cell are shared out over the gridDim.y rows of the grid, vper
// each, so that a mesh of a few hundred wavefronts fills the chip and each thread forms the
// geometry and one or a few slots instead of all 3m+1 one after the other.
template <int DIM, int M, int LIM>
__global__ __launch_bounds__(MH_BLOCK) void k_sweep_cell_row_slots(MhDev S, int usel, int first, int vper) {
  if (late_halted(S.sc)) return;
  const int v0 = (int)blockIdx.y * vper;
  k_sweep_cell_row_body<DIM, M, LIM>(S, xcd_block((int)blockIdx.x, (int)gridDim.x), usel, first, v0,
                                     min(v0 + vper, 3 * M + 1));
}
template <int DIM, int D, int M, int LIM, int L>
__global__ __launch_bounds__(MH_BLOCK) void k_sweep_cell_seg(MhDev S, int usel, int first, int vper) {
  if (late_halted(S.sc)) return;
  const int v0 = (int)blockIdx.y * vper;
  k_sweep_cell_seg_body<DIM, D, M, LIM, L>(S, xcd_block((int)blockIdx.x, (int)gridDim.x), usel, first, v0,
                                           min(v0 + vper, 3 * M + 1));
}
// The order-3 sweep: gridDim.y rows of the grid share out the environments and V q, eper each.
template <int DIM, int D, int M>
__global__ __launch_bounds__(MH_BLOCK, 2) void k_sweep_cell3(MhDev S, int usel, int first, int eper) {
  const int e0 = (int)blockIdx.y * eper;
  k_sweep_cell3_body<DIM, D, M, MH_O3_L>(S, xcd_block((int)blockIdx.x, (int)gridDim.x), usel, first, e0,
                                         min(e0 + eper, M + 1));
}
template <int DIM, int D, int M>
__global__ __launch_bounds__(MH_BLOCK, 2) void k_sweep_cell3_batch(const MhDev* __restrict__ tab,
                                                                const int2* __restrict__ bmap,
                                                                const int* __restrict__ nwork, int usel, int first) {
  const int n = *nwork;
  for (int w = (int)blockIdx.x; w < n; w += (int)gridDim.x) {
    const int2 bm = bmap[w];
    k_sweep_cell3_body<DIM, D, M, MH_O3_L>(tab[bm.x], bm.y, usel, first, 0, M + 1);
    __syncthreads();
  }
}
// (the plain kernels are templates with an unused parameter, so that every translation unit
// that launches one may instantiate it)
template <int U = 0>
__global__ __launch_bounds__(MH_BLOCK, MH_NODE_MIN_WAVES) void k_node_lag3_tiled(MhDev S) {
  k_node_lag3_tiled_body(S, blockIdx.x, blockIdx.y, blockIdx.z);
}

template <int U = 0>
__global__ __launch_bounds__(MH_BLOCK) void k_node_lag3_split(MhDev S) {
  k_node_lag3_split_body(S, xcd_block((int)blockIdx.x, (int)gridDim.x));
}

template <int U = 0>
__global__ __launch_bounds__(MH_DT_BLOCK) void k_dt(MhDev S) { k_dt_body(S); }
template <int M>
__global__ __launch_bounds__(MH_BLOCK, MH_CT_MIN_WAVES) void k_cell_lag3_tiled(MhDev S) {
  k_cell_lag3_tiled_body<M>(S, blockIdx.x, blockIdx.y, blockIdx.z);
}
template <int U = 0>
__global__ __launch_bounds__(MH_DT_BLOCK) void k_dt_batch(const MhDev* __restrict__ tab,
                                                          const int* __restrict__ list,
                                                          const int* __restrict__ nlist) {
  const int n = *nlist;
  for (int w = (int)blockIdx.x; w < n; w += (int)gridDim.x) {
    k_dt_body(tab[list[w]]);
    __syncthreads();
  }
}
// The z-marching node kernel over a batch group: work item (case, tile), tile index
// bx + ntx (by + nty bz) with ntx, nty the case's tile counts along x and y.
template <int U = 0>
__global__ __launch_bounds__(MH_BLOCK, MH_NODE_MIN_WAVES) void k_node_lag3_tiled_batch(
    const MhDev* __restrict__ tab, const int2* __restrict__ bmap, const int* __restrict__ nwork) {
  const int n = *nwork;
  for (int w = (int)blockIdx.x; w < n; w += (int)gridDim.x) {
    const int2 bm = bmap[w];
    const MhDev& S = tab[bm.x];
    const int ntx = (S.g.nnx + MH_NTX - 1) / MH_NTX, nty = (S.g.nny + MH_NTY - 1) / MH_NTY;
    k_node_lag3_tiled_body(S, bm.y % ntx, (bm.y / ntx) % nty, bm.y / (ntx * nty));
    __syncthreads();
  }
}

#endif
