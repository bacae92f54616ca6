// mmf_mesh.hip -- the finite-volume step on an explicit interface list
// (the general MeshGeometricalInfo, mesh_info.hpp:31-105 / mesh_info.cpp:86-118):
// any conforming or hanging-face mesh given as owner / neighbour / area /
// normal per face and a volume per cell, order 1 (reconstruction.cpp:90-97).
//
// One kernel per RK stage (k_mesh_stage), one thread per cell: the cell's
// flux tuple once, then its incident faces in increasing face index (the order
// the reference's interface loop reaches them, euler.cpp:153-247: RHS -= A*F
// as owner, += A*F as neighbour), each from the other cell's state or the
// border's or wall's virtual state (euler.cpp:198-225), and the stage update
// with the cell's own volume (main.cpp:409-495).  An incidence is 8 bytes: the
// other cell and the face's kind; the next incidence's state is loaded while
// this one's flux is formed.  Both cells of a face evaluate it: a face kernel
// writing A*F for a cell kernel to sum halves the fluxes, but the 40 bytes per
// face it writes and the cell kernel reads twice cost more (us per step, with a
// face kernel / without: 491,520 octree cells 188 / 116, 61,440 66 / 41, 7,680
// 39 / 33; 3.9 million cells 1341 / 858).  What bounds it now is FP64 issue: 215
// instructions per incidence, a third of them the other cell's tuple.
//
// dt is known before stage 1 (Ctrl::lam_now): stage 3 gathers the maximum of
// the step that follows from the state it writes, and closes the step.  No
// float atomics: every cell sums in the reference's face order, so the results
// are bitwise reproducible and equal to a serial interface loop over the list.
#include <hip/hip_runtime.h>

#include "mmf_device.hpp"
#include "mmf_internal.hpp"
#include "mmf_mesh.hpp"
#include "mmf_stage.hpp"

namespace mmf {

// Cells per block: one wave.  Small meshes do not fill the chip, and their waves
// wait for the chain of their cells' faces; blocks of four waves leave three
// CUs of four idle (us per step, four waves / one: octree of 2,512 cells 38.4 /
// 33.7, with reflecting borders 44.2 / 38.4, 7,680 40.5 / 33.2 and 47.6 / 37.1,
// 15,000 38.8 / 33.4; 61,440 and 491,520 39.2 and 124, both).
constexpr int MB = 64;

__device__ __forceinline__ bool mesh_solved(const MeshDev &m, int64_t c) {
  return m.flags == nullptr || (m.flags[c] & CELL_SOLVED);
}

// euler.cpp:261-376: the virtual state beyond a border or wall face, from the
// fluid side's state and the normal pointing out of the fluid.
__device__ __forceinline__ void mesh_bc_state(const MeshDev &m, uint32_t kind, const double *n, const double *fluid,
                                              double *out) {
  const int bc = (int)(kind & MESH_KIND_BC_MASK) - 1;
  if (bc == BC_REFLECTING || bc == BC_WALL) {
    reflect_general(n, fluid, out);
  } else if (bc == BC_DIRICHLET) {
    prim2cons(m.info + NF * ((kind >> MESH_KIND_SLOT_SHIFT) & 0xffff), out);
  } else {
#pragma unroll
    for (int k = 0; k < NF; ++k) out[k] = fluid[k];
  }
}

// Owner-outward normal of incidence e.
__device__ __forceinline__ void mesh_normal(const MeshDev &m, int64_t e, uint32_t kind, double *n) {
  const uint32_t nc = (kind >> MESH_KIND_NRM_SHIFT) & 7;
  if (nc == MESH_NRM_GENERAL) {
    const int64_t f = m.inc[e] >> 1;
    n[0] = m.normal[f];
    n[1] = m.normal[m.F + f];
    n[2] = m.normal[2 * m.F + f];
  } else {  // +-e_a: the same doubles as the caller's (1 or -1, and +0)
    const double s = (nc & 1) ? -1.0 : 1.0;
    n[0] = (nc >> 1) == 0 ? s : 0.0;
    n[1] = (nc >> 1) == 1 ? s : 0.0;
    n[2] = (nc >> 1) == 2 ? s : 0.0;
  }
}

__device__ __forceinline__ double mesh_area(const MeshDev &m, int64_t e, uint32_t kind) {
  const uint32_t as = (kind >> MESH_KIND_AREA_SHIFT) & 255;
  return (as == MESH_AREA_GENERAL) ? m.area[m.inc[e] >> 1] : m.area_tab[as];
}

__device__ __forceinline__ double normal_velocity(const Tup &t, const double *n) {
  return (t.vel[0] * n[0] + t.vel[1] * n[1] + t.vel[2] * n[2]);  // utils.cpp:37-40
}

// One incidence's contribution to the cell's residual (euler.cpp:237-247 with
// eval_splitting, euler.cpp:42-73): own and other tuple, owner-outward normal
// n, area a; as_neigh: the cell is the face's neighbour (R) side.  The two
// physical fluxes are added whichever side is whose, and R - L is other - own
// up to its sign, so own and other need not be swapped into L and R.
__device__ __forceinline__ double mesh_face(const Tup &own, const Tup &oth, const double *n, double a, bool as_neigh,
                                            double *rhs) {
  const double un = normal_velocity(own, n), uo = normal_velocity(oth, n);
  const double ln = fabs(un) + own.a, lo = fabs(uo) + oth.a;
  const double lambdaL = as_neigh ? lo : ln, lambdaR = as_neigh ? ln : lo;
  const double lam = (lambdaR < lambdaL) ? lambdaL : lambdaR;
  const double s = as_neigh ? 1.0 : -1.0, sl = s * lam, sa = s * a;
  const double mn = own.c[FID_RHO] * un, mo = oth.c[FID_RHO] * uo;
  rhs[0] += sa * (0.5 * ((mn + mo) + sl * (oth.c[0] - own.c[0])));
#pragma unroll
  for (int b = 0; b < 3; ++b) {
    const double fn = mn * own.vel[b] + own.p * n[b], fo = mo * oth.vel[b] + oth.p * n[b];
    rhs[1 + b] += sa * (0.5 * ((fn + fo) + sl * (oth.c[1 + b] - own.c[1 + b])));
  }
  rhs[4] += sa * (0.5 * ((un * own.H + uo * oth.H) + sl * (oth.c[4] - own.c[4])));
  return lam;
}

// What the faces of solved cell c, in state u, bring to the stage-1 maximum of
// a step that starts from it (euler.cpp:232-234): the cell's own side of every
// face, the virtual states, and the side of unsolved neighbours (whose state
// does not change); a solved neighbour brings its own side.
__device__ __forceinline__ double mesh_cell_lam(const MeshDev &m, int64_t c, const double *u, const double *U) {
  // axis-aligned faces between solved cells (and free-flow borders, copies):
  // |u_a| + c along the axes the cell has faces on
  const uint32_t axes = m.lam_axes[c];
  if (axes) return cell_max_eig_axes(u, axes);
  Tup T;
  make_tup_fast(u, T);
  double l = 0.0;
  const int64_t e1 = m.off[c + 1];
  for (int64_t e = m.off[c]; e < e1; ++e) {
    const uint32_t kind = m.adj_kind[e];
    double n[3];
    mesh_normal(m, e, kind, n);
    l = lam_acc(l, fabs(normal_velocity(T, n)) + T.a);
    double v[NF];
    if (kind & MESH_KIND_BC_MASK) {
      if ((kind & MESH_KIND_BC_MASK) - 1 == BC_FREE_FLOW) continue;  // a copy
      const double s = (kind & MESH_KIND_NEIGH) ? -1. : 1.;
      const double loc[3] = {s * n[0], s * n[1], s * n[2]};
      mesh_bc_state(m, kind, loc, u, v);
    } else {
      const int64_t o = m.adj[e];
      if (mesh_solved(m, o)) continue;
#pragma unroll
      for (int k = 0; k < NF; ++k) v[k] = U[k * m.fs + o];
    }
    Tup V;
    make_tup(v, V);
    l = lam_acc(l, fabs(normal_velocity(V, n)) + V.a);
  }
  return l;
}

// Ctrl::lam_now (zero beforehand) from state U.
__global__ __launch_bounds__(MB) void k_mesh_lam(MeshDev m, const double *U, Ctrl *ctrl) {
  const int64_t c = (int64_t)blockIdx.x * MB + threadIdx.x;
  double l = 0.0;
  if (c < m.N && mesh_solved(m, c)) {
    double u[NF];
#pragma unroll
    for (int k = 0; k < NF; ++k) u[k] = U[k * m.fs + c];
    l = mesh_cell_lam(m, c, u, U);
  }
  const unsigned long long b = wave_max_u64(dbits(l));
  if ((threadIdx.x & 63) == 0 && b) atomicMax(&ctrl->lam_now, b);
}

// The other cell and the kind of every incidence, from the face arrays.
__global__ __launch_bounds__(MB) void k_mesh_adjacency(MeshDev m, int64_t n, int32_t *adj, uint32_t *adj_kind) {
  const int64_t e = (int64_t)blockIdx.x * MB + threadIdx.x;
  if (e >= n) return;
  const int32_t v = m.inc[e], f = v >> 1;
  adj[e] = (v & 1) ? m.owner[f] : m.neigh[f];
  adj_kind[e] = (uint32_t)m.kind[f] | ((v & 1) ? MESH_KIND_NEIGH : 0u);
}

// Per cell, the axes of its faces if its maximum is that of |u_a| + c along
// them (mesh_cell_lam), else 0.
__global__ __launch_bounds__(MB) void k_mesh_lam_axes(MeshDev m, uint8_t *lam_axes) {
  const int64_t c = (int64_t)blockIdx.x * MB + threadIdx.x;
  if (c >= m.N) return;
  uint32_t axes = 0;
  bool plain = true;
  for (int64_t e = m.off[c]; e < m.off[c + 1]; ++e) {
    const uint32_t kind = m.adj_kind[e], nc = (kind >> MESH_KIND_NRM_SHIFT) & 7, bc = kind & MESH_KIND_BC_MASK;
    plain = plain && nc != MESH_NRM_GENERAL && (bc ? bc - 1 == BC_FREE_FLOW : mesh_solved(m, m.adj[e]));
    axes |= 1u << (nc >> 1);
  }
  lam_axes[c] = plain ? (uint8_t)axes : 0;
}

// Stage 1 reads X = U and writes W1 (out), stage 2 reads X = W1 and writes W2
// to W, stage 3 reads X = W2 and writes U.  W is the reference's one stage
// buffer: an unsolved cell keeps what it holds there (main.cpp:411-414,
// 447-450), which stage 1 copies beside W1.  RHS only: the residual of X = U
// as rows [cells][5], as the host takes them.
template <int STAGE>
__global__ __launch_bounds__(MB, 4) void k_mesh_stage(MeshDev m, const double *__restrict__ X, const double *U,
                                                   const double *W, double *out, Ctrl *ctrl, int mode) {
  const bool step = mode == MODE_STEP;
  const int64_t c = (int64_t)blockIdx.x * MB + threadIdx.x;
  const int64_t fs = m.fs;
  const bool live = c < m.N, sv = live && mesh_solved(m, c);
  const bool run = !step || ctrl->t < ctrl->tmax;  // main.cpp:377 loop guard
  const double dt = step ? step_dt_early(ctrl) : 0.0;
  double lam = 0.0, lam_nx = 0.0;
  NegCount neg;
  if (sv && run) {
    double Xc[NF], Xo[NF];
    const int64_t e0 = m.off[c], e1 = m.off[c + 1];
    // other cell and kind of this incidence and the next one
    int32_t o = 0, o_nx = 0;
    uint32_t kind = 0, kind_nx = 0;
    if (e0 < e1) {
      o = m.adj[e0];
      kind = m.adj_kind[e0];
    }
    if (e0 + 1 < e1) {
      o_nx = m.adj[e0 + 1];
      kind_nx = m.adj_kind[e0 + 1];
    }
#pragma unroll
    for (int k = 0; k < NF; ++k) Xc[k] = X[k * fs + c];
#pragma unroll
    for (int k = 0; k < NF; ++k) Xo[k] = X[k * fs + (o < 0 ? (int32_t)c : o)];
    double a = (e0 < e1) ? mesh_area(m, e0, kind) : 0.0;
    Tup Tc;
    make_tup_fast(Xc, Tc);
    double rhs[NF] = {0., 0., 0., 0., 0.};  // euler.cpp:142-148
    for (int64_t e = e0; e < e1; ++e) {
      // the next incidence's state and the one after it
      double Xn[NF];
      int32_t o2 = 0;
      uint32_t kind2 = 0;
#pragma unroll
      for (int k = 0; k < NF; ++k) Xn[k] = X[k * fs + (o_nx < 0 ? (int32_t)c : o_nx)];
      const double a_nx = (e + 1 < e1) ? mesh_area(m, e + 1, kind_nx) : 0.0;
      if (e + 2 < e1) {
        o2 = m.adj[e + 2];
        kind2 = m.adj_kind[e + 2];
      }
      const bool as_neigh = kind & MESH_KIND_NEIGH;
      double n[3];
      mesh_normal(m, e, kind, n);
      bool count = !as_neigh;
      if (kind & MESH_KIND_BC_MASK) {
        // the fluid side is this cell: the boundary state sees its outward
        // normal (euler.cpp:219-222); the flux keeps the owner's
        const double s = as_neigh ? -1. : 1.;
        const double loc[3] = {s * n[0], s * n[1], s * n[2]};
        double v[NF];
        mesh_bc_state(m, kind, loc, Xc, v);
#pragma unroll
        for (int k = 0; k < NF; ++k) Xo[k] = v[k];
        count = true;
      } else if (as_neigh && m.flags) {
        count = !(m.flags[o] & CELL_SOLVED);
      }
      Tup To;
      make_tup_fast(Xo, To);
      lam = lam_acc(lam, mesh_face(Tc, To, n, a, as_neigh, rhs));
      if (count && (tup_negative(Tc) | tup_negative(To))) neg.add(Tc, To);
#pragma unroll
      for (int k = 0; k < NF; ++k) Xo[k] = Xn[k];
      a = a_nx;
      o = o_nx;
      kind = kind_nx;
      o_nx = o2;
      kind_nx = kind2;
    }
    if (!step) {
#pragma unroll
      for (int k = 0; k < NF; ++k) out[NF * c + k] = rhs[k];
    } else {
      double x[NF], q[NF], nu[NF];
#pragma unroll
      for (int k = 0; k < NF; ++k) x[k] = dt * rhs[k];
      const double V = m.vol[c];  // rawGetCellVolume
      div5(x, V, quot_rcp(V), quot_divisor(V), q);
#pragma unroll
      for (int k = 0; k < NF; ++k) {
        // stage 1: u + q (main.cpp:421), 2: main.cpp:457, 3: main.cpp:493
        nu[k] = rk_update_q<STAGE>(STAGE == 1 ? 0.0 : U[k * fs + c], Xc[k], q[k]);
        out[k * fs + c] = nu[k];
      }
      if (STAGE == 3) lam_nx = mesh_cell_lam(m, c, nu, U);
    }
  } else if (live && run) {
    if (!step) {
#pragma unroll
      for (int k = 0; k < NF; ++k) out[NF * c + k] = 0.0;
    } else if (STAGE == 1) {
#pragma unroll
      for (int k = 0; k < NF; ++k) out[k * fs + c] = W[k * fs + c];
    }
  }
  if (!run) return;  // uniform over the grid
  if (__any(neg.p | neg.r)) neg.flush(ctrl, threadIdx.x);
  if (STAGE == 1 && step) return;  // its maximum was known before the step
  block_max_to<MB>(ctrl, step ? STAGE - 1 : 3, lam, threadIdx.x);
  if (STAGE == 3 && step) {
    block_lam_to<MB>(ctrl, lam_nx, threadIdx.x);
    close_step<true>(ctrl, threadIdx.x);
  }
}

hipError_t launch_mesh_stage(const MeshDev &m, int stage, const double *X, const double *U, const double *W,
                             double *out, Ctrl *ctrl, int mode, hipStream_t s) {
  const dim3 grid((unsigned)((m.N + MB - 1) / MB)), block(MB);
  switch (stage) {
    case 1: hipLaunchKernelGGL(k_mesh_stage<1>, grid, block, 0, s, m, X, U, W, out, ctrl, mode); break;
    case 2: hipLaunchKernelGGL(k_mesh_stage<2>, grid, block, 0, s, m, X, U, W, out, ctrl, mode); break;
    default: hipLaunchKernelGGL(k_mesh_stage<3>, grid, block, 0, s, m, X, U, W, out, ctrl, mode);
  }
  return hipGetLastError();
}

hipError_t launch_mesh_lam(const MeshDev &m, const double *U, Ctrl *ctrl, hipStream_t s) {
  hipLaunchKernelGGL(k_mesh_lam, dim3((unsigned)((m.N + MB - 1) / MB)), dim3(MB), 0, s, m, U, ctrl);
  return hipGetLastError();
}

hipError_t launch_mesh_adjacency(const MeshDev &m, int64_t n, int32_t *adj, uint32_t *adj_kind, uint8_t *lam_axes,
                                 hipStream_t s) {
  if (n < 1) return hipSuccess;
  hipLaunchKernelGGL(k_mesh_adjacency, dim3((unsigned)((n + MB - 1) / MB)), dim3(MB), 0, s, m, n, adj, adj_kind);
  hipLaunchKernelGGL(k_mesh_lam_axes, dim3((unsigned)((m.N + MB - 1) / MB)), dim3(MB), 0, s, m, lam_axes);
  return hipGetLastError();
}

}  // namespace mmf
