// mmf_brick_o2.hip -- order-2 (limited linear) stage kernel on bricks (gfx950).
//
// A wave owns 8 x 8 cells of an xy plane; in 3D a block stacks four of them to
// an 8 x 8 x 4 brick, in 2D it is one wave.  FP64 issue bounds the order-2
// stage (a face value's flux tuple costs more than its flux), so the brick is
// laid out to build every tuple once and to evaluate every face once:
//   - a cell builds, along each axis, the tuples of its two face values;
//   - the brick's outer faces need the facing value of the cell beyond, two
//     per line of cells: 256 lines in 3D (32 in 2D), one per lane, each lane
//     holding its line's two outer cells, so that all of them take one pass.
// That is 7 tuples and 3 faces per 3D cell (5 and 2 in 2D), the faces above the
// brick in a second evaluation per axis that fills 8 to 32 lanes of a wave.  The
// gather kernel builds 12 (8) and the marching kernel, which it replaces, 10 on 5
// faces.
// The tuple of a cell's upper face value goes to the next cell, and that
// cell's lower face flux back, through LDS.  Along x and y both ends are lanes
// of one wave, whose LDS operations execute in order, so only the z axis has
// block barriers (three, and one after the states are stored).
//
// Border faces: beyond a non-periodic border the outer cell's slot holds the
// border cell's own state, so the one-sided difference is zero and with it the
// slope (reconstruction.cpp:67-97 extension: face value = mean), and the
// line's tuple is that of the virtual state (euler.cpp:261-376).
//
// dt depends on the face values' maximum, which only the stage itself forms:
// stage 1 writes R, stage 2 rebuilds W1 = U + dt R / V where it loads; stage 3
// closes the step.  Residuals are summed in the reference's face order:
// results equal the gather kernel's and the oracle's bit for bit.
#include <hip/hip_runtime.h>

#include "mmf_brick.hpp"
#include "mmf_device.hpp"
#include "mmf_internal.hpp"
#include "mmf_stage.hpp"

namespace mmf {

namespace {

// LDS written by the lanes of a wave, then read by them: the hardware keeps a
// wave's LDS operations in order; this keeps the compiler from moving them.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// minmod() with one magnitude compare (the same value, NaN operands included).
__device__ __forceinline__ double minmod_mag(double a, double b) {
  const bool same = ((a > 0.0) & (b > 0.0)) | ((a < 0.0) & (b < 0.0));
  const double m = (fabs(a) < fabs(b)) ? a : b;
  return same ? m : 0.0;
}

// reconstruction.cpp:67-97 extension: the tuple of mean +/- slope / 2, of the
// mean where that has a non-positive density or pressure.
template <bool UPPER>
__device__ __forceinline__ void face_tup(const double *mean, const double *half, Tup &T) {
  double v[NF];
#pragma unroll
  for (int k = 0; k < NF; ++k) v[k] = UPPER ? mean[k] + half[k] : mean[k] - half[k];
  make_tup_fast(v, T);
  if (__builtin_expect(!(T.c[FID_RHO] > 0.0) || !(T.p > 0.0), 0)) make_tup(mean, T);
}

}  // namespace

template <int DIM, int STAGE, bool P2>
__global__ __launch_bounds__(DIM == 3 ? 256 : 64, 3) void k_brick_o2(GridDev g, const double *X, const double *U,
                                                                     const double *R, double *out, Ctrl *ctrl, int mode,
                                                                     int nbx, int nby) {
  constexpr int BX = 8, BY = 8, BZ = (DIM == 3) ? 4 : 1;
  constexpr int NT = BX * BY * BZ, NW = BZ;
  // outer cells of the lines: x lower, x upper, y lower, y upper (8 per wave
  // each), z lower, z upper
  constexpr int L1 = 8 * BZ, LZ = 4 * L1, NL = LZ + (DIM == 3 ? 128 : 0);
  constexpr int SO = NT + NL;                      // field stride of the states
  constexpr int EH = L1 + (DIM == 3 ? 64 : 0);     // exchange slots of a line: x and y share theirs, z has its own
  constexpr int SE = NT + EH;                      // field stride of the exchange
  __shared__ double sx[NF * SO];
  __shared__ double ex[NTUP * SE];
  __shared__ unsigned long long red[NW];

  const int tid = threadIdx.x, lane = tid & 63, lz = tid >> 6;
  const int lx = lane & 7, ly = lane >> 3;
  const bool step = mode == MODE_STEP;
  const int tile = xcd_range((int)blockIdx.x, (int)gridDim.x);
  const int bz = (DIM == 3) ? tile / (nbx * nby) : 0;
  const int by = (tile / nbx) % nby, bx = tile % nbx;
  const int nx = (int)g.n[0], ny = (int)g.n[1], nz = (DIM == 3) ? (int)g.n[2] : 1;
  const int x0 = bx * BX, y0 = by * BY, z0 = bz * BZ;
  const int w = (nx - x0 < BX) ? nx - x0 : BX;
  const int h = (ny - y0 < BY) ? ny - y0 : BY;
  const int d = (DIM == 3) ? ((nz - z0 < BZ) ? nz - z0 : BZ) : 1;
  const bool valid = lx < w && ly < h && lz < d;
  const int64_t fs = g.fs;
  auto index = [&](int x, int y, int z) { return (uint32_t)x + (uint32_t)nx * ((uint32_t)y + (uint32_t)ny * (uint32_t)z); };
  const uint32_t idx = valid ? index(x0 + lx, y0 + ly, z0 + lz) : index(x0, y0, z0);

  // this lane's line: axis, side, whether its brick edge is a border; its
  // position among the outer cells' slots and the exchange's
  int la = -1, lup = 0, lslot = 0, eslot = 0;
  bool lborder = false;
  int ledge = 0;  // the brick cell at the line's end (thread number)
  uint32_t i1 = idx, i2 = idx;
  {
    int i, j, k;
    if (lane < 32) {
      la = lane >> 4;
      lup = (lane >> 3) & 1;
      const int p = lane & 7;
      lslot = (2 * la + lup) * L1 + 8 * lz + p;
      eslot = 8 * lz + p;
      i = la == 0 ? (lup ? w - 1 : 0) : p;
      j = la == 0 ? p : (lup ? h - 1 : 0);
      k = lz;
    } else if (DIM == 3) {
      la = 2;
      lup = lz >> 1;
      const int p = (lz & 1) * 32 + lane - 32;
      lslot = LZ + 64 * lup + p;
      eslot = L1 + p;
      i = p & 7;
      j = p >> 3;
      k = lup ? d - 1 : 0;
    } else {
      i = j = k = 0;
    }
    if (i >= w || j >= h || k >= d) la = -1;
    if (la >= 0) {
      ledge = i + BX * (j + BY * k);
      const int q[3] = {x0 + i, y0 + j, z0 + k};
      const int n = la == 0 ? nx : la == 1 ? ny : nz;
      const int c = q[la == 2 ? 2 : la];
      int c1 = c + (lup ? 1 : -1), c2 = c + (lup ? 2 : -2);
      if (la == 0 ? g.periodic[0] : la == 1 ? g.periodic[1] : g.periodic[2]) {
        c1 += (c1 < 0) ? n : (c1 >= n) ? -n : 0;
        c2 += (c2 < 0) ? n : (c2 >= n) ? -n : 0;
      } else {
        // beyond the border: the cell inside, so that differences vanish
        lborder = c1 < 0 || c1 >= n;
        c1 = lborder ? c : c1;
        c2 = (c2 < 0 || c2 >= n) ? c1 : c2;
      }
      i1 = index(la == 0 ? c1 : q[0], la == 1 ? c1 : q[1], la == 2 ? c1 : q[2]);
      i2 = index(la == 0 ? c2 : q[0], la == 1 ? c2 : q[1], la == 2 ? c2 : q[2]);
    }
  }

  const bool run = !step || ctrl->t < ctrl->tmax;  // main.cpp:377 loop guard
  double dt = 0.0;
  double Xc[NF], X1[NF], X2[NF], Uc[NF];
  if (STAGE == 2) {
    double rc[NF], r1[NF], r2[NF], x[NF], q[NF];
#pragma unroll
    for (int k = 0; k < NF; ++k) {
      Uc[k] = U[k * fs + idx];
      X1[k] = U[k * fs + i1];
      X2[k] = U[k * fs + i2];
      rc[k] = R[k * fs + idx];
      r1[k] = R[k * fs + i1];
      r2[k] = R[k * fs + i2];
    }
    dt = step_dt(ctrl);
    // main.cpp:421
#pragma unroll
    for (int k = 0; k < NF; ++k) x[k] = dt * rc[k];
    div_vol5<P2>(g, x, q);
#pragma unroll
    for (int k = 0; k < NF; ++k) Xc[k] = Uc[k] + q[k], x[k] = dt * r1[k];
    div_vol5<P2>(g, x, q);
#pragma unroll
    for (int k = 0; k < NF; ++k) X1[k] = X1[k] + q[k], x[k] = dt * r2[k];
    div_vol5<P2>(g, x, q);
#pragma unroll
    for (int k = 0; k < NF; ++k) X2[k] = X2[k] + q[k];
  } else {
#pragma unroll
    for (int k = 0; k < NF; ++k) {
      Xc[k] = X[k * fs + idx];
      X1[k] = X[k * fs + i1];
      X2[k] = X[k * fs + i2];
      Uc[k] = (STAGE == 3) ? U[k * fs + idx] : 0.0;
    }
    if (STAGE == 3) dt = step_dt(ctrl);
  }
#pragma unroll
  for (int k = 0; k < NF; ++k) {
    sx[k * SO + tid] = Xc[k];
    if (la >= 0) sx[k * SO + NT + lslot] = X1[k];
  }
  if (NT > 64) __syncthreads();
  else wave_sync();

  // the line's facing tuple: the upper face value of the cell below the brick
  // or the lower one of the cell above it
  Tup G;
  if (la >= 0) {
    if (lborder) {
      double v[NF];
      border_state(g, 2 * la + lup, la, X1, v);
      make_tup(v, G);
    } else {
      double hs[NF];
#pragma unroll
      for (int k = 0; k < NF; ++k) {
        const double in = sx[k * SO + ledge] - X1[k], on = X1[k] - X2[k];  // towards the brick, and beyond
        const double s = lup ? minmod_mag(-on, -in) : minmod_mag(in, on);
        hs[k] = lup ? -(0.5 * s) : 0.5 * s;
      }
      face_tup<true>(X1, hs, G);
    }
  }

  double lam = 0.0;
  NegCount neg;
  double rhs[NF] = {0., 0., 0., 0., 0.};  // euler.cpp:142-148
  const double halfA = P2 ? 1.0 : g.halfA;
  const int qc[3] = {x0 + lx, y0 + ly, z0 + lz};
#pragma unroll
  for (int a = 0; a < DIM; ++a) {
    const int str = a == 0 ? 1 : a == 1 ? BX : BX * BY;
    const int pos = a == 0 ? lx : a == 1 ? ly : lz, len = a == 0 ? w : a == 1 ? h : d;
    const int line = a == 0 ? 8 * lz + ly : a == 1 ? 8 * lz + lx : lane;  // this cell's line on either side
    const int hm = NT + (a == 2 ? LZ + line : (2 * a) * L1 + line), hp = hm + (a == 2 ? 64 : L1);
    const int eh = NT + (a == 2 ? L1 + line : line);
    const bool first = pos == 0, last = pos + 1 == len;
    auto sync = [&] {
      if (a == 2) __syncthreads();
      else wave_sync();
    };
    double hs[NF];
    {
      const int sm = first ? hm : tid - str, sp = last ? hp : tid + str;
#pragma unroll
      for (int k = 0; k < NF; ++k)
        hs[k] = 0.5 * minmod_mag(sx[k * SO + sp] - Xc[k], Xc[k] - sx[k * SO + sm]);
    }
    Tup TL, T;
    face_tup<true>(Xc, hs, T);
    put_tup<SE>(ex, tid, T);
    if (la == a && !lup) put_tup<SE>(ex, NT + eslot, G);
    face_tup<false>(Xc, hs, TL);
    sync();
    // the cell's lower face; the line's face above the brick
    double F[NF], F2[NF];
    get_tup<SE>(ex, first ? eh : tid - str, T);
    {
      const double l = face_flux_area(T, TL, a, P2, g.A, halfA, F);
      lam = lam_acc(lam, valid ? l : 0.0);
      // each face counted once, as the reference evaluates it
      if (__builtin_expect(valid && (tup_negative(T) | tup_negative(TL)), 0)) neg.add(T, TL);
    }
    const bool above = la == a && lup;
    if (above) {
      get_tup<SE>(ex, ledge, T);
      const double l = face_flux_area(T, G, a, P2, g.A, halfA, F2);
      lam = lam_acc(lam, l);
      if (lborder) neg.add(T, G);
    }
    sync();
#pragma unroll
    for (int k = 0; k < NF; ++k) {
      ex[k * SE + tid] = F[k];
      if (above) ex[k * SE + NT + eslot] = F2[k];
    }
    sync();
    const int up = last ? eh : tid + str;
    if (g.periodic[a] && qc[a] == (int)g.n[a] - 1) {
      // the wrap face is first in the reference-order face list
#pragma unroll
      for (int k = 0; k < NF; ++k) { rhs[k] -= ex[k * SE + up]; rhs[k] += F[k]; }
    } else {
#pragma unroll
      for (int k = 0; k < NF; ++k) { rhs[k] += F[k]; rhs[k] -= ex[k * SE + up]; }
    }
    if (a < 2) wave_sync();
  }

  if (!run) return;  // uniform over the grid: t does not change before the step closes
  if (valid) {
    if (P2) {
#pragma unroll
      for (int k = 0; k < NF; ++k) rhs[k] = g.halfA * rhs[k];
    }
    if (STAGE == 1) {
#pragma unroll
      for (int k = 0; k < NF; ++k) out[k * fs + idx] = rhs[k];
    } else {
      double x[NF], q[NF];
#pragma unroll
      for (int k = 0; k < NF; ++k) x[k] = dt * rhs[k];
      div_vol5<P2>(g, x, q);
#pragma unroll
      for (int k = 0; k < NF; ++k) out[k * fs + idx] = rk_update_q<STAGE>(Uc[k], Xc[k], q[k]);
    }
  }
  if (__any(neg.p | neg.r)) neg.flush(ctrl, tid);
  const unsigned long long m = wave_max_u64(dbits(lam));
  const int slot = step ? STAGE - 1 : 3;
  if (NW == 1) {
    if (tid == 0) stage_max_put(ctrl, slot, m);
  } else {
    if (lane == 0) red[lz] = m;
    __syncthreads();
    if (tid == 0) {
      unsigned long long b = red[0];
#pragma unroll
      for (int i = 1; i < NW; ++i) b = (red[i] > b) ? red[i] : b;
      stage_max_put(ctrl, slot, b);
    }
  }
  if (STAGE == 3 && step) close_step<false>(ctrl, tid);
}

template <int DIM, bool P2>
static hipError_t launch_brick_o2_p(const GridDev &g, int stage, int mode, const double *U, const double *R,
                                    const double *W, double *oR, double *oW, double *oU, Ctrl *ctrl, hipStream_t s) {
  const int nbx = (int)((g.n[0] + 7) / 8), nby = (int)((g.n[1] + 7) / 8), nbz = (DIM == 3) ? (int)((g.n[2] + 3) / 4) : 1;
  const dim3 grid((unsigned)nbx * nby * nbz), block(DIM == 3 ? 256 : 64);
  switch (stage) {
    case 1: hipLaunchKernelGGL((k_brick_o2<DIM, 1, P2>), grid, block, 0, s, g, U, U, R, oR, ctrl, mode, nbx, nby); break;
    case 2: hipLaunchKernelGGL((k_brick_o2<DIM, 2, P2>), grid, block, 0, s, g, U, U, R, oW, ctrl, mode, nbx, nby); break;
    default: hipLaunchKernelGGL((k_brick_o2<DIM, 3, P2>), grid, block, 0, s, g, W, U, R, oU, ctrl, mode, nbx, nby);
  }
  return hipGetLastError();
}

bool brick_o2_supported(const GridDev &g) {
  return g.order == 2 && !g.bslot && !g.flags && g.N < BRICK_MAX_CELLS &&
         padded_cells(g, 8, 8, g.dim == 3 ? 4 : 1) < LAUNCH_THREADS;
}

hipError_t launch_stage_brick_o2(const GridDev &g, int stage, int mode, const double *U, const double *R,
                                 const double *W, double *oR, double *oW, double *oU, Ctrl *ctrl, hipStream_t s) {
  const bool p2 = g.pow2A && g.pow2V;
  if (g.dim == 3)
    return p2 ? launch_brick_o2_p<3, true>(g, stage, mode, U, R, W, oR, oW, oU, ctrl, s)
              : launch_brick_o2_p<3, false>(g, stage, mode, U, R, W, oR, oW, oU, ctrl, s);
  return p2 ? launch_brick_o2_p<2, true>(g, stage, mode, U, R, W, oR, oW, oU, ctrl, s)
            : launch_brick_o2_p<2, false>(g, stage, mode, U, R, W, oR, oW, oU, ctrl, s);
}

}  // namespace mmf
