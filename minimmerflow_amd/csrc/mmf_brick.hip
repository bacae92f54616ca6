// mmf_brick.hip -- order-1 stage kernel of small and ordinary grids (gfx950).
//
// A block owns a brick of BX x BY x BZ cells, one thread per cell, and the
// brick's one-cell halo, at most one halo cell per thread.  Every thread
// loads its cell and its halo cell at once (no load waits for another: the
// per-cell gather kernel it replaces here spent most of a launch on a chain of
// dependent neighbour loads and 64-bit index divisions, and built the flux
// tuple of every neighbour again: seven tuples per 3D cell instead of two),
// builds both flux tuples -- every division and the square root of the
// reference's per-face evaluation -- into LDS, and after one barrier evaluates
// the faces of its cell from the neighbours' slots.  A border face's halo slot
// holds the virtual state's tuple, so the faces have no border branches.  The
// tuples are the unit of work, so the brick needs no march and no second
// barrier, and a launch is one pass of about one load latency, two tuples and
// 2 DIM faces.
//
// dt is known before stage 1 (Ctrl::lam_now, as in the marching kernel):
// stage 1 writes W1 = U + dt R / V, stage 3 gathers the next step's maximum
// and closes the step, so a step is three launches.
//
// Each cell's residual is summed in the reference's face order: results equal
// the gather kernel's and the oracle's bit for bit.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "mmf_brick.hpp"
#include "mmf_device.hpp"
#include "mmf_batch.hpp"
#include "mmf_internal.hpp"
#include "mmf_stage.hpp"

namespace mmf {

// One brick's stage: brick (bx, by, bz) of grid g, block blk of the nblk that
// advance the grid.  MASK: the grid has cell flags (every fluid cell solved).  P2: A and V are
// powers of two (the faces hand over unscaled sums, scaled once at the update;
// the same doubles).
template <int DIM, int BX, int BY, int BZ, int STAGE, bool MASK, bool P2>
__device__ __forceinline__ void brick_stage(const GridDev &g, const double *X, const double *U, double *out, Ctrl *ctrl,
                                            int mode, int bx, int by, int bz, unsigned int blk, unsigned int nblk) {
  constexpr int NT = BX * BY * BZ;
  constexpr int HX = BY * BZ, HY = BX * BZ, HZ = (DIM == 3) ? BX * BY : 0;
  constexpr int XM = NT, XP = XM + HX, YM = XP + HX, YP = YM + HY, ZM = YP + HY, ZP = ZM + HZ;
  constexpr int H = 2 * (HX + HY + HZ);
  constexpr int NS = NT + H;
  constexpr int NW = (NT + 63) / 64;
  static_assert(H <= NT, "one halo cell per thread");
  __shared__ double lds[NTUP * NS];
  __shared__ uint8_t lfl[MASK ? NS : 1];
  __shared__ unsigned int sneg[NW];
  __shared__ unsigned long long red[2 * NW];

  const int tid = threadIdx.x;
  const bool step = mode == MODE_STEP;
  const int nx = (int)g.n[0], ny = (int)g.n[1], nz = (DIM == 3) ? (int)g.n[2] : 1;
  const int x0 = bx * BX, y0 = by * BY, z0 = bz * BZ;
  const int w = (nx - x0 < BX) ? nx - x0 : BX;
  const int h = (ny - y0 < BY) ? ny - y0 : BY;
  const int d = (DIM == 3) ? ((nz - z0 < BZ) ? nz - z0 : BZ) : 1;
  auto index = [&](int x, int y, int z) { return (uint32_t)x + (uint32_t)nx * ((uint32_t)y + (uint32_t)ny * (uint32_t)z); };

  const int lx = tid % BX, ly = (tid / BX) % BY, lz = (DIM == 3) ? tid / (BX * BY) : 0;
  const bool valid = lx < w && ly < h && lz < d;
  const uint32_t idx = valid ? index(x0 + lx, y0 + ly, z0 + lz) : index(x0, y0, z0);

  // this thread's halo cell (hside: the side it lies on, -1 for none); across
  // a non-periodic border the inner cell, whose virtual state it builds
  int hside = -1;
  bool hborder = false;
  uint32_t hidx = idx;
  if (tid < H) {
    const int s = XM + tid;
    int i, j, k = 0;  // position in the brick, the outer coordinate one off it
    if (s < YM) {
      const int r = (s < XP) ? s - XM : s - XP;
      hside = (s < XP) ? 0 : 1;
      i = (s < XP) ? -1 : w;
      j = r % BY;
      k = r / BY;
    } else if (s < ZM || DIM == 2) {
      const int r = (s < YP) ? s - YM : s - YP;
      hside = (s < YP) ? 2 : 3;
      j = (s < YP) ? -1 : h;
      i = r % BX;
      k = r / BX;
    } else {
      const int r = (s < ZP) ? s - ZM : s - ZP;
      hside = (s < ZP) ? 4 : 5;
      k = (s < ZP) ? -1 : d;
      i = r % BX;
      j = r / BX;
    }
    const int a = hside >> 1;
    if ((a == 0 || i < w) && (a == 1 || j < h) && (a == 2 || k < d)) {
      int q[3] = {x0 + i, y0 + j, z0 + k};
      const int n[3] = {nx, ny, nz};
#pragma unroll
      for (int b = 0; b < DIM; ++b) {
        if (q[b] >= 0 && q[b] < n[b]) continue;
        if (g.periodic[b]) q[b] += (q[b] < 0) ? n[b] : -n[b];
        else {
          hborder = true;
          q[b] += (q[b] < 0) ? 1 : -1;
        }
      }
      hidx = index(q[0], q[1], q[2]);
    } else {
      hside = -1;
    }
  }

  // every load of the launch, none dependent on another
  const int64_t fs = g.fs;
  double Xc[NF], Xh[NF], Uc[NF];
#pragma unroll
  for (int k = 0; k < NF; ++k) Xc[k] = X[k * fs + idx];
#pragma unroll
  for (int k = 0; k < NF; ++k) Xh[k] = X[k * fs + hidx];
#pragma unroll
  for (int k = 0; k < NF; ++k) Uc[k] = (STAGE >= 2) ? U[k * fs + idx] : 0.0;
  uint8_t fc = CELL_FLUID | CELL_SOLVED, fh = CELL_FLUID | CELL_SOLVED;
  if (MASK) {
    fc = g.flags[idx];
    fh = g.flags[hidx];
  }
  const bool run = !step || ctrl->t < ctrl->tmax;  // main.cpp:377 loop guard
  const double dt = step ? step_dt_early(ctrl) : 0.0;

  const bool solved = valid && (!MASK || (fc & CELL_SOLVED));
  double lam = 0.0;  // stage maximum: the larger side of every face (euler.cpp:232-234)
  Tup Tc;
  make_tup_fast(Xc, Tc);
  put_tup<NS>(lds, tid, Tc);
  bool neg_here = valid && tup_negative(Tc);
  if (solved) {
    // every cell has faces along every axis
    double um = fabs(Tc.vel[0]);
#pragma unroll
    for (int a = 1; a < DIM; ++a) um = lam_acc(um, fabs(Tc.vel[a]));
    lam = um + Tc.a;
  }
  if (MASK) lfl[tid] = fc;
  if (hside >= 0) {
    const int a = hside >> 1;
    if (hborder) {  // euler.cpp:261-376
      double v[NF];
      border_state(g, hside, a, Xh, v);
#pragma unroll
      for (int k = 0; k < NF; ++k) Xh[k] = v[k];
    }
    Tup Th;
    make_tup_fast(Xh, Th);
    put_tup<NS>(lds, XM + tid, Th);
    neg_here = neg_here || tup_negative(Th);
    if (MASK) lfl[XM + tid] = fh;
    if (hborder && (!MASK || (fh & CELL_SOLVED))) {
      const double ua = (a == 0) ? Th.vel[0] : (a == 1) ? Th.vel[1] : Th.vel[2];
      lam = lam_acc(lam, fabs(ua) + Th.a);
    }
  }
  // a state with negative pressure or density somewhere in the block: its
  // faces are then counted (below) instead of every face always
  const unsigned long long nb = __ballot(neg_here);
  if ((tid & 63) == 0) sneg[tid >> 6] = nb != 0;
  __syncthreads();

  unsigned int anyneg = 0;
#pragma unroll
  for (int i = 0; i < NW; ++i) anyneg |= sneg[i];

  double lam_nx = 0.0;
  NegCount neg;
  if (solved) {
    const int slot_m[3] = {lx > 0 ? tid - 1 : XM + ly + BY * lz, ly > 0 ? tid - BX : YM + lx + BX * lz,
                           lz > 0 ? tid - BX * BY : ZM + lx + BX * ly};
    const int slot_p[3] = {lx + 1 < w ? tid + 1 : XP + ly + BY * lz, ly + 1 < h ? tid + BX : YP + lx + BX * lz,
                           lz + 1 < d ? tid + BX * BY : ZP + lx + BX * ly};
    // the neighbour's tuple across a face; a fluid-solid face's virtual state
    // is the reflected own state (main.cpp:271-275, euler.cpp:347-356)
    auto across = [&](int slot, int a, Tup &N) {
      if (MASK && ((lfl[slot] ^ fc) & CELL_FLUID)) {
        double v[NF];
        reflect_axis(Tc.c, a, v);
        make_tup(v, N);
        return true;
      }
      get_tup<NS>(lds, slot, N);
      return false;
    };
    const double halfA = P2 ? 1.0 : g.halfA;
    const int qc[3] = {x0 + lx, y0 + ly, z0 + lz};
    double rhs[NF] = {0., 0., 0., 0., 0.};  // euler.cpp:142-148
    bool wall_any = false;
#pragma unroll
    for (int a = 0; a < DIM; ++a) {
      double Fm[NF], Fp[NF];
      {
        Tup N;
        const bool wall = across(slot_m[a], a, N);
        const double l = face_flux_area(N, Tc, a, P2, g.A, halfA, Fm);
        if (MASK && wall) lam = lam_acc(lam, l);
        wall_any = wall_any || wall;
      }
      {
        Tup N;
        const bool wall = across(slot_p[a], a, N);
        const double l = face_flux_area(Tc, N, a, P2, g.A, halfA, Fp);
        if (MASK && wall) lam = lam_acc(lam, l);
        wall_any = wall_any || wall;
      }
      if (g.periodic[a] && qc[a] == (int)g.n[a] - 1) {
        // the wrap face is first in the reference-order face list
#pragma unroll
        for (int k = 0; k < NF; ++k) { rhs[k] -= Fp[k]; rhs[k] += Fm[k]; }
      } else {
#pragma unroll
        for (int k = 0; k < NF; ++k) { rhs[k] += Fm[k]; rhs[k] -= Fp[k]; }
      }
    }
    if (anyneg || wall_any) {
      // once per face, as the reference evaluates it: every upper face, and
      // the lower ones that no solved cell has as its upper face
#pragma unroll
      for (int a = 0; a < DIM; ++a) {
        Tup N;
        const bool border = !g.periodic[a] && qc[a] == 0;
        const bool wall = across(slot_m[a], a, N);
        if (border || wall || (MASK && !(lfl[slot_m[a]] & CELL_SOLVED))) neg.add(N, Tc);
        across(slot_p[a], a, N);
        neg.add(Tc, N);
      }
    }

    double nu[NF];
    if (P2) {
#pragma unroll
      for (int k = 0; k < NF; ++k) rhs[k] = g.halfA * rhs[k];
    }
    if (STAGE == 1 && !step) {
#pragma unroll
      for (int k = 0; k < NF; ++k) nu[k] = rhs[k];
    } else {
      double x[NF], q[NF];
#pragma unroll
      for (int k = 0; k < NF; ++k) x[k] = dt * rhs[k];
      div_vol5<P2>(g, x, q);
#pragma unroll
      for (int k = 0; k < NF; ++k) nu[k] = rk_update_q<STAGE>(Uc[k], Tc.c[k], q[k]);
    }
    if (run) {
#pragma unroll
      for (int k = 0; k < NF; ++k) out[k * fs + idx] = nu[k];
    }
    if (STAGE == 3) {
      // the next step's stage-1 maximum: this cell's, and the virtual states
      // its border and wall faces will have
      lam_nx = cell_max_eig<DIM>(nu);
#pragma unroll
      for (int a = 0; a < DIM; ++a) {
        bool refl = false;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const int slot = s ? slot_p[a] : slot_m[a];
          const bool border = !g.periodic[a] && (s ? qc[a] == (int)g.n[a] - 1 : qc[a] == 0);
          if (border) {
            const int bc = g.bc[2 * a + s];
            refl = refl || bc == BC_REFLECTING || bc == BC_WALL;
            if (bc == BC_DIRICHLET) lam_nx = lam_acc(lam_nx, fabs(lds[(5 + a) * NS + slot]) + lds[9 * NS + slot]);
          } else if (MASK) {
            refl = refl || !(lfl[slot] & CELL_FLUID);
          }
        }
        if (refl) {
          double v[NF];
          Tup V;
          reflect_axis(nu, a, v);
          make_tup(v, V);
          lam_nx = lam_acc(lam_nx, fabs(V.vel[a]) + V.a);
        }
      }
    }
  } else if (MASK && valid && run && STAGE != 3) {
    // unsolved (solid) cells: a residual of zero
    GridDev gp = g;
    gp.pow2V = P2;
#pragma unroll
    for (int k = 0; k < NF; ++k)
      out[k * fs + idx] = (STAGE == 1) ? (step ? Xc[k] + div_vol(gp, dt * 0.0) : 0.0) : Uc[k];
  }

  if (!run) return;  // uniform over the grid: t does not change before the step closes
  if (anyneg || MASK) neg.flush(ctrl, tid);
  if (STAGE == 1 && step) return;  // its maximum was known before the step
  const unsigned long long ml = wave_max_u64(dbits(lam));
  const unsigned long long mn = (STAGE == 3) ? wave_max_u64(dbits(lam_nx)) : 0ull;
  if ((tid & 63) == 0) {
    red[tid >> 6] = ml;
    red[NW + (tid >> 6)] = mn;
  }
  if (NW > 1) __syncthreads();
  if (tid == 0) {
    unsigned long long m = ml, n = mn;
#pragma unroll
    for (int i = 1; i < NW; ++i) {
      m = (red[i] > m) ? red[i] : m;
      n = (red[NW + i] > n) ? red[NW + i] : n;
    }
    stage_max_put(ctrl, step ? STAGE - 1 : 3, m, blk);
    if (STAGE == 3) lam_put(ctrl, n, blk);
  }
  if (STAGE == 3 && step) close_step<true>(ctrl, tid, blk, nblk);
}

template <int DIM, int BX, int BY, int BZ, int STAGE, bool MASK, bool P2>
__global__ __launch_bounds__(BX *BY *BZ) void k_brick(GridDev g, const double *X, const double *U, double *out,
                                                      Ctrl *ctrl, int mode, int nbx, int nby) {
  const int tile = xcd_range((int)blockIdx.x, (int)gridDim.x);
  const int bz = (DIM == 3) ? tile / (nbx * nby) : 0;
  brick_stage<DIM, BX, BY, BZ, STAGE, MASK, P2>(g, X, U, out, ctrl, mode, tile % nbx, (tile / nbx) % nby, bz, blockIdx.x,
                                                gridDim.x);
}

// ---- one launch per step: small 2D grids without a body ------------------------
// A block advances O x O cells (O = R - 6) by a whole step: it loads the R x R
// cells around them, one per thread, and forms W1, W2 and the new state on
// regions that shrink by a ring per stage, so that only dt crosses blocks, and
// that is known before the step.  A slot one cell outside a border that is not
// periodic holds the virtual state of its inner cell: its thread rebuilds it
// at every stage from the inner cell's state.  A block repeats its neighbours'
// rings (2.0 tuples and 1.5 cell updates per cell and stage), which costs
// less than the launches, the loads and the stores of two more stages do while
// the grid does not fill the chip.  The new state goes to another buffer: the
// neighbours still read the old one.
// 16 x 16 regions: us per step of one grid alone / of three on three streams,
// three launches a step and this one:
//   64 x 64 periodic     16.3 / 8.0    11.5 / 5.7
//   64 x 64 reflecting   17.5 / 8.3    14.6 / 6.1 (15.3 / 6.4 with division
//                        sequences in the reflected states)
//   128 x 128 inflow     16.7 / 7.8    12.0 / 6.0
//   256 x 200 inflow     18.7 / 9.0    15.9 / 8.3
//   255 x 256 reflecting 21.1 / 10.1   18.4 / 10.4
//   300 x 300 inflow     22.3 / 11.1   21.9 / 12.9
// so up to 2^16 cells, where a chip of blocks is about full (three fit a CU:
// 768).  Thin grids reach that earlier and then wait for blocks of mostly empty
// regions: 12,000 x 1 (1200 blocks) 21.8 / 9.0 and 19.1 / 12.7, 60,000 x 1 44 / 29
// and 66 / 61; so up to 768 blocks.  What is left is one launch's latency, the
// chain of three stages and the step's close.
template <int R, bool P2>
__global__ __launch_bounds__(R *R) void k_brick_step(GridDev g, const double *X, double *out, Ctrl *ctrl, int nbx) {
  constexpr int NT = R * R, O = R - 6, NW = NT / 64;
  __shared__ double lds[2][NTUP * NT];
  __shared__ unsigned int sneg[3][NW];
  __shared__ unsigned long long red[3][NW];

  const int tid = threadIdx.x, lx = tid % R, ly = tid / R;
  const int tile = xcd_range((int)blockIdx.x, (int)gridDim.x);
  const int x0 = (tile % nbx) * O, y0 = (tile / nbx) * O;
  const int n[2] = {(int)g.n[0], (int)g.n[1]};
  auto owned = [&](int x, int y) {  // unwrapped
    return x >= x0 && x < x0 + O && x < n[0] && y >= y0 && y < y0 + O && y < n[1];
  };
  int q[2] = {x0 - 3 + lx, y0 - 3 + ly};
  const bool own = owned(q[0], q[1]);
  // the slot's cell, or the inner cell of the virtual state it holds
  int side = -1, inner = tid;
  bool alive = true, own_inner = false;
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    if (g.periodic[a]) continue;
    if (q[a] < -1 || q[a] > n[a]) alive = false;
    else if (q[a] < 0 || q[a] == n[a]) {
      if (side >= 0) alive = false;  // outside two borders
      const int in = (q[a] < 0) ? 1 : -1;
      side = 2 * a + (in < 0);
      q[a] += in;
      inner = tid + in * (a ? R : 1);
    }
  }
  if (side >= 0 && alive) own_inner = owned(q[0], q[1]);
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    if (!g.periodic[a]) continue;
    while (q[a] < 0) q[a] += n[a];
    while (q[a] >= n[a]) q[a] -= n[a];
  }
  const uint32_t idx = alive ? (uint32_t)q[0] + (uint32_t)n[0] * (uint32_t)q[1] : (uint32_t)x0 + (uint32_t)n[0] * (uint32_t)y0;
  const int64_t fs = g.fs;
  double U[NF], S[NF];
#pragma unroll
  for (int k = 0; k < NF; ++k) S[k] = U[k] = X[k * fs + idx];
  const bool run = ctrl->t < ctrl->tmax;  // main.cpp:377 loop guard
  if (!run) {                             // uniform; the state stays, in the buffer that is then the current one
    if (own) {
#pragma unroll
      for (int k = 0; k < NF; ++k) out[k * fs + idx] = U[k];
    }
    return;
  }
  const double dt = step_dt_early(ctrl);
  const bool borders = (!g.periodic[0] && (x0 <= 3 || x0 + O + 3 > n[0])) || (!g.periodic[1] && (y0 <= 3 || y0 + O + 3 > n[1]));

  NegCount neg;
  unsigned int anyneg = 0;
  double lam[3] = {0.0, 0.0, 0.0};  // maxima of stages 2 and 3, and of the new state

  auto stage = [&](auto STAGE_) {
    constexpr int STAGE = decltype(STAGE_)::value;
    double *buf = lds[(STAGE - 1) & 1], *nxt = lds[STAGE & 1];
    Tup T;
    bool neg_here = false;
    if (alive && lx >= STAGE - 1 && lx <= R - STAGE && ly >= STAGE - 1 && ly <= R - STAGE) {
      if (side >= 0) {
        double v[NF];
        if (STAGE > 1) {
#pragma unroll
          for (int k = 0; k < NF; ++k) S[k] = buf[k * NT + inner];
        }
        const int bc = g.bc[side];  // euler.cpp:261-376
        if (bc == BC_REFLECTING || bc == BC_WALL) reflect_axis_quot(S, side >> 1, v);
        else border_state(g, side, side >> 1, S, v);
#pragma unroll
        for (int k = 0; k < NF; ++k) S[k] = v[k];
      }
      // one tuple for both kinds of slots: a wave holds some of each
      make_tup_fast(S, T);
      double ls = 0.0;
      if (own) ls = lam_acc(fabs(T.vel[0]), fabs(T.vel[1])) + T.a;
      if (own_inner) ls = fabs((side & 2) ? T.vel[1] : T.vel[0]) + T.a;
      if (STAGE > 1) lam[STAGE - 2] = ls;
      neg_here = tup_negative(T);
      put_tup<NT>(buf, tid, T);
    }
    const unsigned long long nb = __ballot(neg_here);
    if ((tid & 63) == 0) sneg[STAGE - 1][tid >> 6] = nb != 0;
    __syncthreads();
    unsigned int an = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) an |= sneg[STAGE - 1][i];
    anyneg |= an;

    if (alive && side < 0 && lx >= STAGE && lx < R - STAGE && ly >= STAGE && ly < R - STAGE) {
      const int off[2] = {1, R};
      const double halfA = P2 ? 1.0 : g.halfA;
      double rhs[NF] = {0., 0., 0., 0., 0.};  // euler.cpp:142-148
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        double Fm[NF], Fp[NF];
        Tup N;
        get_tup<NT>(buf, tid - off[a], N);
        face_flux_area(N, T, a, P2, g.A, halfA, Fm);
        get_tup<NT>(buf, tid + off[a], N);
        face_flux_area(T, N, a, P2, g.A, halfA, Fp);
        if (g.periodic[a] && q[a] == n[a] - 1) {
          // the wrap face is first in the reference-order face list
#pragma unroll
          for (int k = 0; k < NF; ++k) { rhs[k] -= Fp[k]; rhs[k] += Fm[k]; }
        } else {
#pragma unroll
          for (int k = 0; k < NF; ++k) { rhs[k] += Fm[k]; rhs[k] -= Fp[k]; }
        }
      }
      if (an && own) {
        // once per face: every upper face, and the lower ones on a border
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          Tup N;
          if (!g.periodic[a] && q[a] == 0) {
            get_tup<NT>(buf, tid - off[a], N);
            neg.add(N, T);
          }
          get_tup<NT>(buf, tid + off[a], N);
          neg.add(T, N);
        }
      }
      double x[NF], dq[NF];
#pragma unroll
      for (int k = 0; k < NF; ++k) x[k] = dt * (P2 ? g.halfA * rhs[k] : rhs[k]);
      div_vol5<P2>(g, x, dq);
#pragma unroll
      for (int k = 0; k < NF; ++k) S[k] = rk_update_q<STAGE>(U[k], T.c[k], dq[k]);
      if (STAGE < 3 && borders) {  // for the virtual states of the next stage
#pragma unroll
        for (int k = 0; k < NF; ++k) nxt[k * NT + tid] = S[k];
      }
      if (STAGE == 3 && own) {
#pragma unroll
        for (int k = 0; k < NF; ++k) out[k * fs + idx] = S[k];
        // the next step's stage-1 maximum: this cell's, and the virtual states
        // its border faces will have
        double l = cell_max_eig<2>(S);
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          bool refl = false;
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            if (g.periodic[a] || q[a] != (s ? n[a] - 1 : 0)) continue;
            const int bc = g.bc[2 * a + s], slot = s ? tid + off[a] : tid - off[a];
            refl = refl || bc == BC_REFLECTING || bc == BC_WALL;
            if (bc == BC_DIRICHLET) l = lam_acc(l, fabs(buf[(5 + a) * NT + slot]) + buf[9 * NT + slot]);
          }
          if (refl) {
            double v[NF];
            Tup V;
            reflect_axis_quot(S, a, v);
            make_tup_fast(v, V);
            l = lam_acc(l, fabs(V.vel[a]) + V.a);
          }
        }
        lam[2] = l;
      }
    }
    if (STAGE < 3 && borders) __syncthreads();
  };
  stage(std::integral_constant<int, 1>{});
  stage(std::integral_constant<int, 2>{});
  stage(std::integral_constant<int, 3>{});

  if (anyneg) neg.flush(ctrl, tid);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const unsigned long long m = wave_max_u64(dbits(lam[i]));
    if ((tid & 63) == 0) red[i][tid >> 6] = m;
  }
  __syncthreads();
  if (tid < 3) {
    unsigned long long m = red[tid][0];
#pragma unroll
    for (int i = 1; i < NW; ++i) m = (red[tid][i] > m) ? red[tid][i] : m;
    if (tid < 2) stage_max_put(ctrl, tid + 1, m, blockIdx.x);
    else lam_put(ctrl, m, blockIdx.x);
  }
  close_step<true>(ctrl, tid, blockIdx.x, gridDim.x);
}

constexpr int STEP_R = 16;

hipError_t launch_step_brick(const GridDev &g, const double *in, double *out, Ctrl *ctrl, hipStream_t s) {
  constexpr int O = STEP_R - 6;
  const int nbx = (int)((g.n[0] + O - 1) / O), nby = (int)((g.n[1] + O - 1) / O);
  const dim3 grid((unsigned)nbx * nby), block(STEP_R * STEP_R);
  if (g.pow2A && g.pow2V) hipLaunchKernelGGL((k_brick_step<STEP_R, true>), grid, block, 0, s, g, in, out, ctrl, nbx);
  else hipLaunchKernelGGL((k_brick_step<STEP_R, false>), grid, block, 0, s, g, in, out, ctrl, nbx);
  return hipGetLastError();
}

bool step_brick_supported(const GridDev &g) {
  return brick_supported(g) && g.dim == 2 && g.flags == nullptr && g.N < STEP_BRICK_MAX_CELLS &&
         padded_cells(g, STEP_R - 6, STEP_R - 6, 1) <= STEP_BRICK_MAX_BLOCKS * (STEP_R - 6) * (STEP_R - 6);
}

// ---- batches: one block per brick of every case --------------------------------
// bricks[2 i], [2 i + 1]: case and brick number of block i, in case order, the
// blocks of an XCD a contiguous run of them.
constexpr int BATCH_BX = 16, BATCH_BY = 16;

template <int STAGE>
__global__ __launch_bounds__(BATCH_BX *BATCH_BY) void k_brick_batch(const BatchCase *cases, const int *bricks, double *U,
                                                                    double *R, double *W) {
  const int i = xcd_range((int)blockIdx.x, (int)gridDim.x);
  const BatchCase &bc = cases[__builtin_amdgcn_readfirstlane(bricks[2 * i])];
  const int b = __builtin_amdgcn_readfirstlane(bricks[2 * i + 1]);
  const GridDev &g = bc.g;
  const int nbx = ((int)g.n[0] + BATCH_BX - 1) / BATCH_BX, nby = ((int)g.n[1] + BATCH_BY - 1) / BATCH_BY;
  double *Ub = U + bc.offset, *Rb = R + bc.offset, *Wb = W + bc.offset;
  const double *X = (STAGE == 1) ? Ub : (STAGE == 2) ? Rb : Wb;
  double *out = (STAGE == 1) ? Rb : (STAGE == 2) ? Wb : Ub;
  brick_stage<2, BATCH_BX, BATCH_BY, 1, STAGE, false, false>(g, X, Ub, out, bc.ctrl, MODE_STEP, b % nbx, b / nbx, 0,
                                                             (unsigned)b, (unsigned)(nbx * nby));
}

__global__ __launch_bounds__(256) void k_batch_lam_zero(const BatchCase *cases, int ncases) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < ncases) cases[i].ctrl->lam_now = 0ull;
}

// Every case's Ctrl::lam_now from its state.
__global__ __launch_bounds__(BATCH_BX *BATCH_BY) void k_batch_lam(const BatchCase *cases, const int *bricks,
                                                                  const double *U) {
  const int i = xcd_range((int)blockIdx.x, (int)gridDim.x);
  const BatchCase &bc = cases[__builtin_amdgcn_readfirstlane(bricks[2 * i])];
  const int b = __builtin_amdgcn_readfirstlane(bricks[2 * i + 1]);
  const int nbx = ((int)bc.g.n[0] + BATCH_BX - 1) / BATCH_BX;
  const int64_t x = (int64_t)(b % nbx) * BATCH_BX + threadIdx.x % BATCH_BX;
  const int64_t y = (int64_t)(b / nbx) * BATCH_BY + threadIdx.x / BATCH_BX;
  double l = 0.0;
  if (x < bc.g.n[0] && y < bc.g.n[1]) {
    uint32_t sides = 0;
    l = grid_cell_lam<true>(bc.g, U + bc.offset, (uint32_t)(x + bc.g.n[0] * y), sides);
    if (sides) l = lam_acc(l, dirichlet_lam(bc.g, sides));
  }
  const unsigned long long m = wave_max_u64(dbits(l));
  if ((threadIdx.x & 63) == 0 && m) atomicMax(&bc.ctrl->lam_now, m);
}

int64_t batch_bricks(const GridDev &g) {
  return ((g.n[0] + BATCH_BX - 1) / BATCH_BX) * ((g.n[1] + BATCH_BY - 1) / BATCH_BY);
}

hipError_t launch_batch_bricks(int stage, const BatchCase *cases, const int *bricks, int nbricks, double *U, double *R,
                               double *W, hipStream_t s) {
  const dim3 grid((unsigned)nbricks), block(BATCH_BX * BATCH_BY);
  switch (stage) {
    case 1: hipLaunchKernelGGL(k_brick_batch<1>, grid, block, 0, s, cases, bricks, U, R, W); break;
    case 2: hipLaunchKernelGGL(k_brick_batch<2>, grid, block, 0, s, cases, bricks, U, R, W); break;
    default: hipLaunchKernelGGL(k_brick_batch<3>, grid, block, 0, s, cases, bricks, U, R, W);
  }
  return hipGetLastError();
}

hipError_t launch_batch_lam(const BatchCase *cases, int ncases, const int *bricks, int nbricks, const double *U,
                            hipStream_t s) {
  hipLaunchKernelGGL(k_batch_lam_zero, dim3((unsigned)((ncases + 255) / 256)), dim3(256), 0, s, cases, ncases);
  hipLaunchKernelGGL(k_batch_lam, dim3((unsigned)nbricks), dim3(BATCH_BX * BATCH_BY), 0, s, cases, bricks, U);
  return hipGetLastError();
}

template <int DIM, int BX, int BY, int BZ, bool MASK, bool P2>
static hipError_t launch_brick_p(const GridDev &g, int stage, int mode, const double *U, const double *R,
                                 const double *W, double *oR, double *oW, double *oU, Ctrl *ctrl, hipStream_t s) {
  const int nbx = (int)((g.n[0] + BX - 1) / BX), nby = (int)((g.n[1] + BY - 1) / BY);
  const int nbz = (int)((g.n[2] + BZ - 1) / BZ);
  const dim3 grid((unsigned)nbx * nby * nbz), block(BX * BY * BZ);
  // stage 2 reads the W1 that stage 1 wrote into R's buffer
  switch (stage) {
    case 1:
      hipLaunchKernelGGL((k_brick<DIM, BX, BY, BZ, 1, MASK, P2>), grid, block, 0, s, g, U, U, oR, ctrl, mode, nbx, nby);
      break;
    case 2:
      hipLaunchKernelGGL((k_brick<DIM, BX, BY, BZ, 2, MASK, P2>), grid, block, 0, s, g, R, U, oW, ctrl, mode, nbx, nby);
      break;
    default:
      hipLaunchKernelGGL((k_brick<DIM, BX, BY, BZ, 3, MASK, P2>), grid, block, 0, s, g, W, U, oU, ctrl, mode, nbx, nby);
  }
  return hipGetLastError();
}

bool brick_supported(const GridDev &g) {
  // a thread per cell of the bricks, up to 64 times the cells of a thin grid
  const int64_t threads = (g.dim == 3) ? padded_cells(g, 8, 8, 4) : padded_cells(g, 16, 16, 1);
  return g.order == 1 && !g.bslot && (g.flags == nullptr || g.ghost_free) && g.N < BRICK_MAX_CELLS &&
         threads < LAUNCH_THREADS;
}

template <int DIM, int BX, int BY, int BZ>
static hipError_t launch_brick_s(const GridDev &g, int stage, int mode, const double *U, const double *R,
                                 const double *W, double *oR, double *oW, double *oU, Ctrl *ctrl, hipStream_t s) {
  const bool p2 = g.pow2A && g.pow2V;
  if (g.flags)
    return p2 ? launch_brick_p<DIM, BX, BY, BZ, true, true>(g, stage, mode, U, R, W, oR, oW, oU, ctrl, s)
              : launch_brick_p<DIM, BX, BY, BZ, true, false>(g, stage, mode, U, R, W, oR, oW, oU, ctrl, s);
  return p2 ? launch_brick_p<DIM, BX, BY, BZ, false, true>(g, stage, mode, U, R, W, oR, oW, oU, ctrl, s)
            : launch_brick_p<DIM, BX, BY, BZ, false, false>(g, stage, mode, U, R, W, oR, oW, oU, ctrl, s);
}

// 3D: 8 x 8 x 4 cells, 256 of them with exactly 256 halo cells: two tuples per
// thread, 45 KB of LDS (three blocks per CU).  16 x 8 x 4, 8 x 8 x 8 and 16 x
// 16 x 4 build fewer halo tuples (1.9, 1.75, 1.6 per cell) but put fewer
// blocks on the chip: 32^3 27 / 28 / 36 against 23 us per step, 100 x 90 x 84
// 159 / 112 / 140 against 108.
// 2D: 16 x 16 cells (1.25 tuples per cell) once that gives every CU a block,
// 8 x 8 below: 500 x 400 30.8 against 33.8 us per step, 64^2 20.2 against 19.1.
hipError_t launch_stage_brick(const GridDev &g, int stage, int mode, const double *U, const double *R, const double *W,
                              double *oR, double *oW, double *oU, Ctrl *ctrl, hipStream_t s) {
  if (g.dim == 3) return launch_brick_s<3, 8, 8, 4>(g, stage, mode, U, R, W, oR, oW, oU, ctrl, s);
  if (brick_width_2d(g) == 16) return launch_brick_s<2, 16, 16, 1>(g, stage, mode, U, R, W, oR, oW, oU, ctrl, s);
  return launch_brick_s<2, 8, 8, 1>(g, stage, mode, U, R, W, oR, oW, oU, ctrl, s);
}

}  // namespace mmf
