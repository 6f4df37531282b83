// qeq_small.h — the FP64 QEq solve (CG_v2, fix_qeq_reax_sunway.cpp:983-1167)
// for small systems and batches of them: one launch per iteration.
//
// The general solve (qeq_cg.h) takes three dependent launches an iteration:
// product, vector updates, scalars.  With few panels none of them fills the
// chip and each costs its launch and the latency of its own loads: 17 us of
// kernels and 6 of gaps an iteration on a 648-water box, where this takes 9
// (64 clusters, 47,000 atoms: 41 and 31).  Here a workgroup
// forms its panel's rows of the product, updates those rows and writes the
// panel's partial dots, and the next launch's workgroups each sum the dots of
// their own system and advance the scalars.  That needs the panels' rows in
// atom order: the dots are then summed in exactly the general solve's order
// (64 rows by a wave butterfly, four of those to a tile of 256 rows, the
// tiles by a butterfly), and so are the row sums, so every iterate has the
// same bits.  (The order matters: this recurrence turns a last-bit change of
// a dot into 1e-8 of the charges.)
#pragma once

#include <type_traits>

#include "qeq_cg.h"

namespace swr_cg {

// The rule: FP64, every system at most SMALL_ROWS rows (its vector fits in
// LDS and its dots are at most 48 panels), and at most SMALL_PANELS panels in
// all, the workgroups a chip still runs nearly side by side.  Beyond, the
// values stream from HBM and the general solve's panel lists read 10 bytes an
// entry where this reads 12 (128 clusters, 1,700 panels: the two are equal;
// 512 clusters, 6,100 panels: a first form of this one took 1.0 ms more).
constexpr int SMALL_ROWS = 3072;
constexpr int SMALL_PANELS = 1024;
static_assert(SMALL_ROWS <= SWR_WAVE * UT, "a small system's tiles fit one wave");
static_assert(UT % SWR_PANEL_ROWS == 0, "tiles are whole panels");

// The eight vectors of one row of the pipelined CG, side by side (128 bytes a
// row): eight lanes load and store a row.  Only what other rows read (d) and
// the solution (x) are arrays of their own.
enum { CGL_X = 0, CGL_P, CGL_SS, CGL_V, CGL_Z, CGL_R, CGL_U, CGL_W, CGL_COUNT };

struct SmallVecs {
  double2 *x;           // [n] warm start in, solution out
  const double2 *b;     // [n] right-hand sides
  const double *Hd;     // [n] preconditioner
  double2 *state;       // [n][CGL_COUNT]
  double2 *d[2];        // [n] M^-1 w of alternate iterations
};

// Partial dots of the panels: [CG_PART_ROWS][pstride] rows.  A step reads the rows
// the step before wrote and writes others (its own panels may finish before
// another panel has read).
constexpr int SMALL_PART_ODD = 6;   // rows 0-5: PH_S3, then every second step; rows 6-9: the others
static_assert(SMALL_PART_ODD + 4 <= CG_PART_ROWS, "partials rows");

// What a panel's workgroup needs of its place: its rows [r0, r1), its system
// and the system's rows [s0, s1) and panels [p0, p1).
struct SmallPanel {
  int r0, r1, s0, s1, sys, p0, p1, pad;
};

struct SmallArgs {
  const DevParams *P;
  const int *type, *firstnbr, *numnbrs, *jlist;
  const double *val;
  const SmallPanel *panel;
  SmallVecs V;
  const CgScalars *cin;   // scalars before this step
  CgScalars *cout;        // scalars this step computed (another buffer)
  const double *part_in;
  double *part_out;
  int pstride;
  int nsys, imax;
  double tol;
  int *iters_out, *done_count;
  DevStatus *status;
  int par_in;             // which d the step multiplies
};

// Sums of the ND dots of a system over its panels [b0, b1), in the order of
// k_cg_upd and k_cg_scalars (four panels to a tile, then the tiles), by one
// wave, on all its lanes.
template <int ND>
__device__ __forceinline__ void small_dots(const double *__restrict__ part, int pstride, int b0, int b1,
                                           double *out) {
  constexpr int TP = UT / SWR_PANEL_ROWS;   // panels per tile
  const int t0 = b0 + TP * lane_id();
  double v[ND][TP];
#pragma unroll
  for (int k = 0; k < ND; k++)
#pragma unroll
    for (int w = 0; w < TP; w++) v[k][w] = t0 + w < b1 ? part[(size_t)k * pstride + t0 + w] : 0.0;
#pragma unroll
  for (int k = 0; k < ND; k++) {
    double acc = 0.0;
#pragma unroll
    for (int w = 0; w < TP; w++) acc += v[k][w];
    out[k] = wave_sum(acc);
  }
}

// Field by field (a whole-struct store keeps the scalars in scratch memory).
__device__ __forceinline__ void small_store(CgScalars *o, const CgScalars &c) {
  o->alpha_x = c.alpha_x; o->alpha_a = c.alpha_a; o->beta = c.beta;
  o->sig_old = c.sig_old; o->heta = c.heta;
  o->dg0 = c.dg0; o->dg1 = c.dg1; o->b_norm = c.b_norm;
  o->bdot = c.bdot; o->udot_r = c.udot_r; o->udot_w = c.udot_w;
  o->tol = c.tol;
  o->active_b = c.active_b; o->active_a = c.active_a; o->iter = c.iter; o->done = c.done;
}

// One step of the solve as one launch, a workgroup per 64-row panel: the
// panel's rows of q = eta d + H d (sparse_matvec_C_para,
// fix_qeq_reax_sw64.c:424-466), then those rows' vector updates and the
// panel's partial dots.
//
//   PH_S1..S3  the setup steps of CG_v2 (:1020-1087): r = b - H x, w = H u,
//              z = H m and the six dots
//   PH_A1      the first A step (no product)
//   PH_K       B and C of iteration i, A of iteration i+1 (:1113-1150)
//
// The vector of the whole system sits in LDS (16 bytes a row, 48 KB at most):
// its entries load contiguously and H's columns index it directly, with no
// list of the panel's columns to build first.  From PH_A1 on the first wave
// also sums the dots of the step before over the system's panels and advances
// the scalars (the same in each of its workgroups); the system's first panel
// writes them to the other scalar buffer, counts a finished system and keeps
// its iteration counts.
//
// What bounds a step is the chain of dependent loads, so everything whose
// address is known is requested before anything is waited for: the panel's
// place; then the vector, row extents, state rows and dots; then the first H
// values.  One barrier covers the LDS vector and the scalars.  A step in
// which neither solve goes on to another A step only adds alpha p to x: no
// product.
//
// Returns whether the system goes on (PH_A1, PH_K).
template <int ROWS, int NDOT>
struct SmallLds {
  double2 xl[ROWS];
  double2 ql[SWR_PANEL_ROWS];
  double prod[NDOT][SWR_PANEL_ROWS];   // each row's products
  double sc[6];                        // alpha_x, beta, alpha_a of s and t
  int sflag;                           // active_b, active_a of s and t
};
constexpr bool small_multiplies(int PH) { return PH != PH_A1; }
constexpr int small_dots_out(int PH) { return PH == PH_S3 ? 6 : PH == PH_A1 || PH == PH_K ? 4 : 0; }

template <int PH, int SH, class Lds>
__device__ __forceinline__ bool small_step_body(const SmallArgs &A, const int p, Lds &S) {
  constexpr int NT = SpmvShape<SH>::NT, G = SpmvShape<SH>::G;
  constexpr int U = 2;                                  // (a row's sum does not depend on it)
  constexpr int NW = NT / SWR_WAVE;
  constexpr int EP = SWR_PANEL_ROWS * CGL_COUNT / NT;   // state entries per thread
  constexpr int FU = 4;                                 // vector entries per thread requested at once
  constexpr bool MUL = PH != PH_A1;
  constexpr bool DOTS = PH == PH_S3 || PH == PH_A1 || PH == PH_K;
  constexpr int NDIN = PH == PH_A1 ? 6 : 4;             // dots of the step before
  constexpr int NDOUT = PH == PH_S3 ? 6 : 4;
  auto &xl = S.xl;
  auto &ql = S.ql;
  auto &prod = S.prod;
  auto &sc = S.sc;
  int &sflag = S.sflag;
  const SmallPanel pn = A.panel[p];
  const int r0 = pn.r0, r1 = pn.r1;
  const double2 zero = make_double2(0.0, 0.0);
  if (PH == PH_K) {   // a system that finished before: its scalars move on to the other buffer
    const CgScalars *c = A.cin + 2 * pn.sys;
    if ((c[0].active_a | c[0].active_b | c[1].active_a | c[1].active_b) == 0) {
      if (p == pn.p0 && threadIdx.x < 2) A.cout[2 * pn.sys + threadIdx.x] = c[threadIdx.x];
      return false;
    }
  }

  // ---- requests: the system's vector, row extents, this lane's state entry
  const double2 *dcur = A.par_in ? A.V.d[1] : A.V.d[0];
  const double2 *src = PH == PH_S1 ? A.V.x : PH == PH_S2 ? A.V.d[0] : PH == PH_S3 ? A.V.d[1] : dcur;
  const int ns = pn.s1 - pn.s0, grp = threadIdx.x / G;
  double2 xk[FU];
  int beg = 0, cnt = 0;
  if (MUL) {
    if (r0 + grp < r1) {
      beg = A.firstnbr[r0 + grp];
      cnt = A.numnbrs[r0 + grp];
    }
#pragma unroll
    for (int u = 0; u < FU; u++) {
      const int k = threadIdx.x + u * NT;
      xk[u] = k < ns ? src[pn.s0 + k] : zero;
    }
  }
  const int l = threadIdx.x % CGL_COUNT;
  double2 own[EP], dv[EP];
  double co[EP];
  int ty[EP];
#pragma unroll
  for (int e = 0; e < EP; e++) {
    const int row = r0 + (int)(threadIdx.x + e * NT) / CGL_COUNT;
    own[e] = dv[e] = zero;
    co[e] = 0.0;
    ty[e] = 0;
    if (row < r1) {
      if (PH != PH_S1 && PH != PH_S2) own[e] = A.V.state[(size_t)row * CGL_COUNT + l];
      // the vector the product multiplies (lane Z adds eta of it; B uses it in lane V)
      if (MUL && (l == CGL_Z || (PH == PH_K && l == CGL_V))) dv[e] = src[row];
      if (MUL && l == CGL_Z) ty[e] = A.type[row];
      if ((PH == PH_S1 || PH == PH_S3) && l == CGL_R) dv[e] = A.V.b[row];
      if (PH == PH_S1 && l == CGL_X) own[e] = A.V.x[row];
      if (l == CGL_W || (PH == PH_S1 && l == CGL_U) || (PH == PH_S3 && l == CGL_V)) co[e] = A.V.Hd[row];
    }
  }

  // ---- scalars of this step (first wave)
  if ((PH == PH_A1 || PH == PH_K) && threadIdx.x < SWR_WAVE) {
    CgScalars c0 = {}, c1 = {};
    unsigned bad = 0;
    bool fin0 = false, fin1 = false;
    double t[NDIN];
    small_dots<NDIN>(A.part_in, A.pstride, pn.p0, pn.p1, t);
    if constexpr (PH == PH_A1) {
      bad |= cg_setup_scalars(c0, t[0], t[1], t[2], A.tol, A.imax);
      bad |= cg_setup_scalars(c1, t[3], t[4], t[5], A.tol, A.imax);
      fin0 = c0.done;
      fin1 = c1.done;
    } else {
      c0 = A.cin[2 * pn.sys];
      c1 = A.cin[2 * pn.sys + 1];
      auto advance = [&](CgScalars &c, double l0, double l1, bool &fin) {
        if (c.active_a) {
          cg_after_A(c, l0, l1, A.imax);
          if (!isfinite(c.alpha_a) || !isfinite(c.beta)) bad = 1;
          if (!c.active_a) {   // this step's B ends the solve
            c.done = 1;
            fin = true;
          }
        } else {
          c.active_b = 0;
        }
      };
      advance(c0, t[0], t[1], fin0);
      advance(c1, t[2], t[3], fin1);
    }
    if (threadIdx.x == 0) {
      sc[0] = c0.alpha_x; sc[1] = c0.beta; sc[2] = c0.alpha_a;
      sc[3] = c1.alpha_x; sc[4] = c1.beta; sc[5] = c1.alpha_a;
      sflag = (PH == PH_K ? (c0.active_b ? 1 : 0) | (c1.active_b ? 2 : 0) : 0) | (c0.active_a ? 4 : 0) |
              (c1.active_a ? 8 : 0);
      if (p == pn.p0) {
        small_store(A.cout + 2 * pn.sys, c0);
        small_store(A.cout + 2 * pn.sys + 1, c1);
        if (fin0) A.iters_out[2 * pn.sys] = c0.iter;
        if (fin1) A.iters_out[2 * pn.sys + 1] = c1.iter;
        if ((fin0 || fin1) && c0.done && c1.done) atomicAdd(A.done_count, 1);
        if (bad) atomicOr(&A.status->flags, SWR_F_NAN);
      }
    }
  }

  // ---- the first row pass's values are requested, then the vector goes to LDS
  RowBatch<double, double, U, int4> first;
  bool any = false;
  if (MUL) {
    row_batch0<double, double, G, U>(cnt, reinterpret_cast<const int4 *>(A.jlist + beg), A.val + beg, first);
#pragma unroll
    for (int u = 0; u < FU; u++) {
      const int k = threadIdx.x + u * NT;
      if (k < ns) xl[k] = xk[u];
      any |= xk[u].x != 0.0 || xk[u].y != 0.0;
    }
    for (int k = threadIdx.x + FU * NT; k < ns; k += NT) {
      const double2 v = src[pn.s0 + k];
      xl[k] = v;
      any |= v.x != 0.0 || v.y != 0.0;
    }
  }
#pragma unroll
  for (int e = 0; e < EP; e++)
    if (MUL && l == CGL_Z) co[e] = A.P->eta[ty[e]];
  bool b0 = false, b1 = false, a0 = true, a1 = true;
  bool multiply = MUL;
  if (PH == PH_S1) {
    // a solve from zero history multiplies the zero vector first: its rows are zero
    multiply = __syncthreads_or(any);
  } else {
    lds_barrier();
  }
  if (PH == PH_A1 || PH == PH_K) {
    const int f = sflag;
    b0 = f & 1;
    b1 = f & 2;
    a0 = f & 4;
    a1 = f & 8;
    if (f == 0) return false;   // both solves finished
    if (PH == PH_K) multiply = a0 || a1;
  }
  const double ax0 = sc[0], be0 = sc[1], aa0 = sc[2], ax1 = sc[3], be1 = sc[4], aa1 = sc[5];

  // ---- product
  if (MUL) {
    const double2 *xs = xl - pn.s0;
    auto xv = [&](int j) { return xs[j]; };
    for (int rb = r0; rb < r1; rb += NT / G) {
      const int rr = rb + grp;
      const bool live = rr < r1;
      double2 q = zero;
      if (multiply) {
        if (rb == r0) {
          q = row_sum4<double, double, G, U, true>(cnt, reinterpret_cast<const int4 *>(A.jlist + beg), A.val + beg, xv,
                                                   &first);
        } else {
          beg = live ? A.firstnbr[rr] : 0;
          cnt = live ? A.numnbrs[rr] : 0;
          q = row_sum4<double, double, G, U>(cnt, reinterpret_cast<const int4 *>(A.jlist + beg), A.val + beg, xv);
        }
      }
      if (live && lane_id() % G == 0) ql[rr - r0] = q;
    }
    lds_barrier();
  }

  // ---- updates: lane l of a row's eight owns entry l of its state
  const int base = lane_id() - l;
  auto from = [&](const double2 &v, int lane) {
    return make_double2(__shfl(v.x, base + lane, SWR_WAVE), __shfl(v.y, base + lane, SWR_WAVE));
  };
#pragma unroll
  for (int e = 0; e < EP; e++) {
    const int row = r0 + (int)(threadIdx.x + e * NT) / CGL_COUNT;
    const bool live = row < r1;
    double2 v = own[e];
    // the row's q on every lane: eta d + sum, formed in lane Z
    double2 q = zero;
    if (MUL && live && l == CGL_Z && (PH == PH_S1 || multiply)) {
      q = ql[row - r0];
      q.x = co[e] * dv[e].x + q.x;
      q.y = co[e] * dv[e].y + q.y;
    }
    if (PH == PH_S1) {
      const double2 qz = from(q, CGL_Z);
      const double2 r = from(make_double2(dv[e].x - qz.x, dv[e].y - qz.y), CGL_R);
      if (l == CGL_R) v = r;
      if (l == CGL_U) v = make_double2(r.x * co[e], r.y * co[e]);
      if (live) {
        if (l == CGL_R || l == CGL_U || l == CGL_X) A.V.state[(size_t)row * CGL_COUNT + l] = v;
        if (l == CGL_U) A.V.d[0][row] = v;
      }
    } else if (PH == PH_S2) {
      const double2 w = from(q, CGL_Z);
      if (live && l == CGL_W) {
        A.V.state[(size_t)row * CGL_COUNT + l] = w;
        A.V.d[1][row] = make_double2(w.x * co[e], w.y * co[e]);
      }
    } else if (PH == PH_S3) {
      const double2 u = from(v, CGL_U), w = from(v, CGL_W);
      if (l == CGL_Z) v = q;
      if (l == CGL_P) v = u;
      if (l == CGL_SS) v = w;
      if (l == CGL_V) v = make_double2(w.x * co[e], w.y * co[e]);
      if (live) {
        if (l == CGL_Z || l == CGL_P || l == CGL_SS || l == CGL_V) A.V.state[(size_t)row * CGL_COUNT + l] = v;
      }
      if (l == CGL_R) {   // (zeros past the panel's end)
        prod[0][row - r0] = dv[e].x * dv[e].x;
        prod[1][row - r0] = u.x * v.x;
        prod[2][row - r0] = u.x * w.x;
        prod[3][row - r0] = dv[e].y * dv[e].y;
        prod[NDOUT - 2][row - r0] = u.y * v.y;
        prod[NDOUT - 1][row - r0] = u.y * w.y;
      }
    } else {
      // B: x += alpha p; p = u + p beta; ss = w + ss beta; v = d + v beta   (:1135-1141)
      // C: z = q + z beta                                                   (:1147-1150)
      if (PH == PH_K) {
        const int give = l == CGL_X ? CGL_P : l == CGL_P ? CGL_U : l == CGL_SS ? CGL_W : l;
        double2 o = from(v, give);
        if (l == CGL_V) o = dv[e];
        if (l == CGL_Z) o = q;
        const bool mine = l < CGL_R;
        if (b0 && mine) v.x = l == CGL_X ? v.x + ax0 * o.x : o.x + v.x * be0;
        if (b1 && mine) v.y = l == CGL_X ? v.y + ax1 * o.y : o.y + v.y * be1;
      }
      // A of the next iteration: r -= alpha ss; u -= alpha v; w -= alpha z; d = M^-1 w (:1113-1123)
      const double2 o = from(v, l >= CGL_R ? l - (CGL_R - CGL_SS) : l);
      if (l >= CGL_R) {
        if (a0) v.x -= aa0 * o.x;
        if (a1) v.y -= aa1 * o.y;
      }
      const double2 u = from(v, CGL_U);
      if (l == CGL_R || l == CGL_W) {   // (zeros past the panel's end)
        const int k = l == CGL_R ? 0 : 1;
        prod[k][row - r0] = a0 ? u.x * v.x : 0.0;
        prod[2 + k][row - r0] = a1 ? u.y * v.y : 0.0;
      }
      if (live) {
        const bool write = l < CGL_R ? b0 || b1 : a0 || a1;
        if (write) A.V.state[(size_t)row * CGL_COUNT + l] = v;
        if (l == CGL_W && (a0 || a1)) {
          double2 *dn = PH == PH_A1 ? A.V.d[0] : A.par_in ? A.V.d[0] : A.V.d[1];
          dn[row] = make_double2(a0 ? v.x * co[e] : 0.0, a1 ? v.y * co[e] : 0.0);
        }
        if (PH == PH_K && l == CGL_X && !a0 && !a1) A.V.x[row] = v;   // both solves end here
      }
    }
  }
  if (!DOTS) return true;
  // ---- the panel's partial dots, each by one wave over the rows
  lds_barrier();
  for (int k = wave_in_block(); k < NDOUT; k += NW) {
    const double v = wave_sum(prod[k][lane_id()]);
    if (lane_id() == 0) A.part_out[(size_t)k * A.pstride + p] = v;
  }
  return true;
}

// Before a solve: no system has finished; a system without rows keeps the
// counts.
__device__ __forceinline__ void small_begin(const SmallArgs &A) {
  for (int k = threadIdx.x; k < 2 * A.nsys; k += blockDim.x) A.iters_out[k] = 1;
  if (threadIdx.x == 0) *A.done_count = 0;
}

template <int PH, int SH>
__global__ void __launch_bounds__(SpmvShape<SH>::NT)
k_cg_small(SmallArgs A) {
  __shared__ SmallLds<small_multiplies(PH) ? SMALL_ROWS : 1, small_dots_out(PH) ? small_dots_out(PH) : 1> S;
  if (PH == PH_S1 && blockIdx.x == 0) small_begin(A);
  small_step_body<PH, SH>(A, blockIdx.x, S);
}

// ---------------------------------------------------------------- tiny systems
// When every system has at most TINY_PANELS panels, one workgroup runs its
// system's whole solve in one launch: the steps above in turn, a barrier
// between steps.  A launch per iteration is 6.5 us of latency for 2 us of
// work, fifteen to twenty times over (charges of 60 atoms 216 us, of 64 such
// systems 265; this 153 and 171, 512 of them 343 either way).  The same
// functions in the same order: the same bits.  With two panels a workgroup
// would take them in turn that the launches spread over the chip: 120 atoms
// 323 us against 280.
constexpr int TINY_PANELS = 1;
constexpr int TINY_ROWS = TINY_PANELS * SWR_PANEL_ROWS;

__global__ void __launch_bounds__(256) k_cg_tiny_begin(SmallArgs A) { small_begin(A); }

// Scalars and dots of step k: step k reads those of step k - 1 and writes the
// other buffers.
__host__ __device__ inline void small_buffers(SmallArgs &A, CgScalars *cgs, double *partials, int ph, int step) {
  const size_t half = 2 * (size_t)A.nsys, odd = (size_t)SMALL_PART_ODD * A.pstride;
  const bool k_odd = ph == PH_K && (step & 1);
  A.cin = cgs + (ph == PH_K && !k_odd ? half : 0);
  A.cout = cgs + (k_odd ? half : 0);
  A.part_in = partials + (k_odd ? odd : 0);
  A.part_out = partials + (ph == PH_S3 || k_odd ? 0 : odd);
  A.par_in = (step - 1) & 1;
}

template <int SH>
__global__ void __launch_bounds__(SpmvShape<SH>::NT)
k_cg_tiny(SmallArgs A, CgScalars *cgs, double *partials, const int *__restrict__ sys_panel) {
  __shared__ SmallLds<TINY_ROWS, 6> S;
  const int p0 = sys_panel[blockIdx.x], p1 = sys_panel[blockIdx.x + 1];
  if (p0 >= p1) return;
  auto phase = [&](auto phc, int step) {
    constexpr int PH = decltype(phc)::value;
    small_buffers(A, cgs, partials, PH, step);
    bool on = true;
    for (int p = p0; p < p1; p++) {
      on = small_step_body<PH, SH>(A, p, S);
      __syncthreads();   // the next step reads what this one stored
    }
    return on;
  };
  phase(std::integral_constant<int, PH_S1>(), 0);
  phase(std::integral_constant<int, PH_S2>(), 0);
  phase(std::integral_constant<int, PH_S3>(), 0);
  if (!phase(std::integral_constant<int, PH_A1>(), 0)) return;
  for (int k = 1; k <= A.imax; k++)
    if (!phase(std::integral_constant<int, PH_K>(), k)) return;
}

// The vectors in CG scratch of CGV_COUNT slots of cap entries.
inline SmallVecs small_vecs(const CgRun<double, double> &R, double2 *base, size_t cap) {
  static_assert(CGL_COUNT + 2 <= CGV_COUNT, "the CG vectors hold the row states");
  SmallVecs V;
  V.x = R.V.x;
  V.b = R.V.b;
  V.Hd = R.V.Hd;
  V.state = base;
  V.d[0] = base + CGL_COUNT * cap;
  V.d[1] = base + (CGL_COUNT + 1) * cap;
  return V;
}

inline SmallArgs small_args(const swr_system *S, const CgRun<double, double> &R, const SmallVecs &V, int ph, int step) {
  SmallArgs A;
  A.P = S->dp;
  A.type = S->type;
  A.firstnbr = S->H_firstnbr;
  A.numnbrs = S->H_numnbrs;
  A.jlist = S->H_jlist;
  A.val = R.val;
  A.panel = (const SmallPanel *)S->small_panel;
  A.V = V;
  A.pstride = R.pstride;
  A.nsys = R.L.nsys;
  small_buffers(A, R.cgs, R.partials, ph, step);
  A.imax = R.imax;
  A.tol = R.tol;
  A.iters_out = R.iters_out;
  A.done_count = R.L.done_count;
  A.status = S->status;
  return A;
}

// The steps of the solve; step 0 is each setup phase, steps 1.. are PH_K.
inline int small_step(swr_system *S, const CgRun<double, double> &R, const SmallVecs &V, int ph, int step) {
  const SmallArgs A = small_args(S, R, V, ph, step);
  const int kt = ph == PH_K ? R.kt_iter : R.kt_setup;
  if (S->cg_tiny) {   // the first step is the whole solve
    if (ph != PH_S1) return SWR_OK;
    swr_kt_begin(S, kt);
    hipLaunchKernelGGL(k_cg_tiny_begin, dim3(1), dim3(256), 0, S->stream, A);
    spmv_dispatch(S->spmv_shape[0], [&](auto shc) {
      constexpr int SH = decltype(shc)::value;
      hipLaunchKernelGGL(k_cg_tiny<SH>, dim3((unsigned)S->sys_row.size() - 1), dim3(SpmvShape<SH>::NT), 0, S->stream, A,
                         R.cgs, R.partials, (const int *)S->sys_panel);
    });
    swr_kt_end(S, kt);
    HIP_CHECK(hipGetLastError());
    return SWR_OK;
  }
  swr_kt_begin(S, kt);
  spmv_dispatch(S->spmv_shape[0], [&](auto shc) {
    constexpr int SH = decltype(shc)::value;
    const dim3 gb(S->npanel), tb(SpmvShape<SH>::NT);
#define SMALL_LAUNCH(PHASE) hipLaunchKernelGGL((k_cg_small<PHASE, SH>), gb, tb, 0, S->stream, A)
    switch (ph) {
      case PH_S1: SMALL_LAUNCH(PH_S1); break;
      case PH_S2: SMALL_LAUNCH(PH_S2); break;
      case PH_S3: SMALL_LAUNCH(PH_S3); break;
      case PH_A1: SMALL_LAUNCH(PH_A1); break;
      default: SMALL_LAUNCH(PH_K); break;
    }
#undef SMALL_LAUNCH
  });
  swr_kt_end(S, kt);
  HIP_CHECK(hipGetLastError());
  return SWR_OK;
}

// Whether every system has at most TINY_PANELS panels (and the rule below holds).
inline bool tiny_rule(const std::vector<int> &sys_row) {
  for (size_t k = 0; k + 1 < sys_row.size(); k++)
    if (sys_row[k + 1] - sys_row[k] > TINY_ROWS) return false;
  return true;
}

// Whether the rule above holds for S's systems.
inline bool small_rule(const std::vector<int> &sys_row, int mixed) {
  long long panels = 0;
  for (size_t k = 0; k + 1 < sys_row.size(); k++) {
    const int rows = sys_row[k + 1] - sys_row[k];
    if (rows > SMALL_ROWS) return false;
    panels += div_up(rows, SWR_PANEL_ROWS);
  }
  return !mixed && panels <= SMALL_PANELS;
}

}  // namespace swr_cg
