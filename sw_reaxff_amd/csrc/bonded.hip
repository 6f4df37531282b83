// bonded.hip — bond and atom energies and the bond-order chain rule of the
// forces:
//
//   Atom_Energy (reaxc_multi_body_sunway.cpp:41-57) = Merge_Bonds_Atom_Energy_C_New
//   (reaxc_multi_body_sw64.c:21-337): per local atom the polarization, lone-pair
//   (+ C-C correction), over- and under-coordination energies, and for each
//   bond the atom owns the bond energy and the terminal triple-bond
//   stabilisation; the coefficients Cdbo/Cdbopi/Cdbopi2 of each bond slot and
//   CdDelta (fCdDelta[.][3]) of the atoms.  (Bonds() itself returns at once,
//   reaxc_bonds_sunway.cpp:49-52.)
//
//   Add_All_dBond_to_Forces_C (reaxc_forces_sw64.c:417-589): over all N atoms
//   and their bonds, the chain rule of the bond-order derivatives into
//   fCdDelta[.][0..2] (the energy gradient, as the non-bonded pass writes it).
//
// The reference loops over atoms and adds into the neighbours' entries as it
// goes.  Here every kernel writes only entries of its own atom, so no
// floating-point atomics are needed and results are the same on every run:
//
//   k_atom_energy     four lanes per local atom: energies (per-atom rows,
//                     summed in a fixed order by sum_row), its own bond
//                     slots' coefficients, its own CdDelta, and the two
//                     per-atom factors (CEover4, CEunder4) its neighbours need;
//   k_atom_energy_nbr one thread per atom (local and ghost): the CdDelta terms
//                     the reference adds to atom j from each bonded local atom
//                     i, read through the bond's reverse slot (sym_index), so
//                     the values are those i's own slot holds;
//   k_dbond_own       four lanes per atom: its own chain-rule terms and the
//                     factor buf_c it passes to its neighbours;
//   k_dbond_nbr       one thread per atom: sum over its bonds of the
//                     neighbour's buf_c times the neighbour's dBOp toward it.
//
// Each atom's terms are added in the reference's order for that atom; only
// the interleaving of its own and its neighbours' terms differs, which moves
// results at the rounding level.
#include "swr_internal.h"
#include "swr_device.h"

#include <algorithm>

namespace {

constexpr int BT = 256;
constexpr double KCALpMOL_to_EV = 23.02;   // reaxc_defs_sunway.h:68

__device__ __forceinline__ double sqr(double x) { return x * x; }

// Local atom i owns bond (i, j) for the bond energy: the smaller orig_id, or
// for two images of one atom the lower in z, then y, then x (:245-255).
__device__ __forceinline__ bool owns_bond(const swr_atom_pack_t &a, const swr_atom_pack_t &b) {
  if (a.orig_id > b.orig_id) return false;
  if (a.orig_id == b.orig_id) {
    if (b.x[2] < a.x[2]) return false;
    if (b.x[2] == a.x[2] && b.x[1] < a.x[1]) return false;
    if (b.x[2] == a.x[2] && b.x[1] == a.x[1] && b.x[0] < a.x[0]) return false;
  }
  return true;
}

// Terminal triple-bond stabilisation of bond (i, j) owned by i (:283-308):
// the energy and, as pairs of factors, the terms for Cdbo of i's slot
// (dbo_x dbo_y), CdDelta of i (x ua) and CdDelta of j (x ub).
struct TripleBond {
  double e, dbo_x, dbo_y, x, ua, ub;
};

// Whether it applies; t is only then set.
__device__ __forceinline__ bool triple_bond(const DevParams *__restrict__ P, int ti, int tj, double BOij,
                                            double dboc_i, double dboc_j, double Delta_i, double Delta_j,
                                            TripleBond &t) {
  const double mi = P->mass[ti], mj = P->mass[tj];
  if (!(BOij >= 1.00 && (P->gp37 == 2 || (mi == 12.0000 && mj == 15.9990) || (mj == 12.0000 && mi == 15.9990))))
    return false;
  const double gp3 = P->gp3, gp4 = P->gp4, gp7 = P->gp7, gp10 = P->gp10;
  const double exphu = exp(-gp7 * sqr(BOij - 2.50));
  const double exphua1 = exp(-gp3 * (dboc_i - BOij));
  const double exphub1 = exp(-gp3 * (dboc_j - BOij));
  const double exphuov = exp(gp4 * (Delta_i + Delta_j));
  const double hulpov = 1.0 / (1.0 + 25.0 * exphuov);
  t.e = gp10 * exphu * hulpov * (exphua1 + exphub1);
  t.dbo_x = t.e;
  t.dbo_y = gp3 - 2.0 * gp7 * (BOij - 2.50);
  t.x = -gp10 * exphu * hulpov;
  t.ua = gp3 * exphua1 + 25.0 * gp4 * exphuov * hulpov * (exphua1 + exphub1);
  t.ub = gp3 * exphub1 + 25.0 * gp4 * exphuov * hulpov * (exphua1 + exphub1);
  return true;
}

// Lanes of an atom in the passes that spread its bonds, and the atoms of a
// workgroup there.  Most atoms have two to four bonds.
constexpr int BG = 4;
constexpr int AE_ATOMS = BT / BG;

// Butterfly sum of a group of G lanes, on all of them.
template <int G>
__device__ __forceinline__ double group_sum(double v) {
#pragma unroll
  for (int o = G / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, SWR_WAVE);
  return v;
}

// The largest v of a wave whose groups of G lanes each hold one value.
template <int G>
__device__ __forceinline__ int wave_max_groups(int v) {
#pragma unroll
  for (int o = G; o < SWR_WAVE; o <<= 1) v = max(v, __shfl_xor(v, o, SWR_WAVE));
  return v;
}

// One workgroup's fixed-order sum of a per-atom energy row: 1024 running sums
// over every 1024th entry, then a tree over them.  Each thread keeps four of
// the sums and U entries of each in flight (one entry at a time left the row
// waiting for memory: 147 us on 200,000 atoms).  Run by the first workgroups
// of the launch that follows the row's producer.
template <int U>
__device__ __forceinline__ void sum_row(int n, const double *__restrict__ row, double *__restrict__ out) {
  __shared__ double s[BT];
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  const int t = threadIdx.x;
  int base = 0;
  for (; base + 1024 * U <= n; base += 1024 * U) {
    double v[U][4];
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int q = 0; q < 4; q++) v[u][q] = row[base + 1024 * u + BT * q + t];
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int q = 0; q < 4; q++) acc[q] += v[u][q];
  }
  for (; base < n; base += 1024) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int i = base + BT * q + t;
      if (i < n) acc[q] += row[i];
    }
  }
  s[t] = (acc[0] + acc[2]) + (acc[1] + acc[3]);
  __syncthreads();
  for (int o = BT / 2; o > 0; o >>= 1) {
    if (t < o) s[t] += s[t + o];
    __syncthreads();
  }
  if (t == 0) *out = s[0];
}

struct BeArgs {
  const DevParams *P;
  const swr_atom_pack_t *atoms;
  const int *bidx, *bend;
  const swr_bond_t *bonds;
  const swr_bond_order_t *bo;
  const double *BO, *BOpi;       // BOpi: [slot][2]
  const double *Delta, *Delta_lp, *dDelta_lp, *Delta_lp_temp;
  const double *bo_dboc;         // [N][2]
  double *Cdbo, *Cdbopi, *Cdbopi2;
  double *fcd;                   // [N][4]
  double *ce;                    // [2][stride]: CEover4, CEunder4
  double *part;                  // [5][stride]
  size_t stride;
};

// What a workgroup's lanes hand from one part of k_atom_energy to the next.
struct BeAtoms {
  double ovun1[AE_ATOMS], ovun2[AE_ATOMS], cdd[AE_ATOMS], e_lp[AE_ATOMS];   // sums over the bonds
  double over1[AE_ATOMS], over4[AE_ATOMS], under4[AE_ATOMS];                // CEover1, CEover4, CEunder4
};

// A chain of loads and transcendentals per bond and one per atom, at one to
// two waves a SIMD: one thread per atom left it waiting (19 us on 21 atoms, 27
// on 1,944, 464 on 200,000).  Here BG lanes take an atom's bonds, one lane
// per atom the part between the bond loops, and sums over bonds are made in
// bond order, with the operands of each term exchanged, so they round as one
// thread's loop does.
__global__ void __launch_bounds__(BT) k_atom_energy(int n, BeArgs A) {
  __shared__ BeAtoms S;
  const DevParams *__restrict__ P = A.P;
  const int a = threadIdx.x / BG, sl = threadIdx.x % BG;
  const int i = blockIdx.x * AE_ATOMS + a;
  swr_atom_pack_t ai = {};
  ai.type = -1;
  if (i < n) ai = A.atoms[i];
  const int ti = ai.type;
  const bool live = ti >= 0;
  const int b0 = live ? A.bidx[i] : 0, b1 = live ? A.bend[i] : 0;
  const int nbmax = wave_max_groups<BG>(b1 - b0);
  const double Di = live ? A.Delta[i] : 0.0;
  const double dfvl = live && P->mass[ti] > 21.0 ? 0.0 : 1.0;   // 1st-row elements only
  const bool carbon = live && P->p_lp3 > 0.001 && P->is_carbon[ti];
  {
    double sum_ovun1 = 0, sum_ovun2 = 0, e_lp = 0;
    double cdd = live ? A.fcd[4 * (size_t)i + 3] : 0.0;
    for (int m0 = 0; m0 < nbmax; m0 += BG) {
      const int pj = b0 + m0 + sl;
      double x1 = 0, y1 = 0, x2 = 0, y2 = 0;   // terms x1 y1 of sum_ovun1, x2 y2 of sum_ovun2
      double xc = 0, yc = 0, xl = 0, yl = 0;   // carbon: of CdDelta and of e_lp
      bool lp3 = false;
      if (pj < b1) {
        const int j = A.bonds[pj].nbr;
        const int tj = A.atoms[j].type;
        if (tj >= 0) {
          const DevBe &tw = P->be[ti * SWR_MAX_ELEM + tj];
          x1 = tw.p_ovun1 * tw.De_s;
          y1 = A.BO[pj];
          x2 = A.Delta[j] - dfvl * A.Delta_lp_temp[j];
          y2 = A.BOpi[2 * (size_t)pj] + A.BOpi[2 * (size_t)pj + 1];
          if (carbon && P->is_carbon[tj]) {
            const double vov3 = y1 - Di - 0.040 * pow(Di, 4.);
            if (vov3 > 3.) {
              lp3 = true;
              xl = P->p_lp3;
              yl = sqr(vov3 - 3.0);
              xc = 2. * P->p_lp3 * (vov3 - 3.);
              yc = -1. - 0.16 * pow(Di, 3.);
              A.Cdbo[pj] += xc;
            }
          }
        }
      }
      const bool any_lp3 = __ballot(lp3) != 0ull;
#pragma unroll
      for (int q = 0; q < BG; q++) {
        sum_ovun1 += __shfl(x1, q, BG) * __shfl(y1, q, BG);
        sum_ovun2 += __shfl(x2, q, BG) * __shfl(y2, q, BG);
      }
      if (any_lp3) {
#pragma unroll
        for (int q = 0; q < BG; q++) {
          const double c = __shfl(xc, q, BG), d = __shfl(yc, q, BG), e = __shfl(xl, q, BG), f = __shfl(yl, q, BG);
          if (e != 0.0) {
            e_lp += e * f;
            cdd += c * d;
          }
        }
      }
    }
    if (sl == 0) {
      S.ovun1[a] = sum_ovun1;
      S.ovun2[a] = sum_ovun2;
      S.e_lp[a] = e_lp;
      S.cdd[a] = cdd;
    }
  }
  __syncthreads();
  // ---- one lane per atom: the terms of the whole atom
  if (threadIdx.x < AE_ATOMS) {
    const int t = threadIdx.x, i = blockIdx.x * AE_ATOMS + t;
    double e_lp = 0, e_ov = 0, e_un = 0, e_pol = 0, ceo4 = 0, ceu4 = 0;
    swr_atom_pack_t ai = {};
    ai.type = -1;
    if (i < n) ai = A.atoms[i];
    const int ti = ai.type;
    if (ti >= 0) {
      const double q = ai.q;
      e_pol = KCALpMOL_to_EV * (P->chi_e[ti] * q + (P->eta_e[ti] / 2.) * sqr(q));
      const int numbonds = A.bend[i] - A.bidx[i];
      const double sum_ovun1 = S.ovun1[t], sum_ovun2 = S.ovun2[t];
      e_lp = S.e_lp[t];
      double cdd = S.cdd[t];
      // lone pair
      const double p_lp2 = P->p_lp2[ti];
      const double Dlp = A.Delta_lp[i];
      const double expvd2 = exp(-75 * Dlp);
      const double inv_expvd2 = 1. / (1. + expvd2);
      const double p_ovun2 = P->p_ovun2[ti];
      const double dfvl = P->mass[ti] > 21.0 ? 0.0 : 1.0;
      const double dElp = p_lp2 * inv_expvd2 + 75 * p_lp2 * Dlp * expvd2 * sqr(inv_expvd2);
      const double CElp = dElp * A.dDelta_lp[i];
      const double Di = A.Delta[i];
      // over-coordination
      const double p_ovun4 = P->p_ovun4;
      const double exp_ovun1 = P->p_ovun3 * exp(p_ovun4 * sum_ovun2);
      const double inv_exp_ovun1 = 1.0 / (1 + exp_ovun1);
      const double Dlpt = A.Delta_lp_temp[i];
      const double Delta_lpcorr = Di - (dfvl * Dlpt) * inv_exp_ovun1;
      const double exp_ovun2 = exp(p_ovun2 * Delta_lpcorr);
      const double inv_exp_ovun2 = 1.0 / (1.0 + exp_ovun2);
      const double DlpVi = 1.0 / (Delta_lpcorr + P->valency[ti] + 1e-8);
      const double CEover1 = Delta_lpcorr * DlpVi * inv_exp_ovun2;
      e_ov = sum_ovun1 * CEover1;
      const double CEover2 =
          sum_ovun1 * DlpVi * inv_exp_ovun2 * (1.0 - Delta_lpcorr * (DlpVi + p_ovun2 * exp_ovun2 * inv_exp_ovun2));
      const double dDlp = A.dDelta_lp[i];
      const double CEover3 = CEover2 * (1.0 - dfvl * dDlp * inv_exp_ovun1);
      ceo4 = CEover2 * (dfvl * Dlpt) * p_ovun4 * exp_ovun1 * sqr(inv_exp_ovun1);
      // under-coordination
      const double p_ovun5 = P->p_ovun5[ti];
      const double exp_ovun2n = 1.0 / exp_ovun2;
      const double exp_ovun6 = exp(P->p_ovun6 * Delta_lpcorr);
      const double exp_ovun8 = P->p_ovun7 * exp(P->p_ovun8 * sum_ovun2);
      const double inv_exp_ovun2n = 1.0 / (1.0 + exp_ovun2n);
      const double inv_exp_ovun8 = 1.0 / (1.0 + exp_ovun8);
      cdd += CEover3;
      const bool under = numbonds > 0 || P->enobonds;
      double eu = 0.0;
      if (under) eu = -p_ovun5 * (1.0 - exp_ovun6) * inv_exp_ovun2n * inv_exp_ovun8;
      const double CEunder1 =
          inv_exp_ovun2n * (p_ovun5 * P->p_ovun6 * exp_ovun6 * inv_exp_ovun8 + p_ovun2 * eu * exp_ovun2n);
      const double CEunder2 = -eu * P->p_ovun8 * exp_ovun8 * inv_exp_ovun8;
      const double CEunder3 = CEunder1 * (1.0 - dfvl * dDlp * inv_exp_ovun1);
      ceu4 = CEunder1 * (dfvl * Dlpt) * p_ovun4 * exp_ovun1 * sqr(inv_exp_ovun1) + CEunder2;
      if (under) {
        e_un = eu;
        cdd += CEunder3;
        cdd += CElp;
        e_lp += p_lp2 * Dlp * inv_expvd2;
      }
      S.over1[t] = CEover1;
      S.over4[t] = ceo4;
      S.under4[t] = ceu4;
      S.cdd[t] = cdd;
    }
    if (i < n) {
      A.ce[i] = ceo4;
      A.ce[A.stride + i] = ceu4;
      A.part[A.stride + i] = e_lp;
      A.part[2 * A.stride + i] = e_ov;
      A.part[3 * A.stride + i] = e_un;
      A.part[4 * A.stride + i] = e_pol;
    }
  }
  __syncthreads();
  // ---- per bond: over/under-coordination coefficients of this slot, bond
  // energy and triple-bond stabilisation of the bonds this atom owns
  double e_bond = 0.0, cdd = S.cdd[a];
  const double CEover1 = S.over1[a], ceo4 = S.over4[a], ceu4 = S.under4[a];
  for (int m0 = 0; m0 < nbmax; m0 += BG) {
    const int pj = b0 + m0 + sl;
    double eb = 0, e3 = 0;                 // bond energy, triple-bond energy
    TripleBond tb = {};
    bool triple = false;
    if (pj < b1) {
      const int j = A.bonds[pj].nbr;
      const swr_atom_pack_t aj = A.atoms[j];
      const int tj = aj.type;
      if (tj >= 0) {
        const DevBe &tw = P->be[ti * SWR_MAX_ELEM + tj];
        double cdbo = A.Cdbo[pj], cdbopi = A.Cdbopi[pj], cdbopi2 = A.Cdbopi2[pj];
        cdbo += CEover1 * tw.p_ovun1 * tw.De_s;
        const double dj = A.Delta[j] - dfvl * A.Delta_lp_temp[j];
        const double ftmp = ceo4 * dj;
        cdbopi += ftmp;
        cdbopi2 += ftmp;
        const double fu = ceu4 * dj;
        cdbopi += fu;
        cdbopi2 += fu;
        if (owns_bond(ai, aj)) {
          const double BO_s = A.bo[pj].BO_s;
          const double pow_BOs_be2 = BO_s == 0.0 ? 0.0 : pow(BO_s, tw.p_be2);
          const double exp_be12 = exp(tw.p_be1 * (1.0 - pow_BOs_be2));
          const double CEbo = -tw.De_s * exp_be12 * (1.0 - tw.p_be1 * tw.p_be2 * pow_BOs_be2);
          eb = -tw.De_s * BO_s * exp_be12 - tw.De_p * A.BOpi[2 * (size_t)pj] - tw.De_pp * A.BOpi[2 * (size_t)pj + 1];
          cdbo += CEbo;
          cdbopi -= (CEbo + tw.De_p);
          cdbopi2 -= (CEbo + tw.De_pp);
          triple = triple_bond(P, ti, tj, A.BO[pj], A.bo_dboc[2 * (size_t)i], A.bo_dboc[2 * (size_t)j], Di, A.Delta[j],
                               tb);
          if (triple) {
            e3 = tb.e;
            cdbo += tb.dbo_x * tb.dbo_y;
          }
        }
        A.Cdbo[pj] = cdbo;
        A.Cdbopi[pj] = cdbopi;
        A.Cdbopi2[pj] = cdbopi2;
      }
    }
    const bool any_triple = __ballot(triple) != 0ull;
#pragma unroll
    for (int q = 0; q < BG; q++) {
      e_bond += __shfl(eb, q, BG);
      if (any_triple) {
        e_bond += __shfl(e3, q, BG);
        cdd += __shfl(tb.x, q, BG) * __shfl(tb.ua, q, BG);
      }
    }
  }
  if (sl == 0 && i < n) {
    A.part[i] = e_bond;
    if (live) A.fcd[4 * (size_t)i + 3] = cdd;
  }
}

// CdDelta terms of atom j from each bonded local atom i (:270-279 and the
// triple-bond term :305), read through i's slot toward j; the first five
// workgroups sum k_atom_energy's rows.
__global__ void __launch_bounds__(BT) k_atom_energy_nbr(int n, int N, BeArgs A, double *__restrict__ sums) {
  if (blockIdx.x < 5) {
    sum_row<8>(n, A.part + blockIdx.x * A.stride, sums + blockIdx.x);
    return;
  }
  const int j = (blockIdx.x - 5) * BT + threadIdx.x;
  if (j >= N) return;
  const DevParams *__restrict__ P = A.P;
  const swr_atom_pack_t aj = A.atoms[j];
  const int tj = aj.type;
  if (tj < 0) return;
  const int b0 = A.bidx[j], b1 = A.bend[j];
  if (b0 >= b1) return;
  double cdd = A.fcd[4 * (size_t)j + 3];
  const double dDlp_j = A.dDelta_lp[j];
  for (int pk = b0; pk < b1; ++pk) {
    const swr_bond_t b = A.bonds[pk];
    const int i = b.nbr;
    if (i >= n) continue;
    const swr_atom_pack_t ai = A.atoms[i];
    const int ti = ai.type;
    if (ti < 0) continue;
    const int pj = b.sym_index;   // i's slot toward j
    const double dfvl = P->mass[ti] > 21.0 ? 0.0 : 1.0;
    const double ftmp2 = (1.0 - dfvl * dDlp_j) * (A.BOpi[2 * (size_t)pj] + A.BOpi[2 * (size_t)pj + 1]);
    cdd += A.ce[i] * ftmp2;
    cdd += A.ce[A.stride + i] * ftmp2;
    if (owns_bond(ai, aj)) {
      TripleBond t;
      if (triple_bond(P, ti, tj, A.BO[pj], A.bo_dboc[2 * (size_t)i], A.bo_dboc[2 * (size_t)j], A.Delta[i],
                      A.Delta[j], t))
        cdd += t.x * t.ub;
    }
  }
  A.fcd[4 * (size_t)j + 3] = cdd;
}

struct DbArgs {
  const swr_bond_t *bonds;
  const swr_bond_order_t *bo;
  const int *bidx, *bend;
  const double *Cdbo, *Cdbopi, *Cdbopi2;
  const double *dDeltap_self;    // [N][3]
  double *fcd;                   // [N][4]
  double *bufc;                  // [N]
};

// The atom's own terms (the reference's forces on i, :532-548) and buf_c: BG
// lanes per atom over its bonds, whose terms are added in bond order (one
// thread per atom waited bond by bond for four gathers: 16 us on 192 atoms
// with their ghosts, 17 on 1,944, 340 on 200,000).
__global__ void __launch_bounds__(BT) k_dbond_own(int N, DbArgs A) {
  const int tid = blockIdx.x * BT + threadIdx.x;
  const int i = tid / BG, sl = tid % BG;
  const int b0 = i < N ? A.bidx[i] : 0, b1 = i < N ? A.bend[i] : 0;
  const int nbmax = wave_max_groups<BG>(b1 - b0);
  double buf_c = 0.0, f0 = 0.0, f1 = 0.0, f2 = 0.0;
  double ds0 = 0.0, ds1 = 0.0, ds2 = 0.0, cd_i = 0.0;
  if (b0 < b1) {
    ds0 = A.dDeltap_self[3 * (size_t)i];
    ds1 = A.dDeltap_self[3 * (size_t)i + 1];
    ds2 = A.dDeltap_self[3 * (size_t)i + 2];
    f0 = A.fcd[4 * (size_t)i];
    f1 = A.fcd[4 * (size_t)i + 1];
    f2 = A.fcd[4 * (size_t)i + 2];
    cd_i = A.fcd[4 * (size_t)i + 3];
  }
  for (int m0 = 0; m0 < nbmax; m0 += BG) {
    const int pj = b0 + m0 + sl;
    double t0 = 0.0, t1 = 0.0, t2 = 0.0, tc = 0.0;
    if (pj < b1) {
      const swr_bond_t b = A.bonds[pj];
      const int j = b.nbr, sym = b.sym_index;
      const swr_bond_order_t &bo = A.bo[pj];
      const double cdbo = A.Cdbo[pj] + A.Cdbo[sym];
      const double cdbopi = A.Cdbopi[pj] + A.Cdbopi[sym];
      const double cdbopi2 = A.Cdbopi2[pj] + A.Cdbopi2[sym];
      const double C1dbo = bo.C1dbo * cdbo, C2dbo = bo.C2dbo * cdbo;
      const double C1dbopi = bo.C1dbopi * cdbopi, C2dbopi = bo.C2dbopi * cdbopi, C3dbopi = bo.C3dbopi * cdbopi;
      const double C1dbopi2 = bo.C1dbopi2 * cdbopi2, C2dbopi2 = bo.C2dbopi2 * cdbopi2,
                   C3dbopi2 = bo.C3dbopi2 * cdbopi2;
      const double cdd = cd_i + A.fcd[4 * (size_t)j + 3];
      const double C1dDelta = bo.C1dbo * cdd, C2dDelta = bo.C2dbo * cdd;
      const double dbx = bo.dBOp[0], dby = bo.dBOp[1], dbz = bo.dBOp[2];
      t0 = C1dbo * dbx; t1 = C1dbo * dby; t2 = C1dbo * dbz;
      t0 += C2dbo * ds0; t1 += C2dbo * ds1; t2 += C2dbo * ds2;
      t0 += C1dDelta * dbx; t1 += C1dDelta * dby; t2 += C1dDelta * dbz;
      t0 += C2dDelta * ds0; t1 += C2dDelta * ds1; t2 += C2dDelta * ds2;
      t0 += C1dbopi * bo.dln_BOp_pi[0]; t1 += C1dbopi * bo.dln_BOp_pi[1]; t2 += C1dbopi * bo.dln_BOp_pi[2];
      t0 += C2dbopi * dbx; t1 += C2dbopi * dby; t2 += C2dbopi * dbz;
      t0 += C3dbopi * ds0; t1 += C3dbopi * ds1; t2 += C3dbopi * ds2;
      t0 += C1dbopi2 * bo.dln_BOp_pi2[0]; t1 += C1dbopi2 * bo.dln_BOp_pi2[1]; t2 += C1dbopi2 * bo.dln_BOp_pi2[2];
      t0 += C2dbopi2 * dbx; t1 += C2dbopi2 * dby; t2 += C2dbopi2 * dbz;
      t0 += C3dbopi2 * ds0; t1 += C3dbopi2 * ds1; t2 += C3dbopi2 * ds2;
      tc = -C2dbo - C2dDelta - C3dbopi - C3dbopi2;
    }
#pragma unroll
    for (int q = 0; q < BG; q++) {
      const double g0 = __shfl(t0, q, BG), g1 = __shfl(t1, q, BG), g2 = __shfl(t2, q, BG), gc = __shfl(tc, q, BG);
      if (b0 + m0 + q < b1) {
        f0 += g0;
        f1 += g1;
        f2 += g2;
        buf_c += gc;
      }
    }
  }
  if (i >= N) return;
  if (sl == 3) A.bufc[i] = buf_c;
  else if (b0 < b1) A.fcd[4 * (size_t)i + sl] = sl == 0 ? f0 : sl == 1 ? f1 : f2;
}
static_assert(BG == 4, "a lane of k_dbond_own writes one column");

// The terms the reference adds to k from each bonded atom i (forces on k,
// :580-584): buf_c of i times i's dBOp toward k.
__global__ void __launch_bounds__(BT) k_dbond_nbr(int N, DbArgs A) {
  const int k = blockIdx.x * BT + threadIdx.x;
  if (k >= N) return;
  const int b0 = A.bidx[k], b1 = A.bend[k];
  if (b0 >= b1) return;
  double f0 = A.fcd[4 * (size_t)k], f1 = A.fcd[4 * (size_t)k + 1], f2 = A.fcd[4 * (size_t)k + 2];
  for (int pk = b0; pk < b1; ++pk) {
    const swr_bond_t b = A.bonds[pk];
    const double c = A.bufc[b.nbr];
    const double *d = A.bo[b.sym_index].dBOp;
    f0 += c * d[0];
    f1 += c * d[1];
    f2 += c * d[2];
  }
  A.fcd[4 * (size_t)k] = f0;
  A.fcd[4 * (size_t)k + 1] = f1;
  A.fcd[4 * (size_t)k + 2] = f2;
}

// ---------------------------------------------------------------- hydrogen bonds
// Hydrogen_Bonds_C (reaxc_hydrogen_bonds_sw64.c:26-283, host loop :145-253):
// a triple is a local H atom j (p_hbond 1), a bond j-i to an acceptor
// (p_hbond 2) with BO >= 0.01, and a hydrogen-bond partner k of j with
// orig_id(k) != orig_id(i) and r0_hb(i, j, k) > 0.  Its energy and CEhb1
// (into Cdbo of j's slot) and the angle/distance terms into fCdDelta of i,
// j and k.  k_hb computes each triple once, half a wave per H atom with its
// lanes over the atom's hydrogen-bond entries: the energy, CEhb1 and j's own
// terms are summed by a fixed butterfly; the terms of i (summed over the
// entries, one set per bond) and of k (summed over the bonds, one set per
// entry) go into fixed-point accumulators (fix_add: 2^-40 resolution for
// every term, sums up to 2^43) by integer adds, whose sums do not depend
// on the order they arrive in; k_hb_fold adds them to fCdDelta and clears them.
// The results are the same on every run.
constexpr double HB_THRESHOLD = 1e-2;   // reaxc_defs_sunway.h:91
constexpr double HB_FIX = 1099511627776.0;   // 2^40

struct HbArgs {
  unsigned int *flags;   // DevStatus::flags
  const DevParams *P;
  const swr_atom_pack_t *atoms;
  const int *bidx, *bend;
  const swr_bond_t *bonds;
  const double *BO;
  const int *Hindex, *hidx, *hend;
  const swr_hbond_t *hbonds;
  double *Cdbo, *fcd, *part;
  unsigned long long *acc;   // [2][N][3] fixed-point terms of i and k (fine, then coarse words)
  size_t coff;               // 3N: offset of the coarse words
};

// One triple (Calculate_Theta, Calculate_dCos_Theta :336-372, energy and
// coefficients :224-235); the cube of 1/(d_ji d_jk) by two products where
// the reference calls p_powd.
struct HbTriple {
  double e, ce1, ce2, ce3;
  double di[3], dj[3], dk[3];
};

__device__ __forceinline__ void hb_triple(const DevHb &hbp, double BOij, const double *dvec_ji, double d_ji,
                                          const double *dvec_jk, double r_jk, HbTriple &t) {
  const double dot = dvec_ji[0] * dvec_jk[0] + dvec_ji[1] * dvec_jk[1] + dvec_ji[2] * dvec_jk[2];
  double cos_theta = dot / (d_ji * r_jk);
  if (cos_theta > 1.) cos_theta = 1.0;
  if (cos_theta < -1.) cos_theta = -1.0;
  const double sqr_d_ji = d_ji * d_ji, sqr_d_jk = r_jk * r_jk;
  const double inv_dists = 1.0 / (d_ji * r_jk);
  const double inv_dists3 = inv_dists * inv_dists * inv_dists;
  const double Cdot_inv3 = dot * inv_dists3;
#pragma unroll
  for (int c = 0; c < 3; c++) {
    t.di[c] = dvec_jk[c] * inv_dists - Cdot_inv3 * sqr_d_jk * dvec_ji[c];
    t.dj[c] = -(dvec_jk[c] + dvec_ji[c]) * inv_dists + Cdot_inv3 * (sqr_d_jk * dvec_ji[c] + sqr_d_ji * dvec_jk[c]);
    t.dk[c] = dvec_ji[c] * inv_dists - Cdot_inv3 * sqr_d_ji * dvec_jk[c];
  }
  // sin^4(theta/2) = ((1 - cos theta)/2)^2: the reference goes through acos
  // and sin; the identity gives the same value to rounding without either
  const double cos_xhz1 = (1.0 - cos_theta);
  double sin_xhz4 = 0.5 * cos_xhz1;
  sin_xhz4 *= sin_xhz4;
  const double exp_hb2 = exp(-hbp.p_hb2 * BOij);
  const double exp_hb3 = exp(-hbp.p_hb3 * (hbp.r0_hb / r_jk + r_jk / hbp.r0_hb - 2.0));
  t.e = hbp.p_hb1 * (1.0 - exp_hb2) * exp_hb3 * sin_xhz4;
  t.ce1 = hbp.p_hb1 * hbp.p_hb2 * exp_hb2 * exp_hb3 * sin_xhz4;
  t.ce2 = -hbp.p_hb1 / 2.0 * (1.0 - exp_hb2) * exp_hb3 * cos_xhz1;
  t.ce3 = -hbp.p_hb3 * (-hbp.r0_hb / (r_jk * r_jk) + 1.0 / hbp.r0_hb) * t.e;
}

// One fixed-point accumulator is a pair of 64-bit words: a fine word in
// units of 2^-40 (range 2^23) and a coarse word in units of 2^-20 (range
// 2^43), coff elements after it.  A term below 2^10 in magnitude goes to the
// fine word whole; a larger one is split exactly into a multiple of 2^-20
// (coarse word) and a remainder of at most 2^-21 (fine word).  Every term
// thus keeps the 2^-40 resolution (at most 2^-41 rounding per add), a term adds
// at most 2^10 to the fine word (8192 terms before it could wrap; k_hb adds the
// terms of a workgroup at once), and the pair holds sums up to 2^43.  Both words are integers, so the sums do not
// depend on the order the adds arrive in.  A non-finite term, a term beyond
// ~3.8e12 (2^62 coarse units), or an add that wraps a word (detected from the
// value atomicAdd returns) raises SWR_F_FIXED_RANGE, which the next swr_sync
// reports as SWR_ERR_NUMERIC.
constexpr double FIX_COARSE = 1048576.0;   // 2^20: coarse units
constexpr double FIX_SPLIT = 1024.0;       // terms at least this large are split

// Whether adding d to the word that held old wrapped it.
__device__ __forceinline__ bool fix_wrapped(unsigned long long old, long long d) {
  const long long o = (long long)old, sum = (long long)(old + (unsigned long long)d);
  return ((o ^ sum) & (d ^ sum)) < 0;
}

__device__ __forceinline__ void fix_word_add(unsigned int *flags, unsigned long long *a, long long d) {
  if (fix_wrapped(atomicAdd(a, (unsigned long long)d), d)) atomicOr(flags, SWR_F_FIXED_RANGE);
}

__device__ __forceinline__ void fix_add(unsigned int *flags, unsigned long long *a, size_t coff, double v) {
  if (!(fabs(v) < FIX_SPLIT)) {
    const double hi = rint(v * FIX_COARSE);
    if (!(fabs(hi) < 4.0e18)) {   // not finite, or beyond ~3.8e12
      atomicOr(flags, SWR_F_FIXED_RANGE);
      return;
    }
    fix_word_add(flags, a + coff, (long long)hi);
    v -= hi * (1.0 / FIX_COARSE);   // exact: |v - hi 2^-20| <= 2^-21
  }
  const long long f = llrint(v * HB_FIX);
  if (f != 0) fix_word_add(flags, a, f);
}

// K fix_adds whose fine-word results are checked for a wrap only after all
// K were issued, so a lane waits for the returned words once per group
// instead of once per add.  Terms of FIX_SPLIT and more (rare) take fix_add.
template <int K>
__device__ __forceinline__ void fix_add_group(unsigned int *flags, unsigned long long *const (&a)[K],
                                              const size_t (&coff)[K], const double (&v)[K]) {
  unsigned long long old[K];
  long long d[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    old[k] = 0ull;
    d[k] = 0;
    if (!(fabs(v[k]) < FIX_SPLIT)) {
      fix_add(flags, a[k], coff[k], v[k]);
    } else {
      d[k] = llrint(v[k] * HB_FIX);
      if (d[k] != 0) old[k] = atomicAdd(a[k], (unsigned long long)d[k]);
    }
  }
  bool wrap = false;
#pragma unroll
  for (int k = 0; k < K; ++k) wrap |= fix_wrapped(old[k], d[k]);
  if (wrap) atomicOr(flags, SWR_F_FIXED_RANGE);
}

// The value of the accumulator pair at a (coarse word coff elements on).
__device__ __forceinline__ double fix_value(const unsigned long long *a, size_t coff) {
  return (double)(long long)a[0] * (1.0 / HB_FIX) + (double)(long long)a[coff] * (1.0 / FIX_COARSE);
}

// A workgroup's sums of the fixed-point terms by atom: neighbouring H atoms
// have mostly the same partners, and a device-wide atomic costs a trip past
// the L2s (which eight XCDs do not share), an LDS one does not.  Words of
// terms below FIX_SPLIT; a workgroup makes at most HB_ATOMS times the bonds of
// an atom adds per atom, so an LDS word cannot wrap.
constexpr int HB_SLOTS = 1024;
struct HbTable {
  int key[HB_SLOTS];
  unsigned long long sum[3][HB_SLOTS];
};

// The slot of atom a, or -1 when it is not there and no slot is free nearby.
__device__ __forceinline__ int hb_slot(HbTable &T, int a) {
  int s = (int)(((unsigned)a * 2654435761u) >> 22);
  for (int q = 0; q < 16; q++) {
    int key = T.key[s];
    if (key != a && key < 0) key = atomicCAS(&T.key[s], -1, a);
    if (key == a || key < 0) return s;
    s = (s + 1) & (HB_SLOTS - 1);
  }
  return -1;
}
static_assert(HB_SLOTS == 1 << (32 - 22), "hb_slot's shift leaves a slot number");

// Component c of atom a += v.
__device__ __forceinline__ void hb_add(const HbArgs &A, HbTable &T, int slot, int a, int c, double v) {
  if (slot < 0 || !(fabs(v) < FIX_SPLIT)) {
    fix_add(A.flags, A.acc + 3 * (size_t)a + c, A.coff, v);
    return;
  }
  const long long d = llrint(v * HB_FIX);
  if (d != 0) atomicAdd(&T.sum[c][slot], (unsigned long long)d);
}

// One hydrogen-bond entry of a lane (k < 0: none).
struct HbEntry {
  int k, type, orig;
  double d, v[3];
};

// Two halves of a wave take an H atom each, of the H atoms among `per`
// consecutive atoms of the workgroup; the lanes take a half's entries, the
// next 32 of them requested ahead.  The chain of
// loads to a first triple (atom, list, entry, far entry) bounds a small pass
// and the atomics a large one (a wave per atom with an atomic per term took
// 28 us on 1,944 atoms, 13 of them without the atomics; 590 on 96,000).  Sums
// over the entries are kept for even and odd sets of 32 apart, which makes
// them the sums of a 64-lane butterfly.
constexpr int HB_G = 32;
constexpr int HB_ATOMS = 64;   // at most, of a workgroup
__global__ void __launch_bounds__(BT) k_hb(int n, int per, HbArgs A) {
  __shared__ HbTable T;
  __shared__ int list[HB_ATOMS], count;
  for (int q = threadIdx.x; q < HB_SLOTS; q += BT) {
    T.key[q] = -1;
    T.sum[0][q] = T.sum[1][q] = T.sum[2][q] = 0ull;
  }
  if (threadIdx.x < SWR_WAVE) {
    const int t = threadIdx.x, j = blockIdx.x * per + t;
    const bool in = t < per && j < n;
    const bool is_h = in && A.Hindex[j] >= 0;
    if (in && !is_h) A.part[j] = 0.0;
    const unsigned long long m = __ballot(is_h);
    if (is_h) list[ballot_rank(m)] = j;
    if (t == 0) count = __popcll(m);
  }
  __syncthreads();
  const DevParams *__restrict__ P = A.P;
  const int sl = threadIdx.x % HB_G, half = (threadIdx.x / HB_G) & 1;
  for (int it = threadIdx.x / HB_G; it < count; it += BT / HB_G) {
    const int j = list[it];
    const int H = A.Hindex[j], tj = A.atoms[j].type;
    const int b0 = A.bidx[j], b1 = A.bend[j];
    const int h0 = A.hidx[H], h1 = A.hend[H];
    auto load = [&](int pk) {
      HbEntry x;
      x.k = -1;
      if (pk < h1) {
        const swr_hbond_t hb = A.hbonds[pk];
        x.k = hb.nbr;
        x.type = A.atoms[hb.nbr].type;
        x.orig = A.atoms[hb.nbr].orig_id;
        x.d = hb.ptr->d;
#pragma unroll
        for (int c = 0; c < 3; c++) x.v[c] = hb.scl * hb.ptr->dvec[c];
        if (x.type < 0) x.k = -1;
      }
      return x;
    };
    const HbEntry first = load(h0 + sl);   // (requested together with the bonds)
    double e[2] = {0.0, 0.0}, f[3][2] = {};
    for (int p0 = b0; p0 < b1; p0 += HB_G) {
      // the acceptors among the atom's bonds
      const int pl = p0 + sl;
      bool acc = false;
      if (pl < b1) {
        const int ti = A.atoms[A.bonds[pl].nbr].type;
        acc = ti >= 0 && P->p_hbond[ti] == 2 && A.BO[pl] >= HB_THRESHOLD;
      }
      unsigned todo = (unsigned)(__ballot(acc) >> (HB_G * half));
      while (todo) {
        const int pi = p0 + __ffs((int)todo) - 1;
        todo &= todo - 1;
        const swr_bond_t bij = A.bonds[pi];
        const int i = bij.nbr;
        const int ti = A.atoms[i].type, oi = A.atoms[i].orig_id;
        const double BOij = A.BO[pi];
        double ce1[2] = {0.0, 0.0}, g[3][2] = {};
        HbEntry next = first;
        // set: even and odd sets of 32 entries in turn
        auto into = [](double (&acc)[2], int set, double v) {
          acc[0] += set ? 0.0 : v;
          acc[1] += set ? v : 0.0;
        };
        int set = 0;
#pragma unroll 1
        for (int pk = h0 + sl; pk - sl < h1; pk += HB_G, set ^= 1) {
          const HbEntry x = next;
          next = load(pk + HB_G);
          if (x.k < 0 || x.orig == oi) continue;
          const DevHb &hbp = P->hb[(ti * SWR_MAX_ELEM + tj) * SWR_MAX_ELEM + x.type];
          if (hbp.r0_hb <= 0.0) continue;
          HbTriple t;
          hb_triple(hbp, BOij, bij.dvec, bij.d, x.v, x.d, t);
          into(e, set, t.e);
          into(ce1, set, t.ce1);
          const int slot = hb_slot(T, x.k);
#pragma unroll
          for (int c = 0; c < 3; c++) {
            into(f[c], set, t.ce2 * t.dj[c] - t.ce3 / x.d * x.v[c]);
            into(g[c], set, t.ce2 * t.di[c]);
            hb_add(A, T, slot, x.k, c, t.ce2 * t.dk[c] + t.ce3 / x.d * x.v[c]);
          }
        }
        const double c1 = group_sum<HB_G>(ce1[0] + ce1[1]);
        const double g0 = group_sum<HB_G>(g[0][0] + g[0][1]), g1 = group_sum<HB_G>(g[1][0] + g[1][1]),
                     g2 = group_sum<HB_G>(g[2][0] + g[2][1]);
        if (sl < 3) hb_add(A, T, hb_slot(T, i), i, sl, sl == 0 ? g0 : sl == 1 ? g1 : g2);
        if (sl == 0) A.Cdbo[pi] += c1;
      }
    }
    const double es = group_sum<HB_G>(e[0] + e[1]);
    const double f0 = group_sum<HB_G>(f[0][0] + f[0][1]), f1 = group_sum<HB_G>(f[1][0] + f[1][1]),
                 f2 = group_sum<HB_G>(f[2][0] + f[2][1]);
    if (sl == 0) A.part[j] = es;
    if (sl < 3) A.fcd[4 * (size_t)j + sl] += sl == 0 ? f0 : sl == 1 ? f1 : f2;
  }
  __syncthreads();
  for (int q = threadIdx.x; q < HB_SLOTS; q += BT) {
    const int a = T.key[q];
    if (a < 0) continue;
    long long d[3];
    unsigned long long old[3] = {0ull, 0ull, 0ull};
#pragma unroll
    for (int c = 0; c < 3; c++) {
      d[c] = (long long)T.sum[c][q];
      if (d[c] != 0) old[c] = atomicAdd(A.acc + 3 * (size_t)a + c, (unsigned long long)d[c]);
    }
    bool wrap = false;
#pragma unroll
    for (int c = 0; c < 3; c++) wrap |= fix_wrapped(old[c], d[c]);
    if (wrap) atomicOr(A.flags, SWR_F_FIXED_RANGE);
  }
}

// fCdDelta += the fixed-point terms; the accumulators are left at zero.  The
// first workgroup sums the energies.
__global__ void __launch_bounds__(BT) k_hb_fold(int n, int N, unsigned long long *__restrict__ acc,
                                                double *__restrict__ fcd, const double *__restrict__ part,
                                                double *__restrict__ sum) {
  if (blockIdx.x == 0) {
    sum_row<16>(n, part, sum);
    return;
  }
  const int a = (blockIdx.x - 1) * BT + threadIdx.x;
  if (a >= N) return;
  const size_t coff = 3 * (size_t)N;
#pragma unroll
  for (int c = 0; c < 3; c++) {
    unsigned long long *w = acc + 3 * (size_t)a + c;
    if (w[0] != 0ull || w[coff] != 0ull) {
      fcd[4 * (size_t)a + c] += fix_value(w, coff);
      w[0] = 0ull;
      w[coff] = 0ull;
    }
  }
}

// ---------------------------------------------------------------- valence angles
// The valence part of Merge_Torsion_Valence_Angles (host form
// reaxc_torsion_angles_sw64.c:812-1117): for every local atom j and pair of
// its bonds j-k (pk) and j-h (ph > pk) with BO above thb_cut and their
// product above thb_cutsq, and every parameter set of (type k, type j,
// type h) with |p_val1| > 0.001: the angle, penalty and coalition energies;
// their coefficients into Cdbo of both bonds and of all of j's bonds
// (CEval6 BO^7), Cdbopi/Cdbopi2 of j's bonds (CEval5), CdDelta of j, k and
// h, and the angle derivative into fCdDelta[.][0..2] of k, j and h.  A group
// of lanes per j writes j's own bond slots and row; the terms of k and h go
// into 64-bit fixed-point accumulators by integer atomics (order-independent
// sums), folded into fCdDelta by k_va_fold.  The centres with angles are
// listed by angle count (k_va_count, k_va_scatter: a centre with
// ten bonds has 45 pairs, one with two bonds one) and the groups take them
// largest first.
constexpr double DEG2RAD_PI = 3.14159265;   // constPI, reaxc_defs_sunway.h:61 (DEG2RAD :55)

// ---------------------------------------------------------------- work lists
// The valence and torsion passes work on items (a centre atom, a central
// bond) of which most have little or no work while a few have dozens of
// angles: items are counted first, bucketed by count and handed out largest
// first, each to a group of as many lanes as it has evaluations.
// Counters: the list length, a histogram of the counts, each bucket's next
// free position and where each group size ends.  Which lane takes which item changes no result: every
// item writes only its own entries and adds into the others through
// fixed-point integer atomics.
constexpr int WL_NB = 128;    // count buckets; counts of WL_NB - 1 and more share the last
enum { WL_NTASK = 0, WL_HIST = 1, WL_CUR = WL_HIST + WL_NB, WL_ABOVE = WL_CUR + WL_NB, WL_CTL_INTS = WL_ABOVE + 6 };
constexpr int WL_NABOVE = 6;   // ctl[WL_ABOVE + q]: items with counts above 32 >> q
__device__ __forceinline__ int wl_bucket(int c) { return c < WL_NB - 1 ? c : WL_NB - 1; }

// Bucket starts, largest count first, into start[0, WL_NB) (every workgroup of
// a scatter pass computes them from the finished histogram); the first
// workgroup also stores what the pass over the list reads.
__device__ __forceinline__ void wl_starts(int *__restrict__ ctl, int *start) {
  if (threadIdx.x < SWR_WAVE) {
    const int l = threadIdx.x;
    // lane l holds buckets b1 = WL_NB - 1 - 2 l and b1 - 1
    const int b1 = WL_NB - 1 - 2 * l;
    const int h1 = ctl[WL_HIST + b1], h0 = ctl[WL_HIST + b1 - 1];
    int incl = h1 + h0;
#pragma unroll
    for (int o = 1; o < SWR_WAVE; o <<= 1) {
      const int up = __shfl_up(incl, o, SWR_WAVE);
      if (l >= o) incl += up;
    }
    start[b1] = incl - h1 - h0;
    start[b1 - 1] = incl - h0;
    if (blockIdx.x == 0 && l == SWR_WAVE - 1) ctl[WL_NTASK] = incl;
  }
  __syncthreads();
  // items with counts above 32, 16, .., 1: where each group size ends
  if (blockIdx.x == 0 && threadIdx.x < WL_NABOVE) ctl[WL_ABOVE + threadIdx.x] = start[SWR_WAVE >> (threadIdx.x + 1)];
}
static_assert(WL_NB == 2 * SWR_WAVE, "a lane of wl_starts holds two buckets");

// Histogram and bucket cursors back to zero, once the list is made.
__device__ __forceinline__ void wl_clear(int *__restrict__ ctl) {
  for (int b = threadIdx.x; b < 2 * WL_NB; b += BT) ctl[WL_HIST + b] = 0;
}
static_assert(WL_CUR == WL_HIST + WL_NB, "wl_clear clears both at once");

// The waves of a listed pass.  An item of count c gets a group of G lanes, the
// power of two at or above c (at most 64), so one round of the group evaluates
// the whole item; items sit in the list in falling count, so the groups of
// each size are consecutive and a wave holds 64 / G groups of one size.  A
// group has at least gmin lanes: finding an item's evaluations among the pairs
// of its bonds is spread over the group too, which is what a short list (few
// waves, each waiting for its own chain of loads) needs, while a long list
// fills the chip with narrow groups and would only evaluate with fewer lanes.
struct WlWave {
  int G;        // lanes per group
  int t;        // this lane's item (live: inside the list)
  int sub;      // lane within the group
  bool live;
};

__device__ __forceinline__ bool wl_wave(const int *__restrict__ ctl, int unit, int gmin, WlWave &w) {
  const int lane = lane_id();
  int first = 0;   // items of wider groups
#pragma unroll
  for (int q = 0; q <= WL_NABOVE; ++q) {
    const int G = SWR_WAVE >> q;
    const bool last = G <= gmin;
    const int end = last || q == WL_NABOVE ? ctl[WL_NTASK] : ctl[WL_ABOVE + q];
    const int waves = (end - first + (1 << q) - 1) >> q;
    if (unit < waves) {
      w.G = G;
      w.t = first + (unit << q) + lane / G;
      w.sub = lane % G;
      w.live = w.t < end;
      return true;
    }
    if (last) return false;
    unit -= waves;
    first = end;
  }
  return false;
}

// Orders a wave's own LDS accesses (each wave has its own slice).
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Running totals of each group, NC components: after a round every lane of the
// group adds its share of the components over the round's evaluations in their
// order, so a total is the sum one thread would have made in a loop over them
// (the trajectory of a run depends on these sums to the last bit, and the
// solve of the charges turns a last bit into 1e-8).
template <int NC>
struct GroupTotals {
  double t[NC][SWR_WAVE];   // [component][the group's first lane]
};
template <int NC>
__device__ __forceinline__ void totals_init(GroupTotals<NC> &T, const WlWave &w) {
  for (int c = w.sub; c < NC; c += w.G) T.t[c][lane_id() - w.sub] = 0.0;
}

// Each group's pending evaluations: (a, b) positions in two bond ranges as
// a << 8 | b, in pair order, at most 2 G - 1 of them.
struct PairQueue {
  unsigned short *q;   // the group's slice (2 G entries) of the wave's LDS
  int n;               // pending
  int r, a, b;         // this lane's next raw pair r = a * mb + b
  int da, db;          // G / mb, G % mb
};

// Tests raw pairs (a < ma, b < mb), G at a time, until every group of the
// wave has G pending or no pairs left; test(a, b) says whether one is an
// evaluation.  The order of the pending ones is the raw order.
template <class Test>
__device__ __forceinline__ void queue_fill(PairQueue &Q, const WlWave &w, int ma, int mb, Test test) {
  const int lane = lane_id(), g0 = lane - w.sub;
  const unsigned long long gm = w.G == SWR_WAVE ? ~0ull : ((1ull << w.G) - 1ull);
  const unsigned long long below = (1ull << w.sub) - 1ull;
  const int R = w.live ? ma * mb : 0;
  while (true) {
    const bool more = Q.n < w.G && Q.r - w.sub < R;   // the same on the group's lanes
    if (!__any(more)) break;
    bool pass = false;
    const int code = Q.a << 8 | Q.b;
    if (more) {
      if (Q.r < R) pass = test(Q.a, Q.b);
      Q.r += w.G;
      Q.a += Q.da;
      Q.b += Q.db;
      if (Q.b >= mb) { Q.b -= mb; Q.a += 1; }
    }
    const unsigned long long m = (__ballot(pass) >> g0) & gm;
    if (pass) Q.q[Q.n + __popcll(m & below)] = (unsigned short)code;
    Q.n += __popcll(m);
  }
  wave_lds_order();
}

// After a round took the first `took` pending pairs.
__device__ __forceinline__ void queue_drop(PairQueue &Q, const WlWave &w, int took) {
  const int rem = Q.n - took;   // at most G - 1
  const unsigned short v = w.sub < rem ? Q.q[took + w.sub] : (unsigned short)0;
  wave_lds_order();
  if (w.sub < rem) Q.q[w.sub] = v;
  Q.n = rem;
  wave_lds_order();
}

__device__ __forceinline__ void queue_init(PairQueue &Q, const WlWave &w, unsigned short *wave_lds, int mb) {
  const int m = mb > 0 ? mb : 1;
  Q.q = wave_lds + 2 * (lane_id() - w.sub);
  Q.n = 0;
  Q.r = w.sub;
  Q.a = w.sub / m;
  Q.b = w.sub - Q.a * m;
  Q.da = w.G / m;
  Q.db = w.G - Q.da * m;
}

// Workgroup histogram of counts c (> 0 adds) into the global one.
__device__ __forceinline__ void wl_hist_flush(int *hist, int *__restrict__ ctl) {
  __syncthreads();
  for (int b = threadIdx.x; b < WL_NB; b += BT)
    if (hist[b]) atomicAdd(&ctl[WL_HIST + b], hist[b]);
}

struct VaArgs {
  unsigned int *flags;   // DevStatus::flags
  const DevParams *P;
  const swr_atom_pack_t *atoms;
  const int *bidx, *bend;
  const swr_bond_t *bonds;
  const double *BO, *BOpi, *bo_dboc;
  const double *Delta, *Delta_val, *vlpex, *nlp, *dDelta_lp;
  double *Cdbo, *Cdbopi, *Cdbopi2, *fcd, *part;
  size_t stride;
  unsigned long long *acc;   // [2][N][4] (fine, then coarse words)
  size_t coff;               // 4N
  int *cnt;                  // [n] angle count, then rank | bucket
  int *order;                // [n] centres with angles, largest count first
  int *ctl;                  // WL_CTL_INTS counters
};

// Angle evaluations of local centre j (slots [b0, b1), type tj >= 0) whose
// first bond is in slot pk: the pairs that pass the body's filters, times
// their parameter sets.
__device__ __forceinline__ int va_count(const VaArgs &A, int tj, int pk, int b1) {
  const DevParams *__restrict__ P = A.P;
  const double thb_cut = P->thb_cut, thb_cutsq = P->thb_cutsq;
  const double BO_jk = A.BO[pk];
  const int k = A.bonds[pk].nbr;
  const int tk = A.atoms[k].type;
  if (!(BO_jk > thb_cut) || A.bend[k] <= A.bidx[k] || tk < 0) return 0;
  int c = 0;
#pragma unroll 4
  for (int ph = pk + 1; ph < b1; ++ph) {
    const double BO_hj = A.BO[ph];
    const int th = A.atoms[A.bonds[ph].nbr].type;
    if (!(BO_hj > thb_cut) || !(BO_jk * BO_hj > thb_cutsq) || th < 0) continue;
    c += P->thb_n[(tk * SWR_MAX_ELEM + tj) * SWR_MAX_ELEM + th];
  }
  return c;
}

// BG lanes per local atom: its count and the histogram; a centre without
// angles gets its zero energy rows here (the valence kernel skips it).
__global__ void __launch_bounds__(BT) k_va_count(int n, VaArgs A) {
  __shared__ int hist[WL_NB];
  for (int b = threadIdx.x; b < WL_NB; b += BT) hist[b] = 0;
  __syncthreads();
  const int tid = blockIdx.x * BT + threadIdx.x;
  const int j = tid / BG, sl = tid % BG;
  const int tj = j < n ? A.atoms[j].type : -1;
  const int b0 = tj >= 0 ? A.bidx[j] : 0, b1 = tj >= 0 ? A.bend[j] : 0;
  int c = 0;
  for (int pk = b0 + sl; pk < b1; pk += BG) c += va_count(A, tj, pk, b1);
#pragma unroll
  for (int o = 1; o < BG; o <<= 1) c += __shfl_xor(c, o, SWR_WAVE);
  if (j < n) {
    if (sl == 0) {
      A.cnt[j] = c;
      if (c > 0) atomicAdd(&hist[wl_bucket(c)], 1);
    } else if (c == 0) {
      A.part[(sl - 1) * A.stride + j] = 0.0;
    }
  }
  wl_hist_flush(hist, A.ctl);
}
static_assert(BG == 4, "a lane of k_va_count clears one energy row");

__global__ void __launch_bounds__(BT) k_va_scatter(int n, VaArgs A) {
  __shared__ int cnt[WL_NB], base[WL_NB], start[WL_NB];
  for (int b = threadIdx.x; b < WL_NB; b += BT) cnt[b] = 0;
  wl_starts(A.ctl, start);
  const int j = blockIdx.x * BT + threadIdx.x;
  int b = -1, r = 0;
  if (j < n && A.cnt[j] > 0) {
    b = wl_bucket(A.cnt[j]);
    r = atomicAdd(&cnt[b], 1);
  }
  __syncthreads();
  for (int q = threadIdx.x; q < WL_NB; q += BT) base[q] = cnt[q] ? start[q] + atomicAdd(&A.ctl[WL_CUR + q], cnt[q]) : 0;
  __syncthreads();
  if (b >= 0) A.order[base[b] + r] = j;
}

// Waves of one-wave workgroups a listed pass starts at most; each wave takes
// its next set of groups that many on (the first ones hold the largest items).
constexpr int WL_MAX_WAVES = 4096;
// Shortest group, by the items of the list: with few of them the pass is bound
// by each item's chain of loads and transcendentals, not by lanes.  Whole passes
// (us) with 16, 4 and 1 lanes at least; one rule for both (angles cross at about
// 9,000 and 78,000 items, torsions at 5,000 and 120,000):
//   valence, water      3,900 items  34  38  49     10,200  60  52  66    36,000 108  72  74
//                      60,000       167 111 122     78,000 209 132 132    96,000 250 149 146
//   valence, clusters   2,600        45  54  76     12,100  80  84 115    62,700 241 196 210
//   torsion, water      3,100        50  54  73      7,200  72  62  81    59,900 321 273 285
//   torsion, clusters   3,600        63  76 127      8,900  97  94 141   127,600 611 477 475
__device__ __forceinline__ int wl_gmin(int ntask) { return ntask <= 4096 ? 16 : ntask <= 65536 ? 4 : 1; }

// One group of lanes per listed centre j (largest angle count first): the
// group's lanes test j's bond pairs and each evaluates one passing pair a
// round.  What bounds the pass is the latency of one pair's transcendentals
// (at 1-2 waves a SIMD), so a centre's pairs side by side instead of in turn
// take the longest centre off the critical path.  Per round the pairs' terms
// go to LDS and each slot and total is summed by one lane in pair order.  One
// thread per centre took 52 us on a 64-water box, 150 us on the 32,000-water one
// and 1.05 ms on 512 clusters; this takes 17 us, 94 us and 0.80 ms.
//
// SETS: parameter sets per angle type that the round's terms have room for; two
// (15 KB instead of 29) let eight waves a CU be resident, and the registers are
// held to that (eight spilled): 512 clusters 1138 -> 804 us, 96,000 water atoms
// 117 -> 92, 1,944 19 either way.
template <int SETS>
__global__ void __launch_bounds__(SWR_WAVE) __attribute__((amdgpu_waves_per_eu(2))) k_valence(VaArgs A) {
  __shared__ unsigned short queue[2 * SWR_WAVE];
  // the round's pairs: Cdbo terms, and per parameter set the centre's terms
  enum { V_ANG = 0, V_PEN, V_COA, V_CE5, V_CE6, V_CDJ, V_G0, V_G1, V_G2, V_NC };
  __shared__ double spk[SWR_WAVE], sph[SWR_WAVE], term[V_NC][SETS][SWR_WAVE];
  __shared__ int sset[SWR_WAVE];
  __shared__ GroupTotals<V_NC> T;
  const int lane = lane_id();
  const int gmin = wl_gmin(A.ctl[WL_NTASK]);
  WlWave w;
  for (int unit = blockIdx.x; wl_wave(A.ctl, unit, gmin, w); unit += gridDim.x) {
    const int j = w.live ? A.order[w.t] : 0;
    const int G = w.G, g0 = lane - w.sub;
    const DevParams *__restrict__ P = A.P;
    const int tj = w.live ? A.atoms[j].type : 0;
    const int b0 = w.live ? A.bidx[j] : 0, b1 = w.live ? A.bend[j] : 0;
    const int m = b1 - b0;
    totals_init(T, w);
    const double thb_cut = P->thb_cut, thb_cutsq = P->thb_cutsq;
    const double Dboc_j = A.bo_dboc[2 * (size_t)j + 1];
    const double p_val3 = P->p_val3[tj], p_val5 = P->p_val5[tj];
    const double p_val6 = P->p_val6, p_val8 = P->p_val8, p_val9 = P->p_val9, p_val10 = P->p_val10;
    // SBO: the group's lanes take a bond each for the exponentials
    double SBOp = 0.0, prod_SBO = 1.0;
    for (int t0 = b0; __any(t0 < b1); t0 += G) {
      const int t = t0 + w.sub;
      double b2 = t < b1 ? A.BO[t] * A.BO[t] : 0.0;
      b2 *= b2;
      b2 *= b2;
      spk[lane] = t < b1 ? A.BOpi[2 * (size_t)t] + A.BOpi[2 * (size_t)t + 1] : 0.0;
      sph[lane] = exp(-b2);
      wave_lds_order();
      for (int e = 0; e < G && t0 + e < b1; ++e) {
        SBOp += spk[g0 + e];
        prod_SBO *= sph[g0 + e];
      }
      wave_lds_order();
    }
    double vlpadj, dSBO2;
    if (A.vlpex[j] >= 0) {
      vlpadj = 0.0;
      dSBO2 = prod_SBO - 1.0;
    } else {
      vlpadj = A.nlp[j];
      dSBO2 = (prod_SBO - 1.0) * (1.0 - p_val8 * A.dDelta_lp[j]);
    }
    const double SBO = SBOp + (1.0 - prod_SBO) * (-Dboc_j - p_val8 * vlpadj);
    const double dSBO1 = -8.0 * prod_SBO * (Dboc_j + p_val8 * vlpadj);
    double SBO2, CSBO2;
    if (SBO <= 0.0) {
      SBO2 = 0.0; CSBO2 = 0.0;
    } else if (SBO <= 1.0) {
      SBO2 = pow(SBO, p_val9); CSBO2 = p_val9 * pow(SBO, p_val9 - 1.0);
    } else if (SBO < 2.0) {
      SBO2 = 2.0 - pow(2.0 - SBO, p_val9); CSBO2 = p_val9 * pow(2.0 - SBO, p_val9 - 1.0);
    } else {
      SBO2 = 2.0; CSBO2 = 0.0;
    }
    const double expval6 = exp(p_val6 * Dboc_j);
    const double exp10 = exp(-p_val10 * (2.0 - SBO2));   // theta_0 and Ctheta_0 of every set
    const double Delta_j = A.Delta[j];
    const double exp_pen3 = exp(-P->p_pen3 * Delta_j), exp_pen4 = exp(P->p_pen4 * Delta_j);
    const double trm_pen34 = 1.0 + exp_pen3 + exp_pen4;
    const double f9_Dj = (2.0 + exp_pen3) / trm_pen34;
    const double Cf9j = (-P->p_pen3 * exp_pen3 * trm_pen34 - (2.0 + exp_pen3) * (-P->p_pen3 * exp_pen3 + P->p_pen4 * exp_pen4)) /
                        (trm_pen34 * trm_pen34);
    const double exp_coa2 = exp(P->p_coa2 * A.Delta_val[j]);
    PairQueue Q;
    queue_init(Q, w, queue, m);
    while (true) {
      queue_fill(Q, w, m, m, [&](int a, int b) {
        if (b <= a) return false;
        const double BO_jk = A.BO[b0 + a], BO_hj = A.BO[b0 + b];
        const int k = A.bonds[b0 + a].nbr, h = A.bonds[b0 + b].nbr;
        const int tk = A.atoms[k].type, th = A.atoms[h].type;
        if (!(BO_jk > thb_cut) || !(BO_hj > thb_cut) || !(BO_jk * BO_hj > thb_cutsq)) return false;
        if (tk < 0 || th < 0 || A.bend[k] <= A.bidx[k]) return false;
        return P->thb_n[(tk * SWR_MAX_ELEM + tj) * SWR_MAX_ELEM + th] != 0;
      });
      const int take = min(Q.n, G);
      if (!__any(take > 0)) break;
      const bool ev = w.sub < take;
      double cdbo_jk = 0.0, cdbo_hj = 0.0;
      int nset = 0;
      if (ev) {
        const int code = Q.q[w.sub];
        const int pk = b0 + (code >> 8), ph = b0 + (code & 255);
        const double BO_jk = A.BO[pk], BO_hj = A.BO[ph];
        const swr_bond_t bjk = A.bonds[pk], bhj = A.bonds[ph];
        const int k = bjk.nbr, h = bhj.nbr;
        const int tk = A.atoms[k].type, th = A.atoms[h].type;
        const double BOA_jk = BO_jk - thb_cut, BOA_hj = BO_hj - thb_cut;
        const int tri = (tk * SWR_MAX_ELEM + tj) * SWR_MAX_ELEM + th;
        nset = P->thb_n[tri];
        // Calculate_Theta / Calculate_dCos_Theta (:1510-1547) with the j-k
        // bond first: di belongs to k, dk to h
        const double dot = bjk.dvec[0] * bhj.dvec[0] + bjk.dvec[1] * bhj.dvec[1] + bjk.dvec[2] * bhj.dvec[2];
        double cos_t = dot / (bjk.d * bhj.d);
        if (cos_t > 1.0) cos_t = 1.0;
        if (cos_t < -1.0) cos_t = -1.0;
        const double theta = acos(cos_t);
        double sin_t = sin(theta);
        if (sin_t < 1.0e-5) sin_t = 1.0e-5;
        const double sq_jk = bjk.d * bjk.d, sq_hj = bhj.d * bhj.d;
        const double inv_d = 1.0 / (bjk.d * bhj.d);
        const double cinv3 = dot * (inv_d * inv_d * inv_d);
        const double bo_k0 = A.bo_dboc[2 * (size_t)k], bo_h0 = A.bo_dboc[2 * (size_t)h];
        // the penalty and coalition factors of the pair, the same for every
        // set; only evaluated when a set has p_pen1 or p_coa1 (a term with a
        // zero prefactor is zero either way)
        const bool need_pc = P->thb_pc[tri] != 0;
        const double pen2 = need_pc ? exp(-P->p_pen2 * (BOA_jk - 2.0) * (BOA_jk - 2.0)) *
                                          exp(-P->p_pen2 * (BOA_hj - 2.0) * (BOA_hj - 2.0))
                                    : 0.0;
        const double coa = need_pc ? 1.0 / (1. + exp_coa2) * exp(-P->p_coa3 * (bo_k0 - BOA_jk) * (bo_k0 - BOA_jk)) *
                                         exp(-P->p_coa3 * (bo_h0 - BOA_hj) * (bo_h0 - BOA_hj)) *
                                         exp(-P->p_coa4 * (BOA_jk - 1.5) * (BOA_jk - 1.5)) *
                                         exp(-P->p_coa4 * (BOA_hj - 1.5) * (BOA_hj - 1.5))
                                   : 0.0;
        double ck[4] = {0.0, 0.0, 0.0, 0.0}, chh[4] = {0.0, 0.0, 0.0, 0.0};
        for (int c = 0; c < nset; ++c) {
          const DevThb &q = P->thb[tri][c];
          const double p_val1 = q.p_val1, p_val2 = q.p_val2, p_val4 = q.p_val4, p_val7 = q.p_val7;
          const double pjk = pow(BOA_jk, p_val4 - 1.0), phj = pow(BOA_hj, p_val4 - 1.0);
          const double exp3jk = exp(-p_val3 * (pjk * BOA_jk));
          const double f7_jk = 1.0 - exp3jk;
          const double Cf7jk = p_val3 * p_val4 * pjk * exp3jk;
          const double exp3hj = exp(-p_val3 * (phj * BOA_hj));
          const double f7_hj = 1.0 - exp3hj;
          const double Cf7hj = p_val3 * p_val4 * phj * exp3hj;
          const double expval7 = exp(-p_val7 * Dboc_j);
          const double trm8 = 1.0 + expval6 + expval7;
          const double f8_Dj = p_val5 - ((p_val5 - 1.0) * (2.0 + expval6) / trm8);
          const double Cf8j = ((1.0 - p_val5) / (trm8 * trm8)) *
                              (p_val6 * expval6 * trm8 - (2.0 + expval6) * (p_val6 * expval6 - p_val7 * expval7));
          const double theta_0 = (180.0 - q.theta_00 * (1.0 - exp10)) * DEG2RAD_PI / 180.0;
          const double expval2theta = exp(-p_val2 * (theta_0 - theta) * (theta_0 - theta));
          const double expval12theta = p_val1 >= 0 ? p_val1 * (1.0 - expval2theta) : p_val1 * -expval2theta;
          const double CEval1 = Cf7jk * f7_hj * f8_Dj * expval12theta;
          const double CEval2 = Cf7hj * f7_jk * f8_Dj * expval12theta;
          const double CEval3 = Cf8j * f7_hj * f7_jk * expval12theta;
          const double CEval4 = -2.0 * p_val1 * p_val2 * f7_jk * f7_hj * f8_Dj * expval2theta * (theta_0 - theta);
          const double Ctheta_0 = p_val10 * (q.theta_00 * DEG2RAD_PI / 180.0) * exp10;
          const double CEval5 = -CEval4 * Ctheta_0 * CSBO2;
          const double CEval8 = -CEval4 / sin_t;
          term[V_ANG][c][lane] = f7_jk * f7_hj * f8_Dj * expval12theta;
          // penalty
          const double ep = q.p_pen1 * f9_Dj * pen2;
          term[V_PEN][c][lane] = ep;
          const double CEpen1 = ep * Cf9j / f9_Dj;
          const double tp = -2.0 * P->p_pen2 * ep;
          const double CEpen2 = tp * (BOA_jk - 2.0), CEpen3 = tp * (BOA_hj - 2.0);
          // coalition
          const double ec = q.p_coa1 * coa;
          term[V_COA][c][lane] = ec;
          const double CEcoa1 = -2 * P->p_coa4 * (BOA_jk - 1.5) * ec;
          const double CEcoa2 = -2 * P->p_coa4 * (BOA_hj - 1.5) * ec;
          const double CEcoa3 = -P->p_coa2 * exp_coa2 * ec / (1 + exp_coa2);
          const double CEcoa4 = -2 * P->p_coa3 * (bo_k0 - BOA_jk) * ec;
          const double CEcoa5 = -2 * P->p_coa3 * (bo_h0 - BOA_hj) * ec;
          cdbo_jk += CEval1 + CEpen2 + (CEcoa1 - CEcoa4);
          cdbo_hj += CEval2 + CEpen3 + (CEcoa2 - CEcoa5);
          term[V_CDJ][c][lane] = (CEval3 + CEval5 * dSBO2) + CEpen1 + CEcoa3;
          ck[3] += CEcoa4;
          chh[3] += CEcoa5;
          term[V_CE5][c][lane] = CEval5;
          term[V_CE6][c][lane] = CEval5 * dSBO1;
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            const double di = bhj.dvec[d] * inv_d - cinv3 * sq_hj * bjk.dvec[d];
            const double dj = -(bhj.dvec[d] + bjk.dvec[d]) * inv_d + cinv3 * (sq_hj * bjk.dvec[d] + sq_jk * bhj.dvec[d]);
            const double dk = bjk.dvec[d] * inv_d - cinv3 * sq_jk * bhj.dvec[d];
            ck[d] += CEval8 * di;
            chh[d] += CEval8 * dk;
            term[V_G0 + d][c][lane] = CEval8 * dj;
          }
        }
        unsigned long long *ak = A.acc + 4 * (size_t)k, *ah = A.acc + 4 * (size_t)h;
        {
          unsigned long long *const ga[8] = {ak, ak + 1, ak + 2, ak + 3, ah, ah + 1, ah + 2, ah + 3};
          const size_t gc[8] = {A.coff, A.coff, A.coff, A.coff, A.coff, A.coff, A.coff, A.coff};
          const double gv[8] = {ck[0], ck[1], ck[2], ck[3], chh[0], chh[1], chh[2], chh[3]};
          fix_add_group<8>(A.flags, ga, gc, gv);
        }
      }
      // the round's Cdbo terms onto j's slots, and its other terms onto the
      // centre's totals: each by one lane, in pair (and set) order
      spk[lane] = cdbo_jk;
      sph[lane] = cdbo_hj;
      sset[lane] = nset;
      wave_lds_order();
      for (int t0 = 0; t0 < m; t0 += G) {
        const int t = t0 + w.sub;
        double v = 0.0;
        bool touched = false;
        for (int e = 0; e < take; ++e) {
          const int code = Q.q[e];
          const bool k = (code >> 8) == t;
          if (k || (code & 255) == t) {
            if (!touched) v = A.Cdbo[b0 + t];
            touched = true;
            v += k ? spk[g0 + e] : sph[g0 + e];
          }
        }
        if (touched) A.Cdbo[b0 + t] = v;
      }
      for (int c = w.sub; c < V_NC; c += G) {
        double v = T.t[c][g0];
        for (int e = 0; e < take; ++e)
          for (int q = 0; q < sset[g0 + e]; ++q) v += term[c][q][g0 + e];
        T.t[c][g0] = v;
      }
      wave_lds_order();
      queue_drop(Q, w, take);
    }
    wave_lds_order();
    const double ce5 = T.t[V_CE5][g0], ce6 = T.t[V_CE6][g0];
    if (ce5 != 0.0 || ce6 != 0.0)
      for (int t = b0 + w.sub; t < b1; t += G) {
        const double bo = A.BO[t];
        const double bo3 = bo * bo * bo;
        A.Cdbo[t] += ce6 * (bo3 * bo3 * bo);
        A.Cdbopi[t] += ce5;
        A.Cdbopi2[t] += ce5;
      }
    if (w.live && w.sub == 0) {
#pragma unroll
      for (int d = 0; d < 3; ++d) A.fcd[4 * (size_t)j + d] += T.t[V_G0 + d][g0];
      A.fcd[4 * (size_t)j + 3] += T.t[V_CDJ][g0];
      A.part[j] = T.t[V_ANG][g0];
      A.part[A.stride + j] = T.t[V_PEN][g0];
      A.part[2 * A.stride + j] = T.t[V_COA][g0];
    }
    wave_lds_order();   // (before the next groups' totals start)
  }
}

// fCdDelta's row a (f, in registers) += the fixed-point terms; the accumulators
// are left at zero.  Whether there were any.
__device__ __forceinline__ bool fold4(int N, int a, unsigned long long *__restrict__ acc, double *f) {
  const size_t coff = 4 * (size_t)N;
  unsigned long long fine[4], coarse[4];
  unsigned long long *w = acc + 4 * (size_t)a;
#pragma unroll
  for (int c = 0; c < 4; c++) {
    fine[c] = w[c];
    coarse[c] = w[coff + c];
  }
  bool any = false;
#pragma unroll
  for (int c = 0; c < 4; c++) {
    if (fine[c] == 0ull && coarse[c] == 0ull) continue;
    const unsigned long long pair[2] = {fine[c], coarse[c]};
    f[c] += fix_value(pair, 1);
    w[c] = 0ull;
    w[coff + c] = 0ull;
    any = true;
  }
  return any;
}

// The end of the valence pass: the first three workgroups sum the energy rows,
// the next clears the work list's counters, the others fold the terms of k
// and h into fCdDelta.
__global__ void __launch_bounds__(BT) k_va_fold(int n, int N, VaArgs A, double *__restrict__ sums) {
  if (blockIdx.x < 3) {
    sum_row<16>(n, A.part + blockIdx.x * A.stride, sums + blockIdx.x);
    return;
  }
  if (blockIdx.x == 3) {
    wl_clear(A.ctl);
    return;
  }
  const int a = (blockIdx.x - 4) * BT + threadIdx.x;
  if (a >= N) return;
  double *fcd = A.fcd + 4 * (size_t)a;
  double f[4] = {fcd[0], fcd[1], fcd[2], fcd[3]};
  if (fold4(N, a, A.acc, f))
#pragma unroll
    for (int c = 0; c < 4; c++) fcd[c] = f[c];
}

// ---------------------------------------------------------------- torsions
// The torsion part of Merge_Torsion_Valence_Angles (host form
// reaxc_torsion_angles_sw64.c:812-1408; Calculate_Omega :21-104).  The work
// is one task per central bond j-k of a local atom j (taken once per
// physical bond: orig_id order, then position for images of one atom): over
// the other bonds j-i of j and the bonds k-l of k, the torsion and
// conjugation energies.  Most bonds make no torsion and a few make dozens,
// so the tasks are listed with their exact quadruple counts and handed to
// lanes in decreasing count (a wave's lanes then do about the same work):
//
//   k_to_count    sixteen lanes per local atom: per bond slot the number of
//                 quadruples the torsion body evaluates (the same filters),
//                 a histogram of the counts;
//   k_to_scatter  one thread per local atom: its central bonds with work
//                 into the list, largest counts first (the order inside a
//                 bucket is arbitrary and changes no result);
//   k_torsion     a group of lanes per listed central bond, one quadruple a
//                 lane: the slot's Cdbopi and Cdbo written directly, j's row terms and energies into
//                 the slot's row entry, Cdbo of j-i and k-l and the terms of
//                 i, k, l into 64-bit fixed-point accumulators by integer
//                 atomics;
//   k_to_fold     one thread per atom: its slots' row entries summed in slot
//                 order into its row and energies, and the accumulators
//                 folded into its row and its slots' Cdbo.
struct ToArgs {
  unsigned int *flags;   // DevStatus::flags
  const DevParams *P;
  const swr_atom_pack_t *atoms;
  const int *bidx, *bend;
  const swr_bond_t *bonds;
  const double *BO, *BOpi, *bo_dboc;
  double *Cdbo, *Cdbopi, *fcd, *part;
  size_t stride;
  unsigned long long *acc;    // [2][N][4] (fine, then coarse words)
  unsigned long long *sacc;   // [2][bond slots]
  size_t coff, scoff;         // 4N, bond slots
  const int *bnbr;            // bonds[].nbr, compact
  int *tc;                    // [bond slots] quadruple count, then rank | bucket
  int2 *task;                 // [bond slots] (j, slot) of the listed central bonds
  int *ctl;                   // WL_CTL_INTS counters
  double *row;                // [bond slots][6] j's row terms and energies per central bond
};


// Calculate_Theta of bonds a (first) and b from one centre; dot: their dot
// product.
__device__ __forceinline__ double theta_of(const swr_bond_t &a, const swr_bond_t &b, double &dot) {
  dot = a.dvec[0] * b.dvec[0] + a.dvec[1] * b.dvec[1] + a.dvec[2] * b.dvec[2];
  double c = dot / (a.d * b.d);
  if (c > 1.0) c = 1.0;
  if (c < -1.0) c = -1.0;
  return acos(c);
}

// Calculate_dCos_Theta of the same: component q of di (a's far atom), dj (the
// centre) and dk (b's far atom).  Apart from the angle, so that the nine
// numbers are not held in registers through the energies between.
struct DCos {
  double inv, ci3, sa, sb;
  __device__ __forceinline__ DCos(const swr_bond_t &a, const swr_bond_t &b, double dot) {
    inv = 1.0 / (a.d * b.d);
    ci3 = dot * (inv * inv * inv);
    sa = a.d * a.d;
    sb = b.d * b.d;
  }
  __device__ __forceinline__ void get(const swr_bond_t &a, const swr_bond_t &b, int q, double &di, double &dj,
                                      double &dk) const {
    di = b.dvec[q] * inv - ci3 * sb * a.dvec[q];
    dj = -(b.dvec[q] + a.dvec[q]) * inv + ci3 * (sb * a.dvec[q] + sa * b.dvec[q]);
    dk = a.dvec[q] * inv - ci3 * sa * b.dvec[q];
  }
};

__device__ __forceinline__ double tan_inv(double s, double c) {
  constexpr double MIN_SINE = 1e-10;   // reaxc_torsion_angles_sw64.c:12
  if (s >= 0 && s <= MIN_SINE) return c / MIN_SINE;
  if (s <= 0 && s >= -MIN_SINE) return c / -MIN_SINE;
  return c / s;
}

// Whether bonds ph (j-i) and pw (k-l) make a torsion with the central bond pk
// (j-k; pj its reverse slot).  All loads are unconditional, so that the tests
// of consecutive pairs overlap their latencies.
__device__ __forceinline__ bool to_pass(const ToArgs &A, int tj, int tk, double BO_jk, int pk, int pj, int ph, int pw,
                                        double thb_cut) {
  const double BO_ij = A.BO[ph], BO_kl = A.BO[pw];
  const int i = A.bnbr[ph], l = A.bnbr[pw];
  const int ti = A.atoms[i].type, tl = A.atoms[l].type;
  if (ph == pk || pw == pj || i == l || ti < 0 || tl < 0) return false;
  if (!(BO_ij > thb_cut) || !(BO_kl > thb_cut) || !(BO_ij * BO_jk * BO_kl > thb_cut)) return false;
  return A.P->tor[((ti * SWR_MAX_ELEM + tj) * SWR_MAX_ELEM + tk) * SWR_MAX_ELEM + tl].cnt != 0;
}

// Sixteen lanes per local atom.  They hold its bonds, a bond each, and find
// the central ones together; for each of those they hold k's bonds, and the
// atom's strong bonds go round by lane exchange, so the quadruples are tested
// without a load but the parameter table's.  (With each pair's bonds gathered
// again the pass waited for them: 10 us on 60 atoms, 80 on 96,000, 500 on 512
// clusters; with four lanes an atom 23 on 1,944.)
constexpr int TO_CNT_LANES = 16;
__global__ void __launch_bounds__(BT) k_to_count(int n, ToArgs A) {
  constexpr int L = TO_CNT_LANES;
  __shared__ int hist[WL_NB];
  for (int b = threadIdx.x; b < WL_NB; b += BT) hist[b] = 0;
  __syncthreads();
  const DevParams *__restrict__ P = A.P;
  const int tid = blockIdx.x * BT + threadIdx.x;
  const int j = tid / L, sl = tid % L, shift = lane_id() & ~(L - 1);
  const double thb_cut = P->thb_cut;
  auto group = [&](bool x) { return (unsigned)(__ballot(x) >> shift) & ((1u << L) - 1u); };
  swr_atom_pack_t aj = {};
  aj.type = -1;
  if (j < n) aj = A.atoms[j];
  const int tj = aj.type;
  const int b0 = j < n ? A.bidx[j] : 0, b1 = j < n ? A.bend[j] : 0;
  for (int c0 = b0; c0 < b1; c0 += L) {
    // this lane's bond as the central one: k, its bonds, the reverse slot
    const int pc = c0 + sl;
    const bool mine = pc < b1;
    double BO = 0.0;
    int k = 0, k0 = 0, k1 = 0, tk = -1, pj = 0;
    bool central = false;
    if (mine && tj >= 0) {
      BO = A.BO[pc];
      k = A.bnbr[pc];
      k0 = A.bidx[k];
      k1 = A.bend[k];
      const swr_atom_pack_t ak = A.atoms[k];
      tk = ak.type;
      pj = A.bonds[pc].sym_index;
      central = BO - thb_cut > 0.0 && k1 > k0 && tk >= 0 && owns_bond(aj, ak);
    }
    if (mine && !central) {
      A.tc[pc] = 0;
#pragma unroll
      for (int q = 0; q < 6; q++) A.row[6 * (size_t)pc + q] = 0.0;
    }
    for (unsigned todo = group(central); todo; todo &= todo - 1) {
      const int e = __ffs((int)todo) - 1, pk = c0 + e;
      const double BO_jk = __shfl(BO, e, L);
      const int w0 = __shfl(k0, e, L), w1 = __shfl(k1, e, L), tc = __shfl(tk, e, L), pr = __shfl(pj, e, L);
      int c = 0;
      for (int ww = w0; ww < w1; ww += L) {
        const int pw = ww + sl;
        double BO_kl = 0.0;
        int l = 0, tl = -1;
        if (pw < w1) {
          BO_kl = A.BO[pw];
          l = A.bnbr[pw];
          tl = A.atoms[l].type;
        }
        const bool far_end = pw < w1 && pw != pr && tl >= 0 && BO_kl > thb_cut;
        for (int h0 = b0; h0 < b1; h0 += L) {
          // the atom's bonds as j-i, a lane each (those of the outer round as they are)
          double BO_ij = BO;
          int i = k, ti = tk;
          if (h0 != c0) {
            const int ph = h0 + sl;
            BO_ij = ph < b1 ? A.BO[ph] : 0.0;
            i = ph < b1 ? A.bnbr[ph] : 0;
            ti = ph < b1 ? A.atoms[i].type : -1;
          }
          unsigned strong = group(ti >= 0 && BO_ij > thb_cut);
          if (h0 == c0) strong &= ~(1u << e);
          for (; strong; strong &= strong - 1) {
            const int q = __ffs((int)strong) - 1;
            const double bij = __shfl(BO_ij, q, L);
            const int ii = __shfl(i, q, L), t4 = __shfl(ti, q, L);
            if (far_end && ii != l && bij * BO_jk * BO_kl > thb_cut &&
                P->tor[((t4 * SWR_MAX_ELEM + tj) * SWR_MAX_ELEM + tc) * SWR_MAX_ELEM + tl].cnt != 0)
              c++;
          }
        }
      }
#pragma unroll
      for (int o = 1; o < L; o <<= 1) c += __shfl_xor(c, o, SWR_WAVE);
      if (c == 0 && sl < 6) A.row[6 * (size_t)pk + sl] = 0.0;
      if (sl == 0) {
        A.tc[pk] = c;
        if (c > 0) atomicAdd(&hist[wl_bucket(c)], 1);
      }
    }
  }
  wl_hist_flush(hist, A.ctl);
}

__global__ void __launch_bounds__(BT) k_to_scatter(int n, ToArgs A) {
  __shared__ int cnt[WL_NB], base[WL_NB], start[WL_NB];
  for (int b = threadIdx.x; b < WL_NB; b += BT) cnt[b] = 0;
  wl_starts(A.ctl, start);
  const int j = blockIdx.x * BT + threadIdx.x;
  const int b0 = j < n ? A.bidx[j] : 0, b1 = j < n ? A.bend[j] : 0;
  for (int pk = b0; pk < b1; ++pk) {   // rank in the workgroup's share of the bucket
    const int c = A.tc[pk];
    if (c > 0) {
      const int b = wl_bucket(c);
      A.tc[pk] = (atomicAdd(&cnt[b], 1) << 8) | b;
    }
  }
  __syncthreads();
  for (int b = threadIdx.x; b < WL_NB; b += BT) base[b] = cnt[b] ? start[b] + atomicAdd(&A.ctl[WL_CUR + b], cnt[b]) : 0;
  __syncthreads();
  for (int pk = b0; pk < b1; ++pk) {
    const int v = A.tc[pk];
    if (v > 0) A.task[base[v & 255] + (v >> 8)] = make_int2(j, pk);
  }
}

// One group of lanes per listed central bond (most quadruples first): the
// group's lanes test the pairs of j-i and k-l bonds and each evaluates one
// quadruple a round.  A quadruple is ~2000 dependent FP64 instructions at one
// wave per SIMD, so what bounded the pass was the longest bond's chain of
// quadruples.  i's terms are summed over the round's quadruples of one j-i
// bond (they are neighbours in the queue) before their fixed-point add, and
// j's, k's and the bond's over all, each by one lane in order, so the large
// cotangent terms of a nearly linear angle cancel in FP64 first.  One lane
// per bond took 87 us on a 64-water box, 133 us on the 32,000-water one and
// 2.38 ms on 512 clusters; this takes 15, 65 us and 1.02 ms.
//
// WAVES: waves per SIMD the registers are held to.  Two (ten of 266 spilled)
// pay once a list keeps every SIMD busy with quadruples (TORSION_TWO_WAVES).
// From this many atoms on.  The host knows the atoms, not the list's length, but
// the line is low enough for both kinds of system: the torsion pass with one and
// with two waves takes 75 and 77 us on 24,000 water atoms (6,600 bonds listed),
// 134 and 126 on 48,000 (24,700), 182 and 175 on 96,000, 1,294 and 1,263 on
// 768,000; on clusters of 23,000 atoms (30,700 bonds) 163 and 142, of 40,000 240
// and 205, of 319,000 1,598 and 1,330.  1,944 atoms: 17 and 19 (the kernel).
constexpr int TORSION_TWO_WAVES = 32768;
template <int WAVES>
__global__ void __launch_bounds__(SWR_WAVE) __attribute__((amdgpu_waves_per_eu(WAVES))) k_torsion(ToArgs A) {
  // the round's quadruples: the bond's and i's terms
  enum { O_FJ = 0, O_FK = 4, O_CDK = 7, O_PI, O_BO, O_TOR, O_CON, O_NC };
  __shared__ unsigned short queue[2 * SWR_WAVE];
  __shared__ double term[O_NC][SWR_WAVE], iterm[4][SWR_WAVE];
  __shared__ int sph[SWR_WAVE];
  __shared__ GroupTotals<O_NC> T;
  constexpr double MIN_SINE = 1e-10;
  const int lane = lane_id();
  const int gmin = wl_gmin(A.ctl[WL_NTASK]);
  const DevParams *__restrict__ P = A.P;
  WlWave w;
  for (int unit = blockIdx.x; wl_wave(A.ctl, unit, gmin, w); unit += gridDim.x) {
    const int2 jp = w.live ? A.task[w.t] : A.task[0];
    const int j = jp.x, pk = jp.y, G = w.G, g0 = lane - w.sub;
    totals_init(T, w);
    const int tj = A.atoms[j].type;
    const int b0 = A.bidx[j], b1 = A.bend[j];
    const double thb_cut = P->thb_cut;
    const double p_tor2 = P->p_tor2, p_tor3 = P->p_tor3, p_tor4 = P->p_tor4, p_cot2 = P->p_cot2;
    const double Delta_j = A.bo_dboc[2 * (size_t)j + 1];
    const double BO_jk = A.BO[pk];
    const swr_bond_t bjk = A.bonds[pk];
    const int k = bjk.nbr;
    const int k0 = A.bidx[k], k1 = A.bend[k];
    const int tk = A.atoms[k].type;
    const int pj = bjk.sym_index;
    const swr_bond_t bkj = A.bonds[pj];
    const double BOA_jk = BO_jk - thb_cut;
    const double Delta_k = A.bo_dboc[2 * (size_t)k + 1];
    const double r_jk = bjk.d;
    const double exp_tor2_jk = exp(-p_tor2 * BOA_jk);
    const double exp_cot2_jk = exp(-p_cot2 * (BOA_jk - 1.5) * (BOA_jk - 1.5));
    const double exp_tor3_DjDk = exp(-p_tor3 * (Delta_j + Delta_k));
    const double exp_tor4_DjDk = exp(p_tor4 * (Delta_j + Delta_k));
    const double exp_tor34_inv = 1.0 / (1.0 + exp_tor3_DjDk + exp_tor4_DjDk);
    const double f11_DjDk = (2.0 + exp_tor3_DjDk) * exp_tor34_inv;
    const double dfn11 = (-p_tor3 * exp_tor3_DjDk +
                          (p_tor3 * exp_tor3_DjDk - p_tor4 * exp_tor4_DjDk) * (2.0 + exp_tor3_DjDk) * exp_tor34_inv) *
                         exp_tor34_inv;
    const double BOpi_jk = A.BOpi[2 * (size_t)pk];
    PairQueue Q;
    queue_init(Q, w, queue, k1 - k0);
    while (true) {
      queue_fill(Q, w, b1 - b0, k1 - k0, [&](int a, int b) {
        return to_pass(A, tj, tk, BO_jk, pk, pj, b0 + a, k0 + b, thb_cut);
      });
      const int take = min(Q.n, G);
      if (!__any(take > 0)) break;
      const bool ev = w.sub < take;
      int ph = -1, i = 0;
      if (ev) {
        const int code = Q.q[w.sub];
        const int pw = k0 + (code & 255);
        ph = b0 + (code >> 8);
        const double BO_ij = A.BO[ph], BO_kl = A.BO[pw];
        const swr_bond_t bij = A.bonds[ph], bkl = A.bonds[pw];
        i = bij.nbr;
        const int l = bkl.nbr;
        const swr_atom_pack_t ai = A.atoms[i], al = A.atoms[l];
        const double xi[3] = {ai.x[0], ai.x[1], ai.x[2]};
        const DevTor &fb = P->tor[((ai.type * SWR_MAX_ELEM + tj) * SWR_MAX_ELEM + tk) * SWR_MAX_ELEM + al.type];
        const double r_ij = bij.d;
        const double BOA_ij = BO_ij - thb_cut;
        double dot_ijk, dot_jkl;
        const double theta_ijk = theta_of(bjk, bij, dot_ijk);
        const double sin_ijk = sin(theta_ijk);
        const double cos_ijk = cos(theta_ijk);
        const double tan_ijk_i = tan_inv(sin_ijk, cos_ijk);
        const double exp_tor2_ij = exp(-p_tor2 * BOA_ij);
        const double exp_cot2_ij = exp(-p_cot2 * (BOA_ij - 1.5) * (BOA_ij - 1.5));
        const double theta_jkl = theta_of(bkj, bkl, dot_jkl);
        const double r_kl = bkl.d;
        const double BOA_kl = BO_kl - thb_cut;
        double sin_jkl = sin(theta_jkl);
        const double cos_jkl = cos(theta_jkl);
        const double tan_jkl_i = tan_inv(sin_jkl, cos_jkl);
        const double dvec_li[3] = {xi[0] - al.x[0], xi[1] - al.x[1], xi[2] - al.x[2]};
        const double r_li = sqrt(dvec_li[0] * dvec_li[0] + dvec_li[1] * dvec_li[1] + dvec_li[2] * dvec_li[2]);
        // Calculate_Omega
        const double *dij = bij.dvec, *djk = bjk.dvec, *dkl = bkl.dvec;
        const double d_ij_jk = dij[0] * djk[0] + dij[1] * djk[1] + dij[2] * djk[2];
        const double d_jk_kl = djk[0] * dkl[0] + djk[1] * dkl[1] + djk[2] * dkl[2];
        const double d_ij_kl = dij[0] * dkl[0] + dij[1] * dkl[1] + dij[2] * dkl[2];
        const double cr[3] = {djk[1] * dkl[2] - djk[2] * dkl[1], djk[2] * dkl[0] - djk[0] * dkl[2],
                              djk[0] * dkl[1] - djk[1] * dkl[0]};
        const double uc = -d_ij_jk * d_jk_kl + r_jk * r_jk * d_ij_kl;
        const double us = -r_jk * (dij[0] * cr[0] + dij[1] * cr[1] + dij[2] * cr[2]);
        const double omega = atan2(us, uc);
        const double htra = r_ij + cos_ijk * (r_kl * cos_jkl - r_jk);
        const double htrb = r_jk - r_ij * cos_ijk - r_kl * cos_jkl;
        const double htrc = r_kl + cos_jkl * (r_ij * cos_ijk - r_jk);
        const double hthd = r_ij * sin_ijk * (r_jk - r_kl * cos_jkl);
        const double hthe = r_kl * sin_jkl * (r_jk - r_ij * cos_ijk);
        const double hnra = r_kl * sin_ijk * sin_jkl;
        const double hnrc = r_ij * sin_ijk * sin_jkl;
        const double hnhd = r_ij * r_kl * cos_ijk * sin_jkl;
        const double hnhe = r_ij * r_kl * sin_ijk * cos_jkl;
        double poem = 2.0 * r_ij * r_kl * sin_ijk * sin_jkl;
        if (poem < 1e-20) poem = 1e-20;
        const double tel = r_ij * r_ij + r_jk * r_jk + r_kl * r_kl - r_li * r_li -
                           2.0 * (r_ij * r_jk * cos_ijk - r_ij * r_kl * cos_ijk * cos_jkl + r_jk * r_kl * cos_jkl);
        double arg = tel / poem;
        if (arg > 1.0) arg = 1.0;
        if (arg < -1.0) arg = -1.0;
        double s_ijk = sin_ijk, s_jkl = sin_jkl;   // clamped copies for the divisions
        if (s_ijk >= 0 && s_ijk <= MIN_SINE) s_ijk = MIN_SINE;
        else if (s_ijk <= 0 && s_ijk >= -MIN_SINE) s_ijk = -MIN_SINE;
        if (s_jkl >= 0 && s_jkl <= MIN_SINE) s_jkl = MIN_SINE;
        else if (s_jkl <= 0 && s_jkl >= -MIN_SINE) s_jkl = -MIN_SINE;
        const double sc = 2.0 / poem;
        const double a_ij = (htra - arg * hnra) / r_ij, a_kl = (htrc - arg * hnrc) / r_kl, a_jk = htrb / r_jk;
        const double t_d = (hthd - arg * hnhd) / s_ijk, t_e = (hthe - arg * hnhe) / s_jkl;
        // torsion and conjugation energies
        const double cos_omega = cos(omega), cos2omega = cos(2. * omega), cos3omega = cos(3. * omega);
        const double exp_tor1 = exp(fb.p_tor1 * (2.0 - BOpi_jk - f11_DjDk) * (2.0 - BOpi_jk - f11_DjDk));
        const double exp_tor2_kl = exp(-p_tor2 * BOA_kl);
        const double exp_cot2_kl = exp(-p_cot2 * (BOA_kl - 1.5) * (BOA_kl - 1.5));
        const double fn10 = (1.0 - exp_tor2_ij) * (1.0 - exp_tor2_jk) * (1.0 - exp_tor2_kl);
        const double CV = 0.5 * (fb.V1 * (1.0 + cos_omega) + fb.V2 * exp_tor1 * (1.0 - cos2omega) +
                                 fb.V3 * (1.0 + cos3omega));
        term[O_TOR][lane] = fn10 * sin_ijk * sin_jkl * CV;
        const double CEtors1 = sin_ijk * sin_jkl * CV;
        const double CEtors2 = -fn10 * 2.0 * fb.p_tor1 * fb.V2 * exp_tor1 * (2.0 - BOpi_jk - f11_DjDk) *
                               (1.0 - cos_omega * cos_omega) * sin_ijk * sin_jkl;
        const double CEtors3 = CEtors2 * dfn11;
        const double CEtors4 = CEtors1 * p_tor2 * exp_tor2_ij * (1.0 - exp_tor2_jk) * (1.0 - exp_tor2_kl);
        const double CEtors5 = CEtors1 * p_tor2 * (1.0 - exp_tor2_ij) * exp_tor2_jk * (1.0 - exp_tor2_kl);
        const double CEtors6 = CEtors1 * p_tor2 * (1.0 - exp_tor2_ij) * (1.0 - exp_tor2_jk) * exp_tor2_kl;
        const double cmn = -fn10 * CV;
        const double CEtors7 = cmn * sin_jkl * tan_ijk_i;
        const double CEtors8 = cmn * sin_ijk * tan_jkl_i;
        const double CEtors9 = fn10 * sin_ijk * sin_jkl *
                               (0.5 * fb.V1 - 2.0 * fb.V2 * exp_tor1 * cos_omega +
                                1.5 * fb.V3 * (cos2omega + 2.0 * cos_omega * cos_omega));
        const double fn12 = exp_cot2_ij * exp_cot2_jk * exp_cot2_kl;
        const double conj = 1.0 + (cos_omega * cos_omega - 1.0) * sin_ijk * sin_jkl;
        term[O_CON][lane] = fb.p_cot1 * fn12 * conj;
        const double Cconj = -2.0 * fn12 * fb.p_cot1 * p_cot2 * conj;
        const double CEconj4 = -fb.p_cot1 * fn12 * (cos_omega * cos_omega - 1.0) * sin_jkl * tan_ijk_i;
        const double CEconj5 = -fb.p_cot1 * fn12 * (cos_omega * cos_omega - 1.0) * sin_ijk * tan_jkl_i;
        const double CEconj6 = 2.0 * fb.p_cot1 * fn12 * cos_omega * sin_ijk * sin_jkl;
        term[O_PI][lane] = CEtors2;
        term[O_FJ + 3][lane] = CEtors3;
        term[O_CDK][lane] = CEtors3;
        iterm[0][lane] = CEtors4 + Cconj * (BOA_ij - 1.5e0);
        term[O_BO][lane] = CEtors5 + Cconj * (BOA_jk - 1.5e0);
        const double cdbo_kl = CEtors6 + Cconj * (BOA_kl - 1.5e0);
        const double c7 = CEtors7 + CEconj4, c8 = CEtors8 + CEconj5, c9 = CEtors9 + CEconj6;
        double fl[3];
        const DCos ijk(bjk, bij, dot_ijk), jkl(bkj, bkl, dot_jkl);
#pragma unroll
        for (int q = 0; q < 3; q++) {
          double ijk_di, ijk_dj, ijk_dk, jkl_di, jkl_dj, jkl_dk;   // of k, j, i; of j, k, l
          ijk.get(bjk, bij, q, ijk_di, ijk_dj, ijk_dk);
          jkl.get(bkj, bkl, q, jkl_di, jkl_dj, jkl_dk);
          const double w_i = sc * (a_ij * dij[q] - dvec_li[q] - t_d * ijk_dk);
          const double w_j = sc * (-a_ij * dij[q] - a_jk * djk[q] - t_d * ijk_dj - t_e * jkl_di);
          const double w_k = sc * (-a_kl * dkl[q] + a_jk * djk[q] - t_d * ijk_di - t_e * jkl_dj);
          const double w_l = sc * (a_kl * dkl[q] + dvec_li[q] - t_e * jkl_dk);
          iterm[1 + q][lane] = c7 * ijk_dk + c9 * w_i;
          term[O_FJ + q][lane] = c7 * ijk_dj + c8 * jkl_di + c9 * w_j;
          term[O_FK + q][lane] = c7 * ijk_di + c8 * jkl_dj + c9 * w_k;
          fl[q] = c8 * jkl_dk + c9 * w_l;
        }
        unsigned long long *al4 = A.acc + 4 * (size_t)l;
        unsigned long long *const ga[4] = {A.sacc + pw, al4, al4 + 1, al4 + 2};
        const size_t gc[4] = {A.scoff, A.coff, A.coff, A.coff};
        const double gv[4] = {cdbo_kl, fl[0], fl[1], fl[2]};
        fix_add_group<4>(A.flags, ga, gc, gv);
      }
      sph[lane] = ph;
      wave_lds_order();
      // i's terms: each j-i bond's quadruples are neighbouring lanes; the
      // first of them sums them
      if (ev && (w.sub == 0 || sph[lane - 1] != ph)) {
        double v[4] = {0.0, 0.0, 0.0, 0.0};
        for (int e = w.sub; e < take && sph[g0 + e] == ph; ++e)
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] += iterm[q][g0 + e];
        if (v[0] != 0.0 || v[1] != 0.0 || v[2] != 0.0 || v[3] != 0.0) {
          unsigned long long *ai4 = A.acc + 4 * (size_t)i;
          unsigned long long *const ga[4] = {A.sacc + ph, ai4, ai4 + 1, ai4 + 2};
          const size_t gc[4] = {A.scoff, A.coff, A.coff, A.coff};
          fix_add_group<4>(A.flags, ga, gc, v);
        }
      }
      // the bond's totals, in quadruple order
      for (int c = w.sub; c < O_NC; c += G) {
        double v = T.t[c][g0];
        for (int e = 0; e < take; ++e) v += term[c][g0 + e];
        T.t[c][g0] = v;
      }
      wave_lds_order();
      queue_drop(Q, w, take);
    }
    wave_lds_order();
    if (w.live && w.sub == 0) {
      const double cdbopi_jk = T.t[O_PI][g0], cdbo_jk = T.t[O_BO][g0];
      if (cdbopi_jk != 0.0) A.Cdbopi[pk] += cdbopi_jk;
      if (cdbo_jk != 0.0) A.Cdbo[pk] += cdbo_jk;
      const double gv[4] = {T.t[O_FK][g0], T.t[O_FK + 1][g0], T.t[O_FK + 2][g0], T.t[O_CDK][g0]};
      if (gv[0] != 0.0 || gv[1] != 0.0 || gv[2] != 0.0 || gv[3] != 0.0) {
        unsigned long long *ak4 = A.acc + 4 * (size_t)k;
        unsigned long long *const ga[4] = {ak4, ak4 + 1, ak4 + 2, ak4 + 3};
        const size_t gc[4] = {A.coff, A.coff, A.coff, A.coff};
        fix_add_group<4>(A.flags, ga, gc, gv);
      }
      double *rw = A.row + 6 * (size_t)pk;
#pragma unroll
      for (int q = 0; q < 4; q++) rw[q] = T.t[O_FJ + q][g0];
      rw[4] = T.t[O_TOR][g0];
      rw[5] = T.t[O_CON][g0];
    }
    wave_lds_order();   // (before the next groups' totals start)
  }
}

// The end of the torsion pass, one thread per atom: j's row and energies from
// its slots' entries in slot order (local atoms), then the fixed-point terms
// into its fCdDelta row and into Cdbo of its bond slots; accumulators are left
// at zero.  The first workgroup clears the work list's counters.
__global__ void __launch_bounds__(BT) k_to_fold(int n, int N, ToArgs A) {
  if (blockIdx.x == 0) {
    wl_clear(A.ctl);
    return;
  }
  const int j = (blockIdx.x - 1) * BT + threadIdx.x;
  if (j >= N) return;
  const int b0 = A.bidx[j], b1 = A.bend[j];
  double *fcd = A.fcd + 4 * (size_t)j;
  double f[4] = {fcd[0], fcd[1], fcd[2], fcd[3]};
  bool any = false;
  if (j < n) {
    double s[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int pk = b0; pk < b1; ++pk) {
      const double *rw = A.row + 6 * (size_t)pk;
#pragma unroll
      for (int q = 0; q < 6; q++) s[q] += rw[q];
    }
    if (A.atoms[j].type >= 0) {
#pragma unroll
      for (int q = 0; q < 4; q++) f[q] += s[q];
      any = true;
    }
    A.part[j] = s[4];
    A.part[A.stride + j] = s[5];
  }
  any |= fold4(N, j, A.acc, f);
  if (any)
#pragma unroll
    for (int c = 0; c < 4; c++) fcd[c] = f[c];
  for (int pk = b0; pk < b1; ++pk) {
    unsigned long long *w = A.sacc + pk;
    if (w[0] != 0ull || w[A.scoff] != 0ull) {
      A.Cdbo[pk] += fix_value(w, A.scoff);
      w[0] = 0ull;
      w[A.scoff] = 0ull;
    }
  }
}

__global__ void __launch_bounds__(BT) k_to_sum(int n, const double *__restrict__ part, size_t stride,
                                               double *__restrict__ sums) {
  sum_row<16>(n, part + blockIdx.x * stride, sums + blockIdx.x);
}

}  // namespace

int swr_atom_energy_run(swr_system *S) {
  const int n = S->n, N = S->N;
  if (!S->bonds || !S->bo_data || !S->fcd || N <= 0) {
    swr_set_error_msg("Atom_Energy needs the bonds and bond orders of the step (swr_bo first)");
    return SWR_ERR_STATE;
  }
  int rc;
  const size_t stride = (size_t)std::max(n, 1);   // rows as long as the local atoms: the getter copies 5n
  if ((rc = swr_reserve(&S->be_part, S->cap_be_part, 5 * stride)) ||
      (rc = swr_reserve(&S->be_ce, S->cap_be_ce, 2 * stride)) ||
      (rc = swr_reserve(&S->be_result, S->cap_be_result, 8)))
    return rc;
  S->be_stride = stride;
  BeArgs A;
  A.P = S->dp;
  A.atoms = S->packed;
  A.bidx = S->bond_index;
  A.bend = S->bond_end;
  A.bonds = S->bonds;
  A.bo = S->bo_data;
  A.BO = S->BO;
  A.BOpi = S->BOpi;
  const double *ws = S->ws;
  A.Delta = ws + (size_t)WS_DELTA * S->Ncap;
  A.Delta_lp = ws + (size_t)WS_DELTA_LP * S->Ncap;
  A.dDelta_lp = ws + (size_t)WS_DDELTA_LP * S->Ncap;
  A.Delta_lp_temp = ws + (size_t)WS_DELTA_LP_TEMP * S->Ncap;
  A.bo_dboc = S->bo_dboc;
  A.Cdbo = S->Cdbo;
  A.Cdbopi = S->Cdbopi;
  A.Cdbopi2 = S->Cdbopi2;
  A.fcd = S->fcd;
  A.ce = S->be_ce;
  A.part = S->be_part;
  A.stride = stride;
  swr_kt_begin(S, KT_ATOM_ENERGY);
  if (n > 0) hipLaunchKernelGGL(k_atom_energy, dim3(div_up(n, AE_ATOMS)), dim3(BT), 0, S->stream, n, A);
  hipLaunchKernelGGL(k_atom_energy_nbr, dim3(5 + div_up(N, BT)), dim3(BT), 0, S->stream, n, N, A, S->be_result);
  swr_kt_end(S, KT_ATOM_ENERGY);
  HIP_CHECK(hipGetLastError());
  return SWR_OK;
}

int swr_dbond_forces_run(swr_system *S) {
  const int N = S->N;
  if (!S->bonds || !S->bo_data || !S->fcd || N <= 0) {
    swr_set_error_msg("Add_All_dBond_to_Forces needs the bonds and bond orders of the step");
    return SWR_ERR_STATE;
  }
  int rc;
  if ((rc = swr_reserve(&S->be_bufc, S->cap_be_bufc, (size_t)S->Ncap))) return rc;
  DbArgs A;
  A.bonds = S->bonds;
  A.bo = S->bo_data;
  A.bidx = S->bond_index;
  A.bend = S->bond_end;
  A.Cdbo = S->Cdbo;
  A.Cdbopi = S->Cdbopi;
  A.Cdbopi2 = S->Cdbopi2;
  A.dDeltap_self = S->dDeltap_self;
  A.fcd = S->fcd;
  A.bufc = S->be_bufc;
  swr_kt_begin(S, KT_DBOND);
  hipLaunchKernelGGL(k_dbond_own, dim3(div_up((long long)N * BG, BT)), dim3(BT), 0, S->stream, N, A);
  hipLaunchKernelGGL(k_dbond_nbr, dim3(div_up(N, BT)), dim3(BT), 0, S->stream, N, A);
  swr_kt_end(S, KT_DBOND);
  HIP_CHECK(hipGetLastError());
  return SWR_OK;
}

int swr_hydrogen_bonds_run(swr_system *S) {
  const int n = S->n, N = S->N;
  if (!S->bonds || !S->BO || !S->fcd || N <= 0 || !S->hbonds) {
    swr_set_error_msg("Hydrogen_Bonds needs the bonds, bond orders and hydrogen-bond lists of the step");
    return SWR_ERR_STATE;
  }
  int rc;
  const size_t old_acc = S->cap_hb_acc;
  if ((rc = swr_reserve(&S->hb_part, S->cap_hb_part, (size_t)std::max(n, 1))) ||
      (rc = swr_reserve(&S->hb_result, S->cap_hb_result, 1)) ||
      (rc = swr_reserve(&S->hb_acc, S->cap_hb_acc, 6 * (size_t)N)))
    return rc;
  // a new accumulator starts at zero; afterwards k_hb_fold leaves it so
  if (S->cap_hb_acc != old_acc)
    HIP_CHECK(hipMemsetAsync(S->hb_acc, 0, sizeof(unsigned long long) * S->cap_hb_acc, S->stream));
  HbArgs A;
  A.P = S->dp;
  A.atoms = S->packed;
  A.bidx = S->bond_index;
  A.bend = S->bond_end;
  A.bonds = S->bonds;
  A.BO = S->BO;
  A.Hindex = S->Hindex;
  A.hidx = S->hbond_index;
  A.hend = S->hbond_end;
  A.hbonds = S->hbonds;
  A.Cdbo = S->Cdbo;
  A.fcd = S->fcd;
  A.part = S->hb_part;
  A.acc = S->hb_acc;
  A.coff = 3 * (size_t)N;
  A.flags = &S->status->flags;
  // atoms per workgroup: few while that fills the chip, more share their
  // partners' sums.  With 8, 16 and 64 of them (us): 6,000 water atoms 39, 40,
  // 65; 7,400 of four clusters 39, 36, 56; 8,000 51, 46, 65; 18,000 75, 74, 82;
  // 24,000 99, 92, 89; 32,000 of thirty clusters 96, 86, 82; 96,000 340, 321, 302
  const int per = n <= 7168 ? 8 : n <= 24576 ? 16 : HB_ATOMS;
  swr_kt_begin(S, KT_HBONDS);
  if (n > 0) hipLaunchKernelGGL(k_hb, dim3(div_up(n, per)), dim3(BT), 0, S->stream, n, per, A);
  hipLaunchKernelGGL(k_hb_fold, dim3(1 + div_up(N, BT)), dim3(BT), 0, S->stream, n, N, S->hb_acc, S->fcd,
                     (const double *)S->hb_part, S->hb_result);
  swr_kt_end(S, KT_HBONDS);
  HIP_CHECK(hipGetLastError());
  return SWR_OK;
}

int swr_valence_angles_run(swr_system *S) {
  const int n = S->n, N = S->N;
  if (!S->bonds || !S->BO || !S->fcd || N <= 0) {
    swr_set_error_msg("Valence_Angles needs the bonds and bond orders of the step (swr_bo first)");
    return SWR_ERR_STATE;
  }
  int rc;
  const size_t stride = (size_t)std::max(n, 1);
  const size_t old_acc = S->cap_va_acc;
  const size_t old_ctl = S->cap_va_ctl;
  if ((rc = swr_reserve(&S->va_part, S->cap_va_part, 3 * stride)) ||
      (rc = swr_reserve(&S->va_result, S->cap_va_result, 4)) ||
      (rc = swr_reserve(&S->va_acc, S->cap_va_acc, 8 * (size_t)N)) ||
      (rc = swr_reserve(&S->va_cnt, S->cap_va_cnt, stride)) ||
      (rc = swr_reserve(&S->va_order, S->cap_va_order, stride)) ||
      (rc = swr_reserve(&S->va_ctl, S->cap_va_ctl, (size_t)WL_CTL_INTS)))
    return rc;
  if (S->cap_va_acc != old_acc)
    HIP_CHECK(hipMemsetAsync(S->va_acc, 0, sizeof(unsigned long long) * S->cap_va_acc, S->stream));
  // the counters start at zero; k_va_fold leaves them so
  if (S->cap_va_ctl != old_ctl) HIP_CHECK(hipMemsetAsync(S->va_ctl, 0, sizeof(int) * S->cap_va_ctl, S->stream));
  S->va_stride = stride;
  VaArgs A;
  A.P = S->dp;
  A.atoms = S->packed;
  A.bidx = S->bond_index;
  A.bend = S->bond_end;
  A.bonds = S->bonds;
  A.BO = S->BO;
  A.BOpi = S->BOpi;
  A.bo_dboc = S->bo_dboc;
  const double *ws = S->ws;
  A.Delta = ws + (size_t)WS_DELTA * S->Ncap;
  A.Delta_val = ws + (size_t)WS_DELTA_VAL * S->Ncap;
  A.vlpex = ws + (size_t)WS_VLPEX * S->Ncap;
  A.nlp = ws + (size_t)WS_NLP * S->Ncap;
  A.dDelta_lp = ws + (size_t)WS_DDELTA_LP * S->Ncap;
  A.Cdbo = S->Cdbo;
  A.Cdbopi = S->Cdbopi;
  A.Cdbopi2 = S->Cdbopi2;
  A.fcd = S->fcd;
  A.part = S->va_part;
  A.stride = stride;
  A.acc = S->va_acc;
  A.coff = 4 * (size_t)N;
  A.flags = &S->status->flags;
  A.cnt = S->va_cnt;
  A.order = S->va_order;
  A.ctl = S->va_ctl;
  swr_kt_begin(S, KT_VALENCE);
  if (n > 0) {
    hipLaunchKernelGGL(k_va_count, dim3(div_up((long long)n * BG, BT)), dim3(BT), 0, S->stream, n, A);
    hipLaunchKernelGGL(k_va_scatter, dim3(div_up(n, BT)), dim3(BT), 0, S->stream, n, A);
    int sets = 0;   // most parameter sets of one angle type
    for (int q = 0; q < SWR_MAX_ELEM * SWR_MAX_ELEM * SWR_MAX_ELEM; q++) sets = std::max(sets, (int)S->hp.thb_n[q]);
    const dim3 waves(std::min(WL_MAX_WAVES, n)), wave(SWR_WAVE);
    if (sets <= 2) hipLaunchKernelGGL(k_valence<2>, waves, wave, 0, S->stream, A);
    else hipLaunchKernelGGL(k_valence<SWR_MAX_THB>, waves, wave, 0, S->stream, A);
  }
  hipLaunchKernelGGL(k_va_fold, dim3(4 + div_up(N, BT)), dim3(BT), 0, S->stream, n, N, A, S->va_result);
  swr_kt_end(S, KT_VALENCE);
  HIP_CHECK(hipGetLastError());
  return SWR_OK;
}

int swr_torsion_angles_run(swr_system *S) {
  const int n = S->n, N = S->N;
  if (!S->bonds || !S->BO || !S->fcd || N <= 0) {
    swr_set_error_msg("Torsion_Angles needs the bonds and bond orders of the step (swr_bo first)");
    return SWR_ERR_STATE;
  }
  int rc;
  const size_t stride = (size_t)std::max(n, 1);
  const int nslots = S->bond_cap;
  const size_t old_acc = S->cap_to_acc, old_sacc = S->cap_to_sacc, old_ctl = S->cap_to_ctl;
  const size_t slots = (size_t)std::max(nslots, 1);
  if ((rc = swr_reserve(&S->to_part, S->cap_to_part, 2 * stride)) ||
      (rc = swr_reserve(&S->to_result, S->cap_to_result, 4)) ||
      (rc = swr_reserve(&S->to_acc, S->cap_to_acc, 8 * (size_t)N)) ||
      (rc = swr_reserve(&S->to_sacc, S->cap_to_sacc, 2 * slots)) ||
      (rc = swr_reserve(&S->to_tc, S->cap_to_tc, slots)) ||
      (rc = swr_reserve(&S->to_task, S->cap_to_task, 2 * slots)) ||
      (rc = swr_reserve(&S->to_row, S->cap_to_row, 6 * slots)) ||
      (rc = swr_reserve(&S->to_ctl, S->cap_to_ctl, (size_t)WL_CTL_INTS)))
    return rc;
  if (S->cap_to_acc != old_acc)
    HIP_CHECK(hipMemsetAsync(S->to_acc, 0, sizeof(unsigned long long) * S->cap_to_acc, S->stream));
  if (S->cap_to_sacc != old_sacc)
    HIP_CHECK(hipMemsetAsync(S->to_sacc, 0, sizeof(unsigned long long) * S->cap_to_sacc, S->stream));
  // the counters start at zero; k_to_fold leaves them so
  if (S->cap_to_ctl != old_ctl) HIP_CHECK(hipMemsetAsync(S->to_ctl, 0, sizeof(int) * S->cap_to_ctl, S->stream));
  S->to_stride = stride;
  ToArgs A;
  A.P = S->dp;
  A.atoms = S->packed;
  A.bidx = S->bond_index;
  A.bend = S->bond_end;
  A.bonds = S->bonds;
  A.BO = S->BO;
  A.BOpi = S->BOpi;
  A.bo_dboc = S->bo_dboc;
  A.Cdbo = S->Cdbo;
  A.Cdbopi = S->Cdbopi;
  A.fcd = S->fcd;
  A.part = S->to_part;
  A.stride = stride;
  A.acc = S->to_acc;
  A.coff = 4 * (size_t)N;
  A.flags = &S->status->flags;
  A.sacc = S->to_sacc;
  A.scoff = slots;
  A.bnbr = S->bond_nbr;
  A.tc = S->to_tc;
  A.task = reinterpret_cast<int2 *>(S->to_task);
  A.ctl = S->to_ctl;
  A.row = S->to_row;
  swr_kt_begin(S, KT_TORSION);
  if (n > 0) {
    hipLaunchKernelGGL(k_to_count, dim3(div_up((long long)n * TO_CNT_LANES, BT)), dim3(BT), 0, S->stream, n, A);
    hipLaunchKernelGGL(k_to_scatter, dim3(div_up(n, BT)), dim3(BT), 0, S->stream, n, A);
    const int waves = (int)std::min<long long>(WL_MAX_WAVES, 8LL * n);
    if (n >= TORSION_TWO_WAVES) hipLaunchKernelGGL(k_torsion<2>, dim3(waves), dim3(SWR_WAVE), 0, S->stream, A);
    else hipLaunchKernelGGL(k_torsion<1>, dim3(waves), dim3(SWR_WAVE), 0, S->stream, A);
  }
  hipLaunchKernelGGL(k_to_fold, dim3(1 + div_up(N, BT)), dim3(BT), 0, S->stream, n, N, A);
  hipLaunchKernelGGL(k_to_sum, dim3(2), dim3(BT), 0, S->stream, n, (const double *)S->to_part, stride, S->to_result);
  swr_kt_end(S, KT_TORSION);
  HIP_CHECK(hipGetLastError());
  return SWR_OK;
}
