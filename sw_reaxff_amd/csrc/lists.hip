// lists.hip — atom pack (a2), Reset (a4), far list (a3), bonds + hbonds
// (a5, a6) and list validation (a7).
//
// The far/bond/hbond pass is one wave per atom i streaming i's Verlet
// candidates 64 at a time:
//   far   : d^2 <= nonb_cut^2, entry written with a wave-ballot compaction in
//           candidate order (write_reax_lists_c_para, pair_reaxc_sw64.c:276-331);
//   bond  : d <= bond_cut and uncorrected BO' >= bo_cut (BOp_single,
//           reaxc_forces_sunway.cpp:677-825; kernel reaxc_forces_sw64.c:1126-1280),
//           gathered in LDS, then sorted by nbr (my_bubble_sort, :31-75);
//   hbond : local H, far entry with d <= hbond_cut and p_hbond(j) == 2
//           (Init_Forces_noQEq_HB_Full_C, reaxc_forces_sw64.c:810-862).
// Far slots of atom i are [voff[i], voff[i+1]) — bounded by its Verlet
// count — so no separate counting pass is needed (the reference uses
// i*maxfar, pair_reaxc_sw64.c:256).
#include <cstring>
#include <type_traits>
#include <vector>

#include "swr_internal.h"
#include "swr_device.h"

namespace {

constexpr int LT = 256;                 // threads per block
constexpr int LW = LT / SWR_WAVE;       // waves per block
constexpr int MB = SWR_MAX_ATOM_BONDS;  // LDS bond slots per atom

// Orders this wave's LDS writes before its later LDS reads (each wave only
// touches its own LDS slice, so no workgroup barrier is needed).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__global__ void k_pack(const int *__restrict__ tag, const int *__restrict__ type, const double *__restrict__ x,
                       const double *__restrict__ q, const DevParams *__restrict__ P, int N,
                       swr_atom_pack_t *__restrict__ out) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  swr_atom_pack_t a;
  a.orig_id = tag[i];
  a.type = P->map[type[i]];
  a.x[0] = x[3 * i]; a.x[1] = x[3 * i + 1]; a.x[2] = x[3 * i + 2];
  a.q = q[i];
  out[i] = a;
}

// An upload of swr_set_atoms ([N] x, y, z, then q if has_q, tag, type, owner if
// has_owner and img in bytes if has_img) into the atom arrays; without owners
// each atom owns itself, without q or img these are zero.
__global__ void k_unpack_atoms(int N, const int *__restrict__ in, int has_q, int has_owner, int has_img,
                               double *__restrict__ x, double *__restrict__ q, int *__restrict__ tag,
                               int *__restrict__ type, int *__restrict__ owner, signed char *__restrict__ img) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  const double *d = reinterpret_cast<const double *>(in);
  for (int c = 0; c < 3; c++) x[3 * (size_t)i + c] = d[3 * (size_t)i + c];
  d += 3 * (size_t)N;
  q[i] = has_q ? d[i] : 0.0;
  const int *w = reinterpret_cast<const int *>(d + (has_q ? N : 0));
  tag[i] = w[i];
  type[i] = w[N + i];
  w += 2 * (size_t)N;
  owner[i] = has_owner ? w[i] : i;
  const signed char *b = reinterpret_cast<const signed char *>(w + (has_owner ? N : 0));
  for (int c = 0; c < 3; c++) img[3 * (size_t)i + c] = has_img ? b[3 * (size_t)i + c] : (signed char)0;
}

// Reset_Atoms / Reset_Neighbor_Lists in two launches: k_reset_sums adds up
// each tile of RS_TILE atoms (local H atoms, their hydrogen-bond capacities,
// bond capacities) and zeroes fCdDelta; k_reset_apply adds the tiles before
// its own and scans its tile.  (Flags, a three-launch scan of the three arrays,
// their use and a fill were six launches of ~4 us each with their gaps, more
// than half of it waiting between them, on all but the largest systems.)
constexpr int RS_T = 256, RS_ITEMS = 4, RS_TILE = RS_T * RS_ITEMS;

struct ResetArgs {
  const swr_atom_pack_t *atoms;
  const DevParams *P;
  int n, N;
  double hbond_cut;
  const int *num_hbonds, *num_bonds;
  int *sums;   // [tiles][3]
};

// (H atoms, hydrogen-bond capacity, bond capacity) of atom i.
__device__ __forceinline__ int3 reset_item(const ResetArgs &A, int i) {
  if (i >= A.N) return make_int3(0, 0, 0);
  const int t = A.atoms[i].type;
  const int h = (i < A.n && A.hbond_cut > 0 && t >= 0 && A.P->p_hbond[t] == 1) ? 1 : 0;
  return make_int3(h, h ? A.num_hbonds[i] : 0, A.num_bonds[i]);
}

__device__ __forceinline__ int3 add3(int3 a, int3 b) { return make_int3(a.x + b.x, a.y + b.y, a.z + b.z); }

// The workgroup's sum of v; excl: the sum of the threads before this one.
__device__ __forceinline__ int3 reset_block_scan(int3 v, int3 *lds, int3 *excl) {
  const int w = wave_in_block(), l = lane_id();
  const int3 inc = make_int3(wave_incl_scan(v.x), wave_incl_scan(v.y), wave_incl_scan(v.z));
  __syncthreads();
  if (l == SWR_WAVE - 1) lds[w] = inc;
  __syncthreads();
  int3 off = make_int3(0, 0, 0), tot = off;
  for (int k = 0; k < RS_T / SWR_WAVE; k++) {
    if (k < w) off = add3(off, lds[k]);
    tot = add3(tot, lds[k]);
  }
  *excl = make_int3(off.x + inc.x - v.x, off.y + inc.y - v.y, off.z + inc.z - v.z);
  return tot;
}

__global__ void __launch_bounds__(RS_T) k_reset_sums(ResetArgs A, double *__restrict__ fcd) {
  __shared__ int3 lds[RS_T / SWR_WAVE];
  const int base = blockIdx.x * RS_TILE;
  int3 v = make_int3(0, 0, 0), ex;
#pragma unroll
  for (int k = 0; k < RS_ITEMS; k++) v = add3(v, reset_item(A, base + k * RS_T + (int)threadIdx.x));
  const int3 tot = reset_block_scan(v, lds, &ex);
  if (threadIdx.x < 3) A.sums[3 * blockIdx.x + threadIdx.x] = threadIdx.x == 0 ? tot.x : threadIdx.x == 1 ? tot.y : tot.z;
  double2 *f = reinterpret_cast<double2 *>(fcd);
#pragma unroll
  for (int k = 0; k < 2 * RS_ITEMS; k++) {
    const long long e = 2LL * base + k * RS_T + threadIdx.x;
    if (e < 2LL * A.N) f[e] = make_double2(0.0, 0.0);
  }
}

__global__ void __launch_bounds__(RS_T)
k_reset_apply(ResetArgs A, int *__restrict__ Hindex, int *__restrict__ bond_index, int *__restrict__ bond_end,
              int *__restrict__ hbond_index, int *__restrict__ hbond_end, DevStatus *st, int bond_cap,
              int hbond_cap) {
  __shared__ int3 lds[RS_T / SWR_WAVE];
  int3 before = make_int3(0, 0, 0), ex;
  for (int k = threadIdx.x; k < (int)blockIdx.x; k += RS_T)
    before = add3(before, make_int3(A.sums[3 * k], A.sums[3 * k + 1], A.sums[3 * k + 2]));
  const int3 off = reset_block_scan(before, lds, &ex);
  const int i0 = blockIdx.x * RS_TILE + threadIdx.x * RS_ITEMS;
  int3 v[RS_ITEMS], sum = make_int3(0, 0, 0);
#pragma unroll
  for (int k = 0; k < RS_ITEMS; k++) {
    v[k] = reset_item(A, i0 + k);
    sum = add3(sum, v[k]);
  }
  const int3 tot = reset_block_scan(sum, lds, &ex);
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
    const int3 all = add3(off, tot);
    st->numH = all.x;
    st->total_hbonds = all.y;
    st->total_bonds = all.z;
    if (all.z > bond_cap) atomicOr(&st->flags, SWR_F_BOND_TOTAL);
    if (all.y > hbond_cap) atomicOr(&st->flags, SWR_F_HBOND_TOTAL);
  }
  int3 at = add3(off, ex);
#pragma unroll
  for (int k = 0; k < RS_ITEMS; k++) {
    if (i0 + k < A.N) {
      bond_index[i0 + k] = bond_end[i0 + k] = at.z;
      Hindex[i0 + k] = v[k].x ? at.x : -1;
      if (v[k].x) hbond_index[at.x] = hbond_end[at.x] = at.y;
    }
    at = add3(at, v[k]);
  }
}

// Per atom, the far-list slots of its bond candidates (d <= bond_cut and
// inside the pair's BO' radius); the bond pass evaluates them.
constexpr int MCAND = 64;

// Streaming 16-byte store: the far list is written once per step and read
// back only sparsely, so it should not displace the gathered atoms in L2.
__device__ __forceinline__ void store_nt(double2 *dst, double2 v) {
  typedef double nd2 __attribute__((ext_vector_type(2)));
  nd2 t = {v.x, v.y};
  __builtin_nontemporal_store(t, reinterpret_cast<nd2 *>(dst));
}

// The r-th far entry of a chunk as four 16-byte pieces in the chunk's LDS
// (rel_box stays 0), turned by r / 4: pieces of one column in their plain
// places would be 64 bytes apart, sixteen entries on four banks of 16 bytes
// (two thirds of the far pass's LDS cycles: 1585 -> 1415 us on 512 clusters,
// 625 -> 549 on 36,000 water atoms, 69 -> 63 on 1,944).
__device__ __forceinline__ void stage_far(double2 *chunk, int r, int j, int tj, int tagj, double d, double qj,
                                          double dx, double dy, double dz) {
  double2 *dst = chunk + 4 * r;
  int4 *p = reinterpret_cast<int4 *>(dst);
  const int t = r >> 2;
  p[t & 3] = make_int4(j, tj, tagj, 0);
  p[(t + 1) & 3] = make_int4(0, 0, __double2loint(d), __double2hiint(d));
  dst[(t + 2) & 3] = make_double2(qj, dx);
  dst[(t + 3) & 3] = make_double2(dy, dz);
}
// Where piece t (counted through the chunk's entries) is.
__device__ __forceinline__ int staged_piece(int t) { return (t & ~3) + ((t + (t >> 4)) & 3); }

// Uncorrected bond order of one pair (BOp_single, reaxc_forces_sunway.cpp:695-717).
struct BOpTerms { double BO, BO_s, pi, pi2, C12, C34, C56; };
__device__ __forceinline__ BOpTerms bop_terms(const DevParams *__restrict__ P, int ei, int ej, double d) {
  const DevTbp &tw = P->tbp[ei * SWR_MAX_ELEM + ej];
  BOpTerms t;
  if (P->r_s[ei] > 0.0 && P->r_s[ej] > 0.0) {
    t.C12 = tw.p_bo1 * pow(d / tw.r_s, tw.p_bo2);
    t.BO_s = (1.0 + P->bo_cut) * exp(t.C12);
  } else t.BO_s = t.C12 = 0.0;
  if (P->r_pi[ei] > 0.0 && P->r_pi[ej] > 0.0) {
    t.C34 = tw.p_bo3 * pow(d / tw.r_p, tw.p_bo4);
    t.pi = exp(t.C34);
  } else t.pi = t.C34 = 0.0;
  if (P->r_pi_pi[ei] > 0.0 && P->r_pi_pi[ej] > 0.0) {
    t.C56 = tw.p_bo5 * pow(d / tw.r_pp, tw.p_bo6);
    t.pi2 = exp(t.C56);
  } else t.pi2 = t.C56 = 0.0;
  t.BO = t.BO_s + t.pi + t.pi2;
  return t;
}

// Pass 1 from a far list that is there (swr_init_forces_noqeq_full): one wave
// per atom reads its far entries 64 at a time, records the bond candidates'
// far slots and writes the hydrogen bonds of local H
// (Init_Forces_noQEq_HB_Full_C, reaxc_forces_sw64.c:810-862).
__global__ void __launch_bounds__(LT)
k_from_far(int n, int N, const DevParams *__restrict__ P, const swr_atom_pack_t *__restrict__ atoms,
           swr_far_neighbor_t *__restrict__ far, const int *__restrict__ far_index, const int *__restrict__ far_end,
           int *__restrict__ cand, int *__restrict__ cand_count, const int *__restrict__ Hindex,
           const int *__restrict__ num_hbonds, const int *__restrict__ hbond_index, int *__restrict__ hbond_end,
           swr_hbond_t *__restrict__ hbonds, int *__restrict__ hb_count, int hbond_cap, DevStatus *st) {
  const int i = blockIdx.x * LW + wave_in_block();
  if (i >= N) return;
  const int lane = lane_id();
  const int ei = atoms[i].type;
  const double bond_cut = P->bond_cut, hbond_cut = P->hbond_cut;
  const long long cbeg = far_index[i], cend = far_end[i];
  int ncand = 0;
  const bool doH = (i < n) && ei >= 0 && P->p_hbond[ei] == 1 && hbond_cut > 0;
  const int H = doH ? Hindex[i] : -1;
  int htop = doH ? hbond_end[H] : 0;
  // capacity of this H's slots, never past the end of the list
  const int hlim = doH ? min(hbond_index[H] + num_hbonds[i], hbond_cap) : 0;
  const double *rbo = P->rbo + (ei >= 0 ? ei : 0) * SWR_MAX_ELEM;
  int *mycand = cand + (size_t)i * MCAND;
  for (long long base = cbeg; base < cend; base += SWR_WAVE) {
    const long long slot = base + lane;
    const bool valid = slot < cend;
    int j = 0, tj = -1;
    double d = 0;
    if (valid) {
      const int4 h0 = *reinterpret_cast<const int4 *>(far + slot);
      j = h0.x;
      tj = h0.y;
      d = far[slot].d;
    }
    const bool iscand = valid && ei >= 0 && tj >= 0 && d <= bond_cut && d <= rbo[tj];
    const unsigned long long cm = __ballot(iscand);
    if (iscand) {
      const int c = ncand + ballot_rank(cm);
      if (c < MCAND) mycand[c] = (int)slot;
    }
    ncand += __popcll(cm);
    if (doH) {
      bool ish = false;
      if (valid && d <= hbond_cut) {
        const int tjj = atoms[j].type;
        ish = tjj >= 0 && P->p_hbond[tjj] == 2;
      }
      const unsigned long long hm = __ballot(ish);
      if (ish) {
        const int pos = htop + ballot_rank(hm);
        if (pos < hlim) {
          swr_hbond_t hb;
          hb.nbr = j;
          hb.scl = 1;
          hb.ptr = far + slot;
          hbonds[pos] = hb;
        }
      }
      htop += __popcll(hm);
    }
  }
  if (lane == 0) {
    cand_count[i] = ncand;
    if (ncand > MCAND) atomicOr(&st->flags, SWR_F_BOND_LDS);
    if (doH) {
      if (htop > hlim) {
        atomicOr(&st->flags, SWR_F_HBOND_CAP);
        atomicMax(&st->need_hbond_cap, htop - hbond_index[H]);
      }
      hbond_end[H] = htop > hlim ? hlim : htop;
      hb_count[i] = htop - hbond_index[H];
    }
  }
}

// Pass 1 from the Verlet list, split between two kinds of waves.
//
// A wave's vector-memory counter (vmcnt) counts loads and stores together
// and retires them in issue order, so a wave that writes its far entries
// and then gathers the next neighbours waits for its own stores to reach
// memory before every gather.  Here FG "gatherer" waves (one atom each)
// only load: per phase each takes one 64-candidate chunk of its atom's
// Verlet row, keeps d^2 <= nonb_cut^2 and stages the compacted 64-byte
// entries (plus hbond and bond-candidate records) in LDS, while FWR
// "writer" waves, which never load from global memory, stream the previous
// phase's staged entries out as contiguous 16-byte nontemporal stores.  One
// LDS barrier per phase; double-buffered staging.  A far list is its Verlet
// row filtered in order (write_reax_lists_c_para, pair_reaxc_sw64.c:276-331).
// CAND: the bond candidates' far slots too; HB: the hydrogen bonds of local H
// too, 2 into their list (as k_from_far), 3 their far slots for later.
// The split (FG gatherers, FWR writers per block) is a template parameter;
// the autotuner picks among the FarShape variants below.
template <int FG, int FWR>
struct FarStage {
  double2 far[2][FG][4 * SWR_WAVE];  // staged entries, 4 pieces each
  int2 hb[2][FG][SWR_WAVE];          // staged hbonds: (nbr, far slot)
  int cand[FG][MCAND];               // bond-candidate far slots of the atom
  double rbo[FG][SWR_MAX_ELEM];      // BO' radius row of the atom's element
  long long dst[2][FG];              // far slot of the phase's first entry
  int cnt[2][FG], hdst[2][FG], hcnt[2][FG];
  int nphase[FG];
};

// Gatherer/writer splits the autotuner chooses from.
template <int SH> struct FarShape;
template <> struct FarShape<SWR_FAR_G4W2> { static constexpr int FG = 4, FWR = 2; };
template <> struct FarShape<SWR_FAR_G4W4> { static constexpr int FG = 4, FWR = 4; };
template <> struct FarShape<SWR_FAR_G6W2> { static constexpr int FG = 6, FWR = 2; };
template <> struct FarShape<SWR_FAR_G8W4> { static constexpr int FG = 8, FWR = 4; };

template <class F>
void far_dispatch(int sh, F &&f) {
  switch (sh) {
    case SWR_FAR_G4W4: f(std::integral_constant<int, SWR_FAR_G4W4>()); break;
    case SWR_FAR_G6W2: f(std::integral_constant<int, SWR_FAR_G6W2>()); break;
    case SWR_FAR_G8W4: f(std::integral_constant<int, SWR_FAR_G8W4>()); break;
    default: f(std::integral_constant<int, SWR_FAR_G4W2>()); break;
  }
}

// A gatherer's neighbour record for one chunk: the id and the packed atom.
struct FarNbr {
  int j;
  swr_atom_pack_t a;
};

template <bool CAND, int HB, int FG, int FWR>
__global__ void __launch_bounds__((FG + FWR) * SWR_WAVE)
k_far_ws(int n, int N, const DevParams *__restrict__ P, const swr_atom_pack_t *__restrict__ atoms,
         const long long *__restrict__ voff, const int *__restrict__ vlist, swr_far_neighbor_t *__restrict__ far,
         int *__restrict__ far_index, int *__restrict__ far_end, int *__restrict__ cand,
         int *__restrict__ cand_count, const int *__restrict__ Hindex, const int *__restrict__ num_hbonds,
         const int *__restrict__ hbond_index, int *__restrict__ hbond_end, swr_hbond_t *__restrict__ hbonds,
         int *__restrict__ hb_count, int hbond_cap, int *__restrict__ hbslot, DevStatus *st) {
  __shared__ FarStage<FG, FWR> S;
  const int w = __builtin_amdgcn_readfirstlane(wave_in_block());
  const int lane = lane_id();
  const bool gatherer = w < FG;

  // ---- gatherer set-up: the atom, its Verlet row, its element's tables
  const int g = gatherer ? w : 0;
  const int i = blockIdx.x * FG + g;
  const bool live = gatherer && i < N;
  swr_atom_pack_t ai = {};
  long long cbeg = 0, cend = 0;
  int ei = -1;
  if (live) {
    ai = atoms[i];
    cbeg = voff[i];
    cend = voff[i + 1];
    ei = __builtin_amdgcn_readfirstlane(ai.type);
  }
  const int nch = live ? (int)((cend - cbeg + SWR_WAVE - 1) / SWR_WAVE) : 0;
  const double nonb_cutsq = P->nonb_cutsq, bond_cut = P->bond_cut, hbond_cut = P->hbond_cut;
  unsigned hmask2 = 0;  // elements with p_hbond == 2 (acceptors)
  for (int e = 0; e < SWR_MAX_ELEM; e++) hmask2 |= (P->p_hbond[e] == 2 ? 1u : 0u) << e;
  const bool doH = HB != 0 && live && i < n && ei >= 0 && P->p_hbond[ei] == 1 && hbond_cut > 0;
  // HB 3 finds the hydrogen bonds before Reset has laid out their list: their
  // far slots go to hbslot, at the atom's own Verlet offset (k_hb_place)
  const int H = (doH && HB == 2) ? Hindex[i] : -1;
  int htop = (doH && HB == 2) ? hbond_end[H] : (doH && HB == 3) ? (int)cbeg : 0;
  const int hlim = (doH && HB == 2) ? min(hbond_index[H] + num_hbonds[i], hbond_cap)
                   : (doH && HB == 3) ? (int)cend : 0;
  if (gatherer) {
    if (CAND && lane < SWR_MAX_ELEM) S.rbo[g][lane] = P->rbo[(ei >= 0 ? ei : 0) * SWR_MAX_ELEM + lane];
    if (lane == 0) {
      S.nphase[g] = nch;
      S.cnt[0][g] = S.cnt[1][g] = 0;
      S.hcnt[0][g] = S.hcnt[1][g] = 0;
    }
  }
  // Software pipeline without register copies (a copy of a loaded value
  // waits for the load): while chunk p is evaluated, chunk p+2's atoms and
  // chunk p+6's ids are requested, into three neighbour-record sets that
  // rotate with period 3 and six id registers that rotate with period 6.
  // An id load thus has four phases to arrive before its atoms are
  // requested (Verlet ids stream from HBM, whose read latency under the
  // far list's write stream is a few microseconds), an atom gather two.
  // Every phase of an active gatherer issues the same loads (indices clamped
  // to the row), and the gatherer, idle-gatherer and writer loops are
  // separate, so the compiler's wait counts let the loads stay in flight.
  const long long clast = cend - 1;
  FarNbr X = {}, Y = {}, Z = {};
  int I0 = 0, I1 = 0, I2 = 0, I3 = 0, I4 = 0, I5 = 0;
  if (nch > 0) {
    I0 = vlist[min(cbeg + lane, clast)];
    I1 = vlist[min(cbeg + SWR_WAVE + lane, clast)];
    I2 = vlist[min(cbeg + 2 * SWR_WAVE + lane, clast)];
    I3 = vlist[min(cbeg + 3 * SWR_WAVE + lane, clast)];
    I4 = vlist[min(cbeg + 4 * SWR_WAVE + lane, clast)];
    I5 = vlist[min(cbeg + 5 * SWR_WAVE + lane, clast)];
    X.a = atoms[I0];
    X.j = I0;
    Y.a = atoms[I1];
    Y.j = I1;
  }
  lds_barrier();
  int nph = 0;
  for (int k = 0; k < FG; k++) nph = max(nph, S.nphase[k]);
  // phases 0..nph (the writers drain phase p-1 in phase p); identical in
  // every wave of the block
  const int nphr = __builtin_amdgcn_readfirstlane(nph + 1);

  const long long far0 = cbeg;
  int nfar = 0, ncand = 0;

  // gatherer phase: evaluate chunk p (cur), request chunk p+2's atoms (ids
  // jaddr) into far2 and then chunk p+6's ids into jfree (in this order:
  // waiting for a chunk's atoms then never waits for the ids requested
  // after them)
  auto gather = [&](int p, const FarNbr &cur, FarNbr &far2, const int &jaddr, int &jfree) {
    const int buf = p & 1;
    const long long k = cbeg + (long long)p * SWR_WAVE + lane;
    far2.a = atoms[jaddr];
    far2.j = jaddr;
    jfree = vlist[min(k + 6 * SWR_WAVE, clast)];
    if (p < nch) {
      const bool valid = k < cend;
      double dx = 0, dy = 0, dz = 0, d = 0;
      bool infar = false;
      if (valid) {
        dx = cur.a.x[0] - ai.x[0]; dy = cur.a.x[1] - ai.x[1]; dz = cur.a.x[2] - ai.x[2];
        const double dsq = dx * dx + dy * dy + dz * dz;
        infar = dsq <= nonb_cutsq;
        if (infar) d = sqrt(dsq);
      }
      const int tj = infar ? cur.a.type : -1;
      const unsigned long long m = __ballot(infar);
      const int r = ballot_rank(m);
      const long long slot = far0 + nfar + r;
      if (infar) stage_far(S.far[buf][g], r, cur.j, tj, cur.a.orig_id, d, cur.a.q, dx, dy, dz);
      if (lane == 0) {
        S.dst[buf][g] = far0 + nfar;
        S.cnt[buf][g] = __popcll(m);
      }
      if (CAND) {
        const bool iscand = infar && ei >= 0 && tj >= 0 && d <= bond_cut && d <= S.rbo[g][tj];
        const unsigned long long cm = __ballot(iscand);
        if (iscand) {
          const int c = ncand + ballot_rank(cm);
          if (c < MCAND) S.cand[g][c] = (int)slot;
        }
        ncand += __popcll(cm);
      }
      if (doH) {
        const bool ish = infar && d <= hbond_cut && tj >= 0 && ((hmask2 >> tj) & 1u);
        const unsigned long long hm = __ballot(ish);
        if (HB >= 2) {
          const int hr = ballot_rank(hm);
          if (ish && htop + hr < hlim) S.hb[buf][g][hr] = make_int2(cur.j, (int)slot);
          if (lane == 0) {
            S.hdst[buf][g] = htop;
            S.hcnt[buf][g] = max(0, min(__popcll(hm), hlim - htop));
          }
        }
        htop += __popcll(hm);
      } else if (HB >= 2 && lane == 0) {
        S.hcnt[buf][g] = 0;
      }
      nfar += __popcll(m);
    } else if (lane == 0) {
      S.cnt[buf][g] = 0;
      S.hcnt[buf][g] = 0;
    }
    lds_barrier();
  };

  if (gatherer && nch > 0) {
    // six phases per trip (the period of the id ring): a loop with one exit,
    // then the last nphr % 6 phases in straight-line code continuing the
    // rotation (early exits from the loop make the compiler's wait counts
    // at its header conservative); nphr is wave-uniform, so every wave of
    // the block passes nphr barriers
    int p = 0;
    for (; p + 6 <= nphr; p += 6) {
      gather(p, X, Z, I2, I0);
      gather(p + 1, Y, X, I3, I1);
      gather(p + 2, Z, Y, I4, I2);
      gather(p + 3, X, Z, I5, I3);
      gather(p + 4, Y, X, I0, I4);
      gather(p + 5, Z, Y, I1, I5);
    }
    if (p < nphr) gather(p, X, Z, I2, I0);
    if (p + 1 < nphr) gather(p + 1, Y, X, I3, I1);
    if (p + 2 < nphr) gather(p + 2, Z, Y, I4, I2);
    if (p + 3 < nphr) gather(p + 3, X, Z, I5, I3);
    if (p + 4 < nphr) gather(p + 4, Y, X, I0, I4);
  } else if (gatherer) {
    for (int p = 0; p < nphr; p++) lds_barrier();
  } else {
    // writer: in phase p, drain phase p-1's staging of its gatherers
    for (int p = 0; p < nphr; p++) {
      if (p > 0) {
        const int pb = (p - 1) & 1;
        for (int gg = w - FG; gg < FG; gg += FWR) {
          const int cnt = S.cnt[pb][gg];
          if (cnt > 0) {
            double2 *dstp = reinterpret_cast<double2 *>(far + S.dst[pb][gg]);
            const double2 *src = S.far[pb][gg];
            for (int t = lane; t < 4 * cnt; t += SWR_WAVE) store_nt(dstp + t, src[staged_piece(t)]);
          }
          if (HB == 3) {
            if (lane < S.hcnt[pb][gg]) hbslot[S.hdst[pb][gg] + lane] = S.hb[pb][gg][lane].y;
          }
          if (HB == 2) {
            const int hc = S.hcnt[pb][gg];
            if (lane < hc) {
              const int2 e = S.hb[pb][gg][lane];
              swr_hbond_t hb;
              hb.nbr = e.x;
              hb.scl = 1;
              hb.ptr = far + e.y;
              hbonds[S.hdst[pb][gg] + lane] = hb;
            }
          }
        }
      }
      lds_barrier();
    }
  }
  if (!live) return;
  // per-atom results (the gatherer's only global stores)
  if (CAND) {
    wave_lds_sync();
    const int nc = min(ncand, MCAND);
    for (int t = lane; t < nc; t += SWR_WAVE) cand[(size_t)i * MCAND + t] = S.cand[g][t];
  }
  if (lane == 0) {
    far_index[i] = (int)far0;
    far_end[i] = (int)(far0 + nfar);
    if (CAND) {
      cand_count[i] = ncand;
      if (ncand > MCAND) atomicOr(&st->flags, SWR_F_BOND_LDS);
    }
    if (doH) {
      if (HB == 3) {
        hb_count[i] = htop - (int)cbeg;
      } else {
        if (htop > hlim) {
          atomicOr(&st->flags, SWR_F_HBOND_CAP);
          atomicMax(&st->need_hbond_cap, htop - hbond_index[H]);
        }
        hbond_end[H] = htop > hlim ? hlim : htop;
        hb_count[i] = htop - hbond_index[H];
      }
    }
  }
}

// The hydrogen bonds that the estimate pass found (HB 3), into the list that
// Reset has laid out since: HP_L lanes per local H atom, entries in order.
// Also raises the candidate overflow again, which growing the lists clears.
constexpr int HP_L = 8;
__global__ void __launch_bounds__(LT)
k_hb_place(int n, int N, const int *__restrict__ Hindex, const int *__restrict__ hb_count,
           const int *__restrict__ num_hbonds, const long long *__restrict__ voff, const int *__restrict__ hbslot,
           swr_far_neighbor_t *far, const int *__restrict__ hbond_index, int *__restrict__ hbond_end,
           swr_hbond_t *__restrict__ hbonds, int hbond_cap, const int *__restrict__ cand_count, DevStatus *st) {
  const int i = (int)(blockIdx.x * LT + threadIdx.x) / HP_L, l = threadIdx.x % HP_L;
  if (i >= N) return;
  if (l == 0 && cand_count[i] > MCAND) atomicOr(&st->flags, SWR_F_BOND_LDS);
  if (i >= n || Hindex[i] < 0) return;
  const int H = Hindex[i], c = hb_count[i], first = hbond_index[H];
  const int lim = min(first + num_hbonds[i], hbond_cap);
  const int *src = hbslot + voff[i];
  for (int k = l; k < c && first + k < lim; k += HP_L) {
    const int s = src[k];
    swr_hbond_t hb;
    hb.nbr = far[s].nbr;
    hb.scl = 1;
    hb.ptr = far + s;
    hbonds[first + k] = hb;
  }
  if (l == 0) {
    if (first + c > lim) {
      atomicOr(&st->flags, SWR_F_HBOND_CAP);
      atomicMax(&st->need_hbond_cap, c);
    }
    hbond_end[H] = first + c > lim ? lim : first + c;
  }
}

// Pass 2: BL lanes per atom, SWR_WAVE / BL atoms per wave, evaluate the
// atom's bond candidates (one per lane, BL at a time), keep BO' >= bo_cut in
// candidate (= far-list) order, sort the bonds by nbr (my_bubble_sort,
// reaxc_forces_sw64.c:31-75) and write the bond records, the per-atom sums
// and BO section 1.  An atom has a handful of candidates (about 3 in water,
// 6 in water/methanol clusters), so wider groups left most lanes idle; a
// bond's LDS slot keeps only its far slot and neighbour, and the write pass
// reads the far entry again.  The per-atom sums run in slot order (one
// lane of the group adds the group's values in order through shuffles).
constexpr int BL = 8;   // lanes per atom in k_bonds

template <bool COUNT_ONLY>
__global__ void __launch_bounds__(LT)
k_bonds(int n, int N, const DevParams *__restrict__ P, const swr_atom_pack_t *__restrict__ atoms,
        const swr_far_neighbor_t *__restrict__ far, const int *__restrict__ cand,
        const int *__restrict__ cand_count, const int *__restrict__ num_bonds, const int *__restrict__ bond_index,
        int *__restrict__ bond_end, swr_bond_t *__restrict__ bonds, int *__restrict__ bond_nbr,
        swr_bond_order_t *__restrict__ bo_data,
        double *__restrict__ BO, double *__restrict__ BOpi, double *__restrict__ Cdbo, double *__restrict__ Cdbopi,
        double *__restrict__ Cdbopi2, double *__restrict__ bo_dboc, double *__restrict__ dDeltap_self,
        int *__restrict__ bond_mark, double *__restrict__ Deltap, double *__restrict__ Deltap_boc,
        int *__restrict__ bond_count, int bond_cap, DevStatus *st) {
  constexpr int APW = SWR_WAVE / BL;   // atoms per wave
  __shared__ int sfar[APW * LW][MB];   // far slot of the atom's m-th bond (candidate order)
  __shared__ int snbr[APW * LW][MB];
  const int w = wave_in_block();
  const int lane = lane_id();
  const int grp = lane / BL, sl = lane % BL;
  const int slot_a = APW * w + grp;  // this atom's LDS row
  const int i0 = (xcd_block(gridDim.x) * LW + w) * APW;
  if (i0 >= N) return;               // every atom of the wave past the end
  const int i = i0 + grp;
  const bool live = i < N;
  const int ei = live ? atoms[i].type : -1;
  const double bo_cut = P->bo_cut;
  const int ncand = live ? min(cand_count[i], MCAND) : 0;
  int ncmax = ncand;                 // uniform loop bound over the wave's atoms
#pragma unroll
  for (int o = BL; o < SWR_WAVE; o <<= 1) ncmax = max(ncmax, __shfl_xor(ncmax, o, SWR_WAVE));
  const int *mycand = cand + (size_t)(live ? i : 0) * MCAND;
  const unsigned long long gmask = (1ull << BL) - 1ull;
  const unsigned long long below = (1ull << sl) - 1ull;
  int nb = 0;
  for (int c0 = 0; c0 < ncmax; c0 += BL) {
    const int c = c0 + sl;
    bool isb = false;
    int fs = 0, jn = 0;
    if (c < ncand && ei >= 0) {
      fs = mycand[c];
      const swr_far_neighbor_t e = far[fs];
      const BOpTerms t = bop_terms(P, ei, e.type, e.d);
      if (t.BO >= bo_cut) {
        isb = true;
        jn = e.nbr;
      }
    }
    const unsigned long long bm = (__ballot(isb) >> (BL * grp)) & gmask;
    if (!COUNT_ONLY && isb) {
      const int slot = nb + __popcll(bm & below);
      if (slot < MB) {
        sfar[slot_a][slot] = fs;
        snbr[slot_a][slot] = jn;
      }
    }
    nb += __popcll(bm);
  }
  if (live && sl == 0) bond_count[i] = nb;
  if (COUNT_ONLY) return;
  const int cap = live ? num_bonds[i] : 0;
  const int start = live ? bond_index[i] : 0;
  const bool over = live && (nb > MB || nb > cap || start + nb > bond_cap);
  if (over && sl == 0) {
    atomicOr(&st->flags, nb > MB ? (SWR_F_BOND_LDS | SWR_F_BOND_CAP) : SWR_F_BOND_CAP);
    atomicMax(&st->need_bond_cap, nb);
    bond_end[i] = start;
  }
  const bool write = live && !over;
  const int nbw = write ? nb : 0;
  int nbmax = nbw;
#pragma unroll
  for (int o = BL; o < SWR_WAVE; o <<= 1) nbmax = max(nbmax, __shfl_xor(nbmax, o, SWR_WAVE));
  wave_lds_sync();
  // bo_dboc[i][0] and dDeltap_self[i] accumulate in candidate order
  // (reaxc_forces_sw64.c:1253,1262), starting from Reset's zeros.
  double tot = 0.0, s0 = 0.0, s1 = 0.0, s2 = 0.0;
  for (int m0 = 0; m0 < nbmax; m0 += BL) {
    const int m = m0 + sl;
    double bm_ = 0.0, g0 = 0.0, g1 = 0.0, g2 = 0.0;
    if (m < nbw) {
      const swr_far_neighbor_t e = far[sfar[slot_a][m]];
      const int jn = snbr[slot_a][m];
      const BOpTerms t = bop_terms(P, ei, e.type, e.d);
      const DevTbp &tw = P->tbp[ei * SWR_MAX_ELEM + e.type];
      const double r2 = e.d * e.d;
      const double Cs = tw.p_bo2 * t.C12 / r2, Cp = tw.p_bo4 * t.C34 / r2, Cpp = tw.p_bo6 * t.C56 / r2;
      const double dv[3] = {e.dvec[0], e.dvec[1], e.dvec[2]};
      const double cdb = -(t.BO_s * Cs + t.pi * Cp + t.pi2 * Cpp);
      swr_bond_order_t o;
      o.BO_s = t.BO_s - bo_cut;
      for (int c = 0; c < 3; c++) {
        o.dln_BOp_s[c] = -t.BO_s * Cs * dv[c];
        o.dln_BOp_pi[c] = -t.pi * Cp * dv[c];
        o.dln_BOp_pi2[c] = -t.pi2 * Cpp * dv[c];
        o.dBOp[c] = cdb * dv[c];
      }
      o.C1dbo = o.C2dbo = o.C3dbo = 0.0;
      o.C1dbopi = o.C2dbopi = o.C3dbopi = o.C4dbopi = 0.0;
      o.C1dbopi2 = o.C2dbopi2 = o.C3dbopi2 = o.C4dbopi2 = 0.0;
      o.CdboReduction = nullptr;
      int rank = 0;
      for (int q = 0; q < nbw; q++) rank += (snbr[slot_a][q] < jn) ? 1 : 0;
      const int p = start + rank;
      swr_bond_t b;
      b.d = e.d; b.dvec[0] = dv[0]; b.dvec[1] = dv[1]; b.dvec[2] = dv[2];
      b.nbr = jn;
      b.dbond_index = start + m;
      b.rel_box[0] = b.rel_box[1] = b.rel_box[2] = 0;
      b.sym_index = 0;
      bonds[p] = b;
      bond_nbr[p] = jn;
      bo_data[p] = o;
      BO[p] = t.BO - bo_cut;
      BOpi[2 * (size_t)p] = t.pi;
      BOpi[2 * (size_t)p + 1] = t.pi2;
      Cdbo[p] = 0.0; Cdbopi[p] = 0.0; Cdbopi2[p] = 0.0;
      bm_ = t.BO - bo_cut;
      g0 = o.dBOp[0]; g1 = o.dBOp[1]; g2 = o.dBOp[2];
    }
    // the group's slots m0 .. m0 + BL - 1 in order, onto its first lane
    for (int k = 0; k < BL; k++) {
      const int src = grp * BL + k;
      const double vb = __shfl(bm_, src, SWR_WAVE), v0 = __shfl(g0, src, SWR_WAVE);
      const double v1 = __shfl(g1, src, SWR_WAVE), v2 = __shfl(g2, src, SWR_WAVE);
      if (m0 + k < nbw) {
        tot += vb; s0 += v0; s1 += v1; s2 += v2;
      }
    }
  }
  if (write && sl == 0) {
    bond_end[i] = start + nb;
    bo_dboc[2 * (size_t)i] = tot;
    bo_dboc[2 * (size_t)i + 1] = 0.0;
    dDeltap_self[3 * (size_t)i] = s0;
    dDeltap_self[3 * (size_t)i + 1] = s1;
    dDeltap_self[3 * (size_t)i + 2] = s2;
    bond_mark[i] = (i < n) ? 0 : 1000;
    // BO section 1 (reaxc_bond_orders_sw64.c:56-64), computed here since it
    // only needs this atom's bond-order sum.
    if (ei >= 0) {
      Deltap[i] = tot - P->valency[ei];
      Deltap_boc[i] = tot - P->valency_val[ei];
    }
  }
}

// Counts come from the list pass (bond_count/hb_count hold the true
// per-atom totals even when a capacity overflowed, so the next capacities
// are large enough to retry the step).
__global__ void k_validate(int n, int N, const int *__restrict__ bond_index, const int *__restrict__ bond_count,
                           int *__restrict__ num_bonds, const int *__restrict__ Hindex,
                           const int *__restrict__ hb_count, int *__restrict__ num_hbonds, double saferzone,
                           int bond_total, DevStatus *st, int *__restrict__ next_totals) {
  __shared__ int sb[8], sh[8];
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  int tb = 0, th = 0;
  if (i < N) {
    const int c = bond_count[i];
    tb = max(c * 2, 25);
    num_bonds[i] = tb;
    const int comp = (i < N - 1) ? bond_index[i + 1] : bond_total;
    if (bond_index[i] + c > comp) atomicOr(&st->flags, SWR_F_BOND_CAP);
    if (i < n) {
      const int H = Hindex[i];
      if (H > -1) {
        const double v = hb_count[i] * saferzone;
        th = (int)(v > 25.0 ? v : 25.0);
        num_hbonds[i] = th;
      }
    }
  }
  // totals of the new capacities: the next step's Reset sizes its lists from
  // them without a host round trip (integer sums: order-independent)
  tb = wave_sum(tb);
  th = wave_sum(th);
  if (lane_id() == 0) { sb[wave_in_block()] = tb; sh[wave_in_block()] = th; }
  __syncthreads();
  if (threadIdx.x == 0) {
    int a = 0, b = 0;
    for (int w = 0; w < (int)blockDim.x / SWR_WAVE; w++) { a += sb[w]; b += sh[w]; }
    atomicAdd(&next_totals[0], a);
    atomicAdd(&next_totals[1], b);
  }
}

// The totals into the status block, left at zero for the next pass, and the
// block into the host's copy (one launch instead of a fill and a copy).
static_assert(sizeof(DevStatus) / 4 <= SWR_WAVE && sizeof(DevStatus) % 4 == 0, "a lane of k_validate_end takes one word");
__global__ void __launch_bounds__(SWR_WAVE) k_validate_end(DevStatus *st, int *__restrict__ next_totals, int *host) {
  constexpr int W = sizeof(DevStatus) / 4, AT = offsetof(DevStatus, next_total_bonds) / 4;
  static_assert(offsetof(DevStatus, next_total_hbonds) == 4 * (AT + 1), "the two totals are neighbours");
  const int l = threadIdx.x;
  if (l >= W) return;
  int *words = reinterpret_cast<int *>(st);
  int v = words[l];
  if (l == AT || l == AT + 1) {
    v = next_totals[l - AT];
    next_totals[l - AT] = 0;
    words[l] = v;
  }
  host[l] = v;
  __threadfence_system();
}

// sort_bonds_C (reaxc_forces_sw64.c:932-971): one in-order pass
// bond_mark[i] = min(bond_mark[i], bond_mark[j]+1).  Its result for ghost i
// is min(1000, 1 + min over bonded j < i of the result at j) (locals stay 0,
// later ghosts still hold 1000).  A relaxation of that recursion from the
// initial marks never goes below it and only follows j < i, so it settles on
// exactly that result whatever the order of the updates.
//
// Its length is what bounds it: the chain of hops from the local atoms to the
// farthest bonded ghost (20 to 30 in water's 12 A shell) of dependent reads.
//
// Up to MARK_BFS ghosts: the recursion is a breadth-first search from the
// local atoms along bonds to higher indices, and only a quarter of the ghosts
// are ever reached, so one workgroup walks it level by level with the visited
// set and the queue in LDS (k_mark_bfs), from a compact list of each ghost's
// higher neighbours (k_mark_up; in LDS too up to BFS_LDS ghosts): exact when
// it ends.
//
// More (k_bond_mark): each ghost lowers its mark from its lower neighbours',
// whose ids it keeps in registers, MARK_SWEEPS times a launch as the others'
// updates land (relaxed atomics): a hop is one gather.  chg[launch] is set when
// the launch changed a mark; a launch in which none changed has reached the
// fixed point, and a launch after it does nothing.  Each launch clears the flag
// of the next (a stale chg[0] only makes the host look one launch further).
//
// Walking the bond list for every hop, 1.6 us each, took 49 us on a 64-water
// box, 76 on 648 waters, 94 on 2,667 and 106 on 32,000 (149 after 200 steps of
// MD); with the ids in registers 32,000 take 59 (87).  Relaxing 1024 ghosts at
// a time to their local fixed point in LDS: 85, but 260 after 200 steps, when
// the chains cross its blocks more often.  Six ids and 8 sweeps: 65 (110).
//
// The search is one workgroup's, so its time grows with the bonds of the
// ghosts it reaches.  A ghost with more than four higher neighbours has its list
// walked by the four lanes it gets (by one lane a lattice with a dozen bonds an
// atom took 204 us at 11,600 ghosts, 382 at 23,500 and 522 at 32,300 where
// walking every list takes 171, 226 and 222; by four 107, 197 and 283).  The line
// lies where the relaxation is the faster one on that lattice (27,700 ghosts:
// 244 and 230 us, 32,300: 263 and 188) while on water the search still is
// (22,900 ghosts: 49 and 58 us, with the call's wait).
constexpr int MARK_BFS = 28672;
static_assert(MARK_BFS <= 0x7ffe, "a ghost's position and two codes in 15 bits");
constexpr int BFS_LDS = 12288;
constexpr int BFS_T = 1024;
constexpr int MARK_FAR = 1000;   // mark of a ghost nothing reaches
constexpr int UP_NONE = 0x7fff, UP_LIST = 0x7ffe, UP_NEAR = 0x8000;

// Per ghost its bonds to higher ghosts: the positions (after n) of up to four,
// UP_NONE for none; UP_LIST as the last when there are more (the list is
// walked instead).  UP_NEAR on the first: the ghost is bonded to a local atom.
__global__ void __launch_bounds__(256)
k_mark_up(int n, int N, const int *__restrict__ bond_index, const int *__restrict__ bond_end,
          const int *__restrict__ bond_nbr, ushort4 *__restrict__ up) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x, g = n + r;
  if (g >= N) return;
  const int p0 = bond_index[g], p1 = bond_end[g];
  int u[4] = {UP_NONE, UP_NONE, UP_NONE, UP_NONE};
  int cnt = 0;
  bool near = false;
#pragma unroll 4
  for (int p = p0; p < p1; p++) {
    const int j = bond_nbr[p];
    near |= j < n;
    if (j > g) {
#pragma unroll
      for (int k = 0; k < 4; k++)
        if (cnt == k) u[k] = j - n;
      cnt++;
    }
  }
  if (cnt > 4) u[3] = UP_LIST;
  up[r] = make_ushort4((unsigned short)(u[0] | (near ? UP_NEAR : 0)), (unsigned short)u[1], (unsigned short)u[2],
                       (unsigned short)u[3]);
}

template <bool LDS>
__global__ void __launch_bounds__(BFS_T)
k_mark_bfs(int n, int N, const int *__restrict__ bond_index, const int *__restrict__ bond_end,
           const int *__restrict__ bond_nbr, const ushort4 *__restrict__ up, int *__restrict__ mark) {
  constexpr int CAP = LDS ? BFS_LDS : MARK_BFS;
  __shared__ unsigned int seen[CAP / 32];
  __shared__ unsigned short queue[CAP];   // every ghost enters at most once
  __shared__ ushort4 lup[LDS ? BFS_LDS : 1];
  __shared__ int qend;
  const int ng = N - n;
  for (int k = threadIdx.x; k < (ng + 31) / 32; k += BFS_T) seen[k] = 0u;
  if (threadIdx.x == 0) qend = 0;
  __syncthreads();
  auto reach = [&](int h, int level) {
    const unsigned int bit = 1u << (h & 31);
    if (atomicOr(&seen[h >> 5], bit) & bit) return;
    queue[atomicAdd(&qend, 1)] = (unsigned short)h;
    mark[n + h] = level;
  };
#pragma unroll 4
  for (int r = threadIdx.x; r < ng; r += BFS_T) {
    const ushort4 v = up[r];
    if (LDS) lup[r] = v;
    if (v.x & UP_NEAR) reach(r, 1);
  }
  __syncthreads();
  const unsigned short *ups = LDS ? reinterpret_cast<const unsigned short *>(lup)
                                  : reinterpret_cast<const unsigned short *>(up);
  int begin = 0;
  for (int level = 2; level < MARK_FAR; level++) {
    const int end = qend;
    __syncthreads();   // (before anyone appends)
    if (begin == end) break;
    // four lanes per atom of the frontier, one of its entries each
    for (int f = begin + (int)threadIdx.x / 4; f < end; f += BFS_T / 4) {
      const int r = queue[f], k = threadIdx.x % 4;
      if (ups[4 * r + 3] == UP_LIST) {
        const int p1 = bond_end[n + r];
#pragma unroll 2
        for (int p = bond_index[n + r] + k; p < p1; p += 4)
          if (bond_nbr[p] - n > r) reach(bond_nbr[p] - n, level);
        continue;
      }
      const int h = ups[4 * r + k] & ~UP_NEAR;
      if (h != UP_NONE) reach(h, level);
    }
    __syncthreads();
    begin = end;
  }
}

constexpr int MARK_T = 256;
constexpr int MARK_NB = 8;       // bonds to lower atoms kept in registers
constexpr int MARK_SWEEPS = 12;   // per launch

__global__ void __launch_bounds__(MARK_T)
k_bond_mark(int n, int N, int launch, const int *__restrict__ bond_index, const int *__restrict__ bond_end,
            const int *__restrict__ bond_nbr, int *__restrict__ mark, int *__restrict__ chg) {
  const bool done = launch > 0 && __hip_atomic_load(&chg[launch - 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0;
  if (blockIdx.x == 0 && threadIdx.x == 0 && launch + 1 < MARK_MAX_LAUNCH)
    __hip_atomic_store(&chg[launch + 1], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (done) return;
  const int g = n + blockIdx.x * MARK_T + threadIdx.x;
  if (g >= N) return;
  const int p1 = bond_end[g];
  int p = bond_index[g];
  int cur = __hip_atomic_load(&mark[g], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int first = cur;
  // the first bonds to lower atoms; the others are walked from p on (rare).
  // Unused places are the ghost itself, which never lowers it, so that a
  // sweep reads all of them at once
  int lower[MARK_NB];
#pragma unroll
  for (int k = 0; k < MARK_NB; k++) lower[k] = g;
  for (int cnt = 0; p < p1 && cnt < MARK_NB; p++) {
    const int j = bond_nbr[p];
    if (j >= g) continue;
#pragma unroll
    for (int k = 0; k < MARK_NB; k++)
      if (cnt == k) lower[k] = j;
    cnt++;
  }
  for (int sweep = 0; sweep < MARK_SWEEPS; sweep++) {
    int v[MARK_NB];
#pragma unroll
    for (int k = 0; k < MARK_NB; k++)
      v[k] = __hip_atomic_load(&mark[lower[k]], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    int best = cur;
#pragma unroll
    for (int k = 0; k < MARK_NB; k++) best = min(best, v[k] + 1);
    for (int q = p; q < p1; q++) {
      const int j = bond_nbr[q];
      if (j < g) best = min(best, __hip_atomic_load(&mark[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1);
    }
    if (best < cur) {
      cur = best;
      __hip_atomic_store(&mark[g], cur, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if (cur < first) atomicOr(&chg[launch], 1);
}
__global__ void k_estimate(int n, int N, const int *__restrict__ bond_count, const int *__restrict__ hb_count,
                           const swr_atom_pack_t *__restrict__ atoms, const DevParams *__restrict__ P,
                           double saferzone, int *__restrict__ num_bonds, int *__restrict__ num_hbonds) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  if (i < n) {
    num_bonds[i] = max(bond_count[i] * 2, 25);
    const int t = atoms[i].type;
    const bool isH = t >= 0 && P->p_hbond[t] == 1 && P->hbond_cut > 0;
    const double v = (isH ? hb_count[i] : 0) * saferzone;
    num_hbonds[i] = (int)(v > 25.0 ? v : 25.0);
  } else {
    num_bonds[i] = 25;
    num_hbonds[i] = 0;
  }
}

__global__ void k_set_flag(DevStatus *st, unsigned int f) { atomicOr(&st->flags, f); }

}  // namespace

// ---------------------------------------------------------------- host side
int swr_lists_pack(swr_system *S) {
  hipLaunchKernelGGL(k_pack, dim3(div_up(S->N, 256)), dim3(256), 0, S->stream, S->tag, S->type, S->x, S->q, S->dp,
                     S->N, S->packed);
  HIP_CHECK(hipGetLastError());
  return SWR_OK;
}

int swr_lists_alloc_bonds(swr_system *S, int bond_cap, int hbond_cap);

// The atoms in one upload and one launch: five to seven copies and a fill took
// ~45 us of a 60-atom evaluation's 600.
int swr_stage_atoms(swr_system *S, const int *tag, const int *type, const double *x, const double *q, const int *owner,
                    const signed char *img) {
  const int N = S->N;
  if (N <= 0) return SWR_OK;
  const size_t bytes = (size_t)N * (24 + (q ? 8 : 0) + 8 + (owner ? 4 : 0) + (img ? 3 : 0));
  int rc;
  if ((rc = swr_reserve(&S->atoms_in, S->cap_atoms_in, (bytes + 3) / 4)) ||
      (rc = swr_stage_ready(S, SWR_STAGE_ATOMS, bytes)))
    return rc;
  char *p = (char *)S->stage[SWR_STAGE_ATOMS].pin;
  auto put = [&](const void *src, size_t each) {
    if (!src) return;
    std::memcpy(p, src, each * N);
    p += each * N;
  };
  put(x, 24);
  put(q, 8);
  put(tag, 4);
  put(type, 4);
  put(owner, 4);
  put(img, 3);
  if ((rc = swr_stage_send(S, SWR_STAGE_ATOMS, S->atoms_in, bytes))) return rc;
  hipLaunchKernelGGL(k_unpack_atoms, dim3(div_up(N, 256)), dim3(256), 0, S->stream, N, (const int *)S->atoms_in,
                     q ? 1 : 0, owner ? 1 : 0, img ? 1 : 0, S->x, S->q, S->tag, S->type, S->owner, S->img);
  HIP_CHECK(hipGetLastError());
  HIP_CHECK(hipStreamSynchronize(S->stream));
  return SWR_OK;
}

int swr_lists_reset(swr_system *S) {
  const int n = S->n, N = S->N;
  const int ntiles = div_up(N, RS_TILE);
  int rc = swr_ensure_tmp(S, sizeof(int) * 3 * (size_t)ntiles);
  if (rc) return rc;
  const ResetArgs A = {S->packed, S->dp, n, N, S->ctl.hbond_cut, S->num_hbonds, S->num_bonds, S->tmp_i};
  swr_kt_begin(S, KT_RESET);
  // Reset_Workspace (reaxc_reset_tools_sunway.cpp:122-131) zeroes fCdDelta,
  // which the non-bonded pass accumulates into
  hipLaunchKernelGGL(k_reset_sums, dim3(ntiles), dim3(RS_T), 0, S->stream, A, S->fcd);
  hipLaunchKernelGGL(k_reset_apply, dim3(ntiles), dim3(RS_T), 0, S->stream, A, S->Hindex, S->bond_index, S->bond_end,
                     S->hbond_index, S->hbond_end, S->status, S->bond_cap, S->hbond_cap);
  swr_kt_end(S, KT_RESET);
  HIP_CHECK(hipGetLastError());
  return SWR_OK;
}

// The far pass's split: the tuned one, else by the workgroups there are.  Four
// writer waves for four gatherers while eight atoms a workgroup would leave
// the last round of 512 of them much of the time (13,000 atoms with their
// ghosts 63 us against 72 with eight gatherers and 72 with two writers; 31,000:
// 141, 154, 160; 47,000 of 64 clusters: 135, 143, 163); beyond, eight atoms
// share a phase's barrier and writes (52,000: 246, 240, 297; 103,000 of 128
// clusters: 295, 277, 347; 187,500: 1452, 1370, 1496).
int swr_far_shape(const swr_system *S) {
  if (S->far_shape >= 0) return S->far_shape;
  return S->N >= 49152 ? SWR_FAR_G8W4 : SWR_FAR_G4W4;
}

// mode 0: the far list; 1: far list, bonds and hydrogen bonds; 2: bonds and
// hydrogen bonds from the far list; 3: far list and counts, for the capacity
// estimate; 4: bonds and hydrogen bonds after a 3 on the same packed atoms,
// which spares new atoms the second far pass (168,000 atoms 850 us of a
// 9.6 ms first pass).
int swr_lists_run(swr_system *S, int mode) {
  {  // k_bonds rewrites bond_mark: finish the last relaxation first
    int rc = swr_quiesce(S);
    if (rc) return rc;
  }
  const int N = S->N;
  double *ws = S->ws;
  int rc = SWR_OK;
  if (mode != 0 && (size_t)N * MCAND > S->cand_cap) {
    if ((rc = swr_alloc(&S->cand, (size_t)S->Ncap * MCAND)) || (rc = swr_alloc(&S->cand_count, S->Ncap))) return rc;
    S->cand_cap = (size_t)S->Ncap * MCAND;
  }
  int *hb_count = S->counts + S->Ncap;
#define BOND_ARGS(k)                                                                                              \
  hipLaunchKernelGGL(k, dim3(div_up(N, (SWR_WAVE / BL) * LW)), dim3(LT), 0, S->stream, S->n, N, S->dp, S->packed,     \
                     S->far, S->cand,                                                                              \
                     S->cand_count, S->num_bonds, S->bond_index, S->bond_end, S->bonds, S->bond_nbr, S->bo_data,    \
                     S->BO, S->BOpi,                                                                               \
                     S->Cdbo, S->Cdbopi, S->Cdbopi2, S->bo_dboc, S->dDeltap_self, S->bond_mark,                    \
                     ws + (size_t)WS_DELTAP * S->Ncap, ws + (size_t)WS_DELTAP_BOC * S->Ncap, S->counts,            \
                     S->bond_cap, S->status)
  if (mode == 3) {
    const long long need = S->vtotal_local >= 0 ? S->vtotal_local : S->vtotal;
    if ((rc = swr_reserve(&S->hbslot, S->cap_hbslot, (size_t)std::max(need, 1LL)))) return rc;
  }
  swr_kt_begin(S, KT_FAR);
  if (mode == 2) {
    hipLaunchKernelGGL(k_from_far, dim3(div_up(N, LW)), dim3(LT), 0, S->stream, S->n, N, S->dp, S->packed, S->far,
                       S->far_index, S->far_end, S->cand, S->cand_count, S->Hindex, S->num_hbonds, S->hbond_index,
                       S->hbond_end, S->hbonds, hb_count, S->hbond_cap, S->status);
  } else if (mode == 4) {
    hipLaunchKernelGGL(k_hb_place, dim3(div_up((long long)N * HP_L, LT)), dim3(LT), 0, S->stream, S->n, N, S->Hindex,
                       hb_count, S->num_hbonds, S->voff, S->hbslot, S->far, S->hbond_index, S->hbond_end, S->hbonds,
                       S->hbond_cap, S->cand_count, S->status);
  } else {
    far_dispatch(swr_far_shape(S), [&](auto shc) {
      constexpr int FG = FarShape<decltype(shc)::value>::FG, FWR = FarShape<decltype(shc)::value>::FWR;
      const dim3 gb(div_up(N, FG)), tb((FG + FWR) * SWR_WAVE);
#define FARWS_ARGS(k)                                                                                            \
  hipLaunchKernelGGL(k, gb, tb, 0, S->stream, S->n, N, S->dp, S->packed, S->voff, S->vlist, S->far, S->far_index,    \
                     S->far_end, S->cand, S->cand_count, S->Hindex, S->num_hbonds, S->hbond_index, S->hbond_end,     \
                     S->hbonds, hb_count, S->hbond_cap, S->hbslot, S->status)
      if (mode == 0) FARWS_ARGS((k_far_ws<false, 0, FG, FWR>));
      else if (mode == 1) FARWS_ARGS((k_far_ws<true, 2, FG, FWR>));
      else FARWS_ARGS((k_far_ws<true, 3, FG, FWR>));
    });
  }
  swr_kt_end(S, KT_FAR);
  if (mode != 0) {
    swr_kt_begin(S, KT_BONDS);
    if (mode == 3) BOND_ARGS((k_bonds<true>));
    else BOND_ARGS((k_bonds<false>));
    swr_kt_end(S, KT_BONDS);
  }
#undef FARWS_ARGS
#undef BOND_ARGS
  HIP_CHECK(hipGetLastError());
  return SWR_OK;
}

// Autotuner hook: the average time of `reps` launches of the far pass (the
// fused far + bond-candidate + hbond form) in gatherer/writer shape sh.
// Each launch follows a Reset, as in a step (the pass appends to the hbond
// lists Reset starts); the caller re-runs the pair stages afterwards.
int swr_lists_time_far(swr_system *S, int sh, int reps, float *ms) {
  int rc = swr_quiesce(S);
  if (rc) return rc;
  const int N = S->N;
  if (N <= 0 || !S->far || !S->packed) return SWR_ERR_STATE;
  if ((size_t)N * MCAND > S->cand_cap) {
    if ((rc = swr_alloc(&S->cand, (size_t)S->Ncap * MCAND)) || (rc = swr_alloc(&S->cand_count, S->Ncap))) return rc;
    S->cand_cap = (size_t)S->Ncap * MCAND;
  }
  int *hb_count = S->counts + S->Ncap;
  std::vector<hipEvent_t> ev(2 * (size_t)std::max(reps, 1));
  for (auto &e : ev) HIP_CHECK(hipEventCreate(&e));
  for (int r = 0; r < reps; r++) {
    if ((rc = swr_lists_reset(S))) return rc;
    (void)hipEventRecord(ev[2 * r], S->stream);
    far_dispatch(sh, [&](auto shc) {
      constexpr int FG = FarShape<decltype(shc)::value>::FG, FWR = FarShape<decltype(shc)::value>::FWR;
      hipLaunchKernelGGL((k_far_ws<true, 2, FG, FWR>), dim3(div_up(N, FG)), dim3((FG + FWR) * SWR_WAVE), 0,
                         S->stream, S->n, N, S->dp, S->packed, S->voff, S->vlist, S->far, S->far_index, S->far_end,
                         S->cand, S->cand_count, S->Hindex, S->num_hbonds, S->hbond_index, S->hbond_end, S->hbonds,
                         hb_count, S->hbond_cap, S->hbslot, S->status);
    });
    (void)hipEventRecord(ev[2 * r + 1], S->stream);
  }
  HIP_CHECK(hipGetLastError());
  HIP_CHECK(hipStreamSynchronize(S->stream));
  double tot = 0.0;
  for (int r = 0; r < reps; r++) {
    float t = 0.f;
    HIP_CHECK(hipEventElapsedTime(&t, ev[2 * r], ev[2 * r + 1]));
    tot += t;
  }
  for (auto &e : ev) (void)hipEventDestroy(e);
  *ms = (float)(tot / std::max(reps, 1));
  return SWR_OK;
}

int swr_lists_estimate(swr_system *S) {
  int rc = swr_lists_run(S, 3);
  if (rc) return rc;
  hipLaunchKernelGGL(k_estimate, dim3(div_up(S->N, 256)), dim3(256), 0, S->stream, S->n, S->N, S->counts,
                     S->counts + S->Ncap, S->packed, S->dp, S->ctl.saferzone, S->num_bonds, S->num_hbonds);
  HIP_CHECK(hipGetLastError());
  return SWR_OK;
}

// Validate_Lists: next capacities and overflow flags; the status block
// (with the capacity totals Reset needs next step) is copied back
// asynchronously and read at the host's next sync.
int swr_lists_validate(swr_system *S) {
  const int n = S->n, N = S->N;
  swr_kt_begin(S, KT_VALIDATE);
  hipLaunchKernelGGL(k_validate, dim3(div_up(N, 256)), dim3(256), 0, S->stream, n, N, S->bond_index, S->counts,
                     S->num_bonds, S->Hindex, S->counts + S->Ncap, S->num_hbonds, S->ctl.saferzone, S->bond_cap,
                     S->status, S->next_totals);
  // the capacity totals travel back with the next sync (next step's Reset)
  hipLaunchKernelGGL(k_validate_end, dim3(1), dim3(SWR_WAVE), 0, S->stream, S->status, S->next_totals,
                     (int *)S->status_host);
  S->status_copy_queued = true;
  S->next_totals_known = false;
  swr_kt_end(S, KT_VALIDATE);
  HIP_CHECK(hipGetLastError());
  return SWR_OK;
}

// bond_mark of sort_bonds_C.  Enqueues the relaxation (one launch more than
// it took last time to find nothing to change, no host wait) and a copy of the
// per-launch change flags; swr_mark_settle checks them at the next sync and
// runs further launches only if the last one still changed a mark.
int swr_lists_mark(swr_system *S) {
  const int n = S->n, N = S->N;
  S->mark_launched = 0;
  if (N <= n) return SWR_OK;
  if (N - n <= MARK_BFS) {   // exact when it ends: nothing to check
    if (int rc = swr_reserve(&S->mark_up, S->cap_mark_up, 4 * (size_t)(N - n))) return rc;
    swr_kt_begin(S, KT_MARK);
    hipLaunchKernelGGL(k_mark_up, dim3(div_up(N - n, 256)), dim3(256), 0, S->stream, n, N, S->bond_index, S->bond_end,
                       S->bond_nbr, (ushort4 *)S->mark_up);
    if (N - n <= BFS_LDS)
      hipLaunchKernelGGL(k_mark_bfs<true>, dim3(1), dim3(BFS_T), 0, S->stream, n, N, S->bond_index, S->bond_end,
                         S->bond_nbr, (const ushort4 *)S->mark_up, S->bond_mark);
    else
      hipLaunchKernelGGL(k_mark_bfs<false>, dim3(1), dim3(BFS_T), 0, S->stream, n, N, S->bond_index, S->bond_end,
                         S->bond_nbr, (const ushort4 *)S->mark_up, S->bond_mark);
    swr_kt_end(S, KT_MARK);
    HIP_CHECK(hipGetLastError());
    return SWR_OK;
  }
  if (!S->mark_chg) {
    int rc = swr_alloc(&S->mark_chg, MARK_MAX_LAUNCH);
    if (rc) return rc;
    if (hipHostMalloc((void **)&S->mark_chg_host, sizeof(int) * MARK_MAX_LAUNCH, 0) != hipSuccess) {
      swr_set_error_msg("hipHostMalloc failed");
      return SWR_ERR_NOMEM;
    }
  }
  const int L = std::min(MARK_MAX_LAUNCH, std::max(2, S->mark_launch_hint + 2));
  swr_kt_begin(S, KT_MARK);
  for (int k = 0; k < L; k++)
    hipLaunchKernelGGL(k_bond_mark, dim3(div_up(N - n, MARK_T)), dim3(MARK_T), 0, S->stream, n, N, k, S->bond_index,
                       S->bond_end, S->bond_nbr, S->bond_mark, S->mark_chg);
  HIP_CHECK(hipMemcpyAsync(S->mark_chg_host, S->mark_chg, sizeof(int) * L, hipMemcpyDeviceToHost, S->stream));
  swr_kt_end(S, KT_MARK);
  HIP_CHECK(hipGetLastError());
  S->mark_launched = L;
  return SWR_OK;
}

// Finishes a pending relaxation: the flags copied at enqueue time are valid
// once the stream has passed them (call after a sync).  Converged when some
// launch changed nothing; otherwise relaxes further, synchronously.  Returns
// 1 when it gave up and raised SWR_F_MARK_DEPTH on the device.
int swr_mark_settle(swr_system *S) {
  if (S->mark_launched <= 0) return SWR_OK;
  const int n = S->n, N = S->N;
  int launch = S->mark_launched;
  S->mark_launched = 0;
  for (int k = 0; k < launch; k++)
    if (S->mark_chg_host[k] == 0) {
      S->mark_launch_hint = k;
      return SWR_OK;
    }
  while (launch < MARK_MAX_LAUNCH) {
    const int l0 = launch;
    for (int k = 0; k < 4 && launch < MARK_MAX_LAUNCH; k++, launch++)
      hipLaunchKernelGGL(k_bond_mark, dim3(div_up(N - n, MARK_T)), dim3(MARK_T), 0, S->stream, n, N, launch,
                         S->bond_index, S->bond_end, S->bond_nbr, S->bond_mark, S->mark_chg);
    HIP_CHECK(hipMemcpyAsync(S->mark_chg_host + l0, S->mark_chg + l0, sizeof(int) * (launch - l0),
                             hipMemcpyDeviceToHost, S->stream));
    HIP_CHECK(hipStreamSynchronize(S->stream));
    for (int k = l0; k < launch; k++)
      if (S->mark_chg_host[k] == 0) {
        S->mark_launch_hint = k;
        return SWR_OK;
      }
  }
  hipLaunchKernelGGL(k_set_flag, dim3(1), dim3(1), 0, S->stream, S->status, (unsigned)SWR_F_MARK_DEPTH);
  HIP_CHECK(hipGetLastError());
  HIP_CHECK(hipStreamSynchronize(S->stream));
  return 1;
}

// Bookkeeping after the host has synchronised with the system's stream.
// Returns 1 when it changed the device status block after that sync.
int swr_after_sync(swr_system *S) {
  if (S->status_copy_queued) {
    S->status_copy_queued = false;
    S->next_totals_known = true;
  }
  return swr_mark_settle(S) == 1;
}

// Waits for and finishes a pending relaxation before list arrays are
// reallocated or the atoms change.
int swr_quiesce(swr_system *S) {
  if (S->mark_launched <= 0) return SWR_OK;
  HIP_CHECK(hipStreamSynchronize(S->stream));
  (void)swr_after_sync(S);
  return SWR_OK;
}
