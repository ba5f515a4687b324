// Fused LJ + Ewald real-space pair kernel over the full Verlet rows, plus the
// cell-walk kernels (LJ when its cutoff exceeds the list guarantee, the
// real-space energy and point queries).  No atomics: every atom gathers its own
// row, its lanes' sums meet in a fixed tree, so FP64 results are reproducible run
// to run.
// No MFMA: the pair loop is a gather over irregular rows, not a contraction.
#include <algorithm>
#include <cstring>

#include "cav_internal.hpp"

namespace cav {

__device__ __forceinline__ double dot_rn_p(double a, double b, double c)
{
  // (a*a + b*b) + c*c with every product and sum rounded on its own, as the
  // reference's Vector::operator* (hipcc contracts to FMA by default)
#pragma clang fp contract(off)
  return (a * a + b * b) + c * c;
}

// erfc(x) = t * P(t) * exp(-x^2), t = 1/(1 + p x): the Hastings form of
// Abramowitz & Stegun 7.1.26 with a degree-8 polynomial whose coefficients
// were fitted here by weighted least squares on [0, 6] (relative error 1.3e-8
// in exact arithmetic, 2.6e-7 evaluated in FP32).  exp(-x^2) is shared with the
// Gaussian term of the Ewald force.
__device__ __forceinline__ float erfc_hastings(float x, float expmx2)
{
  const float t = __builtin_amdgcn_rcpf(fmaf(0.47047f, x, 1.0f));  // v_rcp_f32, 1 ulp
  float p = -5.325673686e-02f;
  p = fmaf(p, t, 2.980402004e-01f);
  p = fmaf(p, t, -6.267941092e-01f);
  p = fmaf(p, t, 5.387638720e-01f);
  p = fmaf(p, t, -1.765473040e-01f);
  p = fmaf(p, t, 2.700992388e-01f);
  p = fmaf(p, t, 2.166366678e-01f);
  p = fmaf(p, t, 2.677430713e-01f);
  p = fmaf(p, t, 2.653150927e-01f);
  return t * p * expmx2;
}

struct PairArgs {
  int n, nt, cap;
  const double *x, *y, *z, *q, *minv;
  const int *type, *id, *mol, *nl, *nn;
  const int *order;   // owned atoms in cell order
  const double4 *xq;  // packed (x, y, z, q) of owned + ghost atoms
  const int2 *tid;    // packed (type, id)
  // LJ per type pair: coef(r) = -c12 r^-14 + c6 r^-8 + cshift
  const double *c12, *c6, *cshift;
  double lj_rc2;
  // Ewald real space
  EwaldAlpha al;
  double ke, two_a_rpi;
  const double *lambda;
  double *ax, *ay, *az;
  double *part;
  int accumulate;  // add into the acceleration instead of overwriting it
  RepGrid reps;  // batched replicas, or none
  // rows as bin-order slots (or nullptr): neighbours are then read from the
  // bin-ordered copies, where the neighbours of cell-ordered atoms lie close
  // together, with the atom index from the list build's bin order
  const int *nlb;
  const double4 *xqs;  // slot_record
  const int *litems;
  const double *qtype;  // charge per type
};

// Neighbours whose loads a lane issues together in the row-gather kernel.
// Measured with 4 / 5 / 6 / 8 (us): mixed, 262144 ions 104 / 101 / 104 / 114, 256
// replicas 276 / 271 / 273 / 283; FP64 with 2 / 3 / 4: 65536 ions 36.0 / 36.0 /
// 36.2 in order, 120 / 128 / 128 beside Ewald_k (its math needs the registers).
template <typename T>
constexpr int pair_u() { return sizeof(T) == 8 ? 2 : 5; }

// LJ per type pair (c12, c6, cshift) staged in LDS as T at kernel start: 3 nt^2
// values, a pair's side by side, converted once instead of per pair.
template <typename T>
__device__ __forceinline__ void stage_lj_tables(const PairArgs &a, int nt2, T *tab)
{
  for (int t = threadIdx.x; t < nt2; t += blockDim.x) {
    tab[3 * t] = (T)a.c12[t];
    tab[3 * t + 1] = (T)a.c6[t];
    tab[3 * t + 2] = (T)a.cshift[t];
  }
}

template <typename T>
__device__ __forceinline__ T recip(T x)
{
  if constexpr (sizeof(T) == 8)
    return 1.0 / x;
  else
    return __builtin_amdgcn_rcpf(x);  // mixed form: v_rcp_f32, 1 ulp
}

// Force coefficient of one listed pair (force on i = coef * (r_j - r_i)), in T =
// double (the reference's arithmetic) or float (mixed form); adds the pair's
// Ewald_r virial term for the reference's list entries.
//   LJ: lj_cell_list.cpp:141-142 skips dr^2 > rc^2; shifted-force coefficients.
//   ER: electrostatic_ewald_r.cpp:162-211, every listed pair, exact zero skipped,
//       lambda of same-molecule pairs (0 skips the pair).
// p: the type-pair entry as the reference indexes it, [lower owned index][partner]
// (pair_entry); counted: the virial's share, once per reference list entry
// (owned j > i or a ghost, and j > i for a ghost too) with id_i < id_j.
template <typename T, bool LJ, bool ER, bool LAM>
__device__ __forceinline__ T pair_coef(const PairArgs &a, const T *tab, int p, bool counted,
                                       bool same_mol, T qi, T keqi, T qj, const double4 &pi4,
                                       double xj, double yj, double zj, T &dx, T &dy, T &dz,
                                       double &vir)
{
  const double dxd = xj - pi4.x, dyd = yj - pi4.y, dzd = zj - pi4.z;
  dx = (T)dxd;
  dy = (T)dyd;
  dz = (T)dzd;
  T r2;
  if constexpr (sizeof(T) == 8)
    r2 = dot_rn_p(dxd, dyd, dzd);  // the exact rounding order of the reference test
  else
    r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
  T coef = 0;
  if constexpr (LJ) {
    if (!(r2 > (T)a.lj_rc2)) {
      const T ri2 = recip(r2);
      const T ri4 = ri2 * ri2, ri8 = ri4 * ri4;
      coef += -tab[3 * p] * (ri8 * ri4 * ri2) + tab[3 * p + 1] * ri8 + tab[3 * p + 2];
    }
  }
  if constexpr (ER) {
    // (a distance whose square is not zero is not)
    if (r2 != 0 || !(dxd == 0 && dyd == 0 && dzd == 0)) {
      T lam = 1;
      bool skip = false;
      if constexpr (LAM) {
        if (same_mol) {
          const T l = (T)a.lambda[p];
          if (l == 0) skip = true;
          lam = l;
        }
      }
      if (!skip) {
        T ce;
        if constexpr (sizeof(T) == 8) {
          double e, ec, ri2;
          ewald_real(r2, a.al, e, ec, ri2);
          const double s = fma(a.two_a_rpi, e, ec) * ri2;
          ce = -lam * a.ke * (double)qi * qj * s;
        } else {
          const float rinv = __frsqrt_rn(r2);
          const float rn = r2 * rinv;
          const float e = __expf(-(float)a.al.a2 * r2);
          const float ec = erfc_hastings((float)a.al.alpha * rn, e);
          const float s = fmaf((float)a.two_a_rpi, e, ec * rinv) * (rinv * rinv);
          ce = -lam * keqi * qj * s;
        }
        coef += ce;
        if (counted) vir += -(double)ce * (double)r2;
      }
    }
  }
  return coef;
}

__device__ __forceinline__ int pair_entry(bool lower, int ti, int tj, int nt)
{
  return lower ? __mul24(tj, nt) + ti : __mul24(ti, nt) + tj;
}

// Deterministic per-block sum of the virial: fixed shuffle tree per wave, then
// the waves in order.
__device__ __forceinline__ void block_virial(double vir, double *part)
{
  __shared__ double s_red[kBlock / 64];
  for (int o = 32; o > 0; o >>= 1) vir += __shfl_xor(vir, o, 64);
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = vir;
  __syncthreads();
  if (threadIdx.x == 0) {
    double v = 0.0;
    for (int w = 0; w < kBlock / 64; ++w) v += s_red[w];
    *part = v;
  }
}

// Row-gather pair kernel: LPA lanes share one atom's row (coalesced row
// reads, balanced work); each lane fetches pair_u<T>() indices, then their (x, y,
// z, q) and (type, id), before computing, so the gathers overlap.  The
// partial forces of an atom's lanes are summed with a fixed shuffle tree, so
// FP64 results stay reproducible.
//
// Gather instructions bound it (N=262144 mixed: the address units take about 24
// clocks for each, of whatever width, 73% of their time; the vector units are
// half busy).  So a slot is one record of two 16-byte loads: the charge is
// looked up by type, and with ids that ascend with the atom index
// (ROWS_SLOTS_ASC) images and the order of a pair are told by id, without the
// slot's atom.  The next row entries are fetched while these are used.  Before,
// with (x, y, z, q), (type, id) and the atom gathered apart (us): mixed, 262144
// ions 110, 256 replicas (540000 atoms, rho 0.2 to 0.8) 381; FP64, 65536 ions
// 41; now 92, 271 and 36.  Planes x, y, z instead of records (a third fewer
// bytes through the L1, but as many instructions) gained nothing.
enum { ROWS_INDEX, ROWS_SLOTS, ROWS_SLOTS_ASC };

template <typename T, bool LJ, bool ER, bool LAM, int ROWS, int LPA = kLPA>
__global__ __launch_bounds__(kBlock) void k_pairs(PairArgs a)
{
  extern __shared__ double dyn_pair[];
  T *tab = reinterpret_cast<T *>(dyn_pair);
  const int nt2 = LJ ? a.nt * a.nt : 0;
  T *qt = tab + 3 * nt2;
  int part_at = blockIdx.x, blk32 = blockIdx.x;
  if (a.reps.rep) {  // the workgroup's replica: shift every array to it
    int blocks;
    const int rr = rep_block(a.reps, blk32, blocks);
    if (rr < 0) return;
    const RepDev &r = a.reps.rep[rr];
    part_at = blk32;
    const int base = r.base, obase = r.obase;
    a.n = r.n;
    a.xq += base;
    a.tid += base;
    a.nn += obase;
    if (a.order) a.order += obase;
    if constexpr (ROWS != ROWS_INDEX) {
      a.nlb += (long)obase * a.cap;
      a.xqs += base;
      a.litems += base;
    }
    a.ax += obase;
    a.ay += obase;
    a.az += obase;
    a.part += r.pbase;
  }
  long blk = blk32;
  if (!a.reps.rep) {
    // XCD-aware order (the grid is a multiple of 8 and dispatch is round-robin
    // over the 8 XCDs): each XCD gets a contiguous run of cell-ordered atoms,
    // so neighbouring atoms' gathers share one L2
    const long per = gridDim.x >> 3;
    blk = (long)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
  }
  const long gid = blk * kBlock + threadIdx.x;
  const int t = (int)(gid / LPA), sub = (int)(gid % LPA);
  double vir = 0.0;
  T fx = 0, fy = 0, fz = 0;
  int i = 0, ti = 0, cnt = 0, moli = 0;
  double4 pi4 = make_double4(0, 0, 0, 0);
  int2 tii = make_int2(0, 0);
  if (t < a.n) {
    i = a.order ? a.order[t] : t;
    pi4 = a.xq[i];
    tii = a.tid[i];
    moli = LAM ? a.mol[i] : 0;
    cnt = a.nn[i];
  }
  // (staged while the atom's own loads are under way)
  stage_lj_tables(a, nt2, tab);
  if constexpr (ROWS != ROWS_INDEX)
    for (int q = threadIdx.x; q < a.nt; q += kBlock) qt[q] = (T)a.qtype[q];
  __syncthreads();
  if (t < a.n) {
    ti = tii.x;
    const T qi = (T)pi4.w;
    const T keqi = (T)(a.ke) * qi;
    const int *row = (ROWS != ROWS_INDEX ? a.nlb : a.nl) + (long)i * a.cap;
    constexpr int U = pair_u<T>();
    // entries past the row (read all the same, rows are padded) stand for slot 0
    // and are skipped below; the next entries are fetched while these are used
    int next[U];
#pragma unroll
    for (int u = 0; u < U; ++u) next[u] = row[sub + u * LPA];
    for (int k0 = sub; k0 < cnt; k0 += U * LPA) {
      int jj[U];
      double xj[U], yj[U], zj[U];
      T qj[U];
      int2 tj[U];
#pragma unroll
      for (int u = 0; u < U; ++u) jj[u] = next[u];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const unsigned k = k0 + u * LPA < cnt ? jj[u] : 0;
        if constexpr (ROWS != ROWS_INDEX) {
          const double4 v = a.xqs[k];
          xj[u] = v.x;
          yj[u] = v.y;
          zj[u] = v.z;
          tj[u] = make_int2(__double2loint(v.w), __double2hiint(v.w));
          if constexpr (ROWS == ROWS_SLOTS) jj[u] = a.litems[k];
        } else {
          const double4 v = a.xq[k];
          xj[u] = v.x;
          yj[u] = v.y;
          zj[u] = v.z;
          qj[u] = (T)v.w;
          tj[u] = a.tid[k];
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) next[u] = row[k0 + (U + u) * LPA];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (k0 + u * LPA >= cnt) break;
        const int type = ROWS != ROWS_INDEX ? tj[u].x & ~kImage : tj[u].x;
        if constexpr (ROWS != ROWS_INDEX) qj[u] = qt[type];
        bool lower, counted = tii.y < tj[u].y;
        if constexpr (ROWS == ROWS_SLOTS_ASC) {
          lower = !(tj[u].x & kImage) && tj[u].y < tii.y;
        } else {
          lower = jj[u] < i;
          counted = counted && jj[u] > i;
        }
        bool same_mol = false;
        if constexpr (LAM) same_mol = moli == a.mol[jj[u]];
        T dx, dy, dz;
        const T coef = pair_coef<T, LJ, ER, LAM>(a, tab, pair_entry(lower, ti, type, a.nt), counted,
                                                 same_mol, qi, keqi, qj[u], pi4, xj[u], yj[u], zj[u],
                                                 dx, dy, dz, vir);
        fx = fma(coef, dx, fx);
        fy = fma(coef, dy, fy);
        fz = fma(coef, dz, fz);
      }
    }
  }
#pragma unroll
  for (int o = 1; o < LPA; o <<= 1) {
    fx += __shfl_xor(fx, o, 64);
    fy += __shfl_xor(fy, o, 64);
    fz += __shfl_xor(fz, o, 64);
  }
  if (t < a.n && sub == 0) {
    const double mi = a.minv[ti];
    if (a.accumulate) {
      a.ax[i] += (double)fx * mi;
      a.ay[i] += (double)fy * mi;
      a.az[i] += (double)fz * mi;
    } else {
      a.ax[i] = (double)fx * mi;
      a.ay[i] = (double)fy * mi;
      a.az[i] = (double)fz * mi;
    }
  }
  block_virial(vir, a.part + part_at);
}

// ------------------------------------- force_field lj and short-range kernel --
//
// The Verlet-list force fields that are not fused into k_pairs: the reference's
// force_field lj (lj.cpp:341-483) and Electrostatic_short_range
// (electrostatic_short_range.cpp:133-258).  Each adds its own pass over the
// same full rows (the reference runs each field as its own loop), with the
// row-gather layout of k_pairs: kLPA lanes per atom, partial forces summed by
// a fixed shuffle tree, one virial partial per block.
struct ListArgs {
  // force_field lj per type pair ([row type][partner type]): coef(r) =
  // -c12 r^-14 + c6 r^-8 + cshift, pair skipped when r^2 > rc2 (rc2 < 0 for
  // eps = 0, which the reference skips)
  const double *ljl;  // [c12 | c6 | cshift | rc2] blocks of nt^2
  int ljl_ignore_intra, ljl_jump;
  double ljl_jump_tol;
  // Electrostatic_short_range
  double sr_rc, sr_rc2, sr_ke, sr_beta1, sr_ext[3];
  const double *sr_lambda;  // nt^2, or nullptr
};

// Force coefficient of one listed pair for the list-based fields.  The
// virial of each field counts the reference's list entries (owned j > i or a
// ghost) with id_i < id_j, from the field's own dr^2 (lj clamps it with
// jump_tol).
template <typename T, bool LJL, bool SR>
__device__ __forceinline__ T list_coef(const PairArgs &a, const ListArgs &b, int nt2, int i, int j,
                                       int ti, int idi, int moli, int molj, const int2 &tj, T qi,
                                       const double4 &pi4, const double4 &pj, T &dx, T &dy, T &dz,
                                       double &vir)
{
  const double dxd = pj.x - pi4.x, dyd = pj.y - pi4.y, dzd = pj.z - pi4.z;
  dx = (T)dxd;
  dy = (T)dyd;
  dz = (T)dzd;
  T r2;
  if constexpr (sizeof(T) == 8)
    r2 = dot_rn_p(dxd, dyd, dzd);
  else
    r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
  const int p = (j < a.n && j < i) ? tj.x * a.nt + ti : ti * a.nt + tj.x;
  const bool counted = (j >= a.n || j > i) && idi < tj.y;
  T coef = 0;
  if constexpr (LJL) {
    if (!(b.ljl_ignore_intra && moli == molj) && !(r2 > (T)b.ljl[3 * nt2 + p])) {
      T d2 = r2;
      if (b.ljl_jump && d2 < (T)b.ljl_jump_tol) d2 = (T)b.ljl_jump_tol;
      const T ri2 = recip(d2);
      const T ri4 = ri2 * ri2, ri8 = ri4 * ri4;
      const T cl = -(T)b.ljl[p] * (ri8 * ri4 * ri2) + (T)b.ljl[nt2 + p] * ri8 + (T)b.ljl[2 * nt2 + p];
      coef += cl;
      if (counted) vir += -(double)cl * (double)d2;
    }
  }
  if constexpr (SR) {
    T lam = 1;
    bool skip = false;
    if (b.sr_lambda && moli == molj) {
      const T l = (T)b.sr_lambda[p];
      if (l == 0) skip = true;
      lam = l;
    }
    if (!skip && r2 < (T)b.sr_rc2) {
      const T qj = (T)pj.w;
      T cs;
      if constexpr (sizeof(T) == 8) {
        const double rn = sqrt(r2);
        cs = -lam * b.sr_ke * (double)qi * qj / (r2 * rn) * (1.0 - pow(rn / b.sr_rc, b.sr_beta1));
      } else {
        const float rinv = __frsqrt_rn(r2);
        const float rn = r2 * rinv;
        const float sh = 1.0f - powf(rn * (float)(1.0 / b.sr_rc), (float)b.sr_beta1);
        cs = -lam * (float)b.sr_ke * qi * qj * (rinv * rinv * rinv) * sh;
      }
      coef += cs;
      if (counted) vir += -(double)cs * (double)r2;
    }
  }
  return coef;
}

template <typename T, bool LJL, bool SR>
__global__ __launch_bounds__(kBlock) void k_pairs_list(PairArgs a, ListArgs b)
{
  const int nt2 = a.nt * a.nt;
  const long per = gridDim.x >> 3;  // XCD-aware order, as k_pairs
  const long blk = (long)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
  const long gid = blk * kBlock + threadIdx.x;
  const int t = (int)(gid / kLPA), sub = (int)(gid % kLPA);
  double vir = 0.0;
  T fx = 0, fy = 0, fz = 0;
  int i = 0, ti = 0;
  T qi = 0;
  if (t < a.n) {
    i = a.order ? a.order[t] : t;
    const double4 pi4 = a.xq[i];
    const int2 tii = a.tid[i];
    ti = tii.x;
    const int moli = a.mol[i];
    qi = (T)pi4.w;
    const int cnt = a.nn[i];
    const int *row = a.nl + (long)i * a.cap;
    constexpr int U = 2;
    for (int k0 = sub; k0 < cnt; k0 += U * kLPA) {
      int jj[U];
      double4 pj[U];
      int2 tj[U];
      int mj[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + u * kLPA;
        jj[u] = k < cnt ? row[k] : -1;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = jj[u] < 0 ? i : jj[u];
        pj[u] = a.xq[j];
        tj[u] = a.tid[j];
        mj[u] = a.mol[j];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (jj[u] < 0) break;
        T dx, dy, dz;
        const T coef = list_coef<T, LJL, SR>(a, b, nt2, i, jj[u], ti, tii.y, moli, mj[u], tj[u], qi,
                                             pi4, pj[u], dx, dy, dz, vir);
        fx = fma(coef, dx, fx);
        fy = fma(coef, dy, fy);
        fz = fma(coef, dz, fz);
      }
    }
  }
#pragma unroll
  for (int o = 1; o < kLPA; o <<= 1) {
    fx += __shfl_xor(fx, o, 64);
    fy += __shfl_xor(fy, o, 64);
    fz += __shfl_xor(fz, o, 64);
  }
  if (t < a.n && sub == 0) {
    const double mi = a.minv[ti];
    double ex = 0, ey = 0, ez = 0;
    if constexpr (SR) {  // the external field, once per atom after its pairs
      ex = b.sr_ext[0] * (double)qi * mi;
      ey = b.sr_ext[1] * (double)qi * mi;
      ez = b.sr_ext[2] * (double)qi * mi;
    }
    if (a.accumulate) {
      a.ax[i] += (double)fx * mi + ex;
      a.ay[i] += (double)fy * mi + ey;
      a.az[i] += (double)fz * mi + ez;
    } else {
      a.ax[i] = (double)fx * mi + ex;
      a.ay[i] = (double)fy * mi + ey;
      a.az[i] = (double)fz * mi + ez;
    }
  }
  block_virial(vir, a.part + blockIdx.x);
}

// ----------------------------------------------------- cell-staged pair kernel --
//
// One workgroup per cell: the cell's de-duplicated 27-stencil is staged in LDS
// in the order the list build walked it (stencil cells in order, each in bin
// order), from the bin-ordered copies (x, y, z, q) and (type, id) refreshed
// every step; each Verlet entry carries its position in that order, so every
// j of the cell's owned atoms is an LDS read.  Lanes per atom adapt to the
// cell's owned count; the partial forces of an atom's lanes are summed with a
// fixed shuffle tree.  A cell whose stencil exceeds the LDS tile falls back to
// gathering its rows from the global copies.  The tile is sized per launch
// from the largest stencil met so far (a flag word the kernel raises).
constexpr int kPairCand = 1024;
constexpr int kPairLds = sizeof(double4) + sizeof(int2) + sizeof(int);  // bytes per staged atom

struct CellPairArgs {
  int nbins, cap, seen;
  const int *start, *st_off, *st, *items;
  const double4 *xqs;
  const int2 *tids;
  const unsigned short *nll;
  int *flags;
};

template <typename T, bool LJ, bool ER>
__global__ __launch_bounds__(kBlock) void k_pairs_cells(PairArgs a, CellPairArgs ca)
{
  // staged stencil: (x, y, z, q)[cap], then (type, id)[cap], then slot index[cap],
  // then the LJ tables (3 nt^2 values of T)
  extern __shared__ double4 lds[];
  double4 *lq = lds;
  int2 *lt = reinterpret_cast<int2 *>(lq + ca.cap);
  int *lj = reinterpret_cast<int *>(lt + ca.cap);
  T *tab = reinterpret_cast<T *>(lj + ca.cap);
  const int nt2 = LJ ? a.nt * a.nt : 0;
  stage_lj_tables(a, nt2, tab);
  __shared__ int s_base[32], s_off[33];
  __shared__ int sh_nc, sh_self;
  __shared__ T s_f[3][kBlock];  // partial forces of the atoms' lanes
  const long per = gridDim.x >> 3;  // XCD-aware cell order, as k_pairs
  const int b = (int)((long)(blockIdx.x & 7) * per + (blockIdx.x >> 3));
  double vir = 0.0;
  if (b < ca.nbins) {
    const int s0 = ca.start[b], e0 = ca.start[b + 1];
    const int sb = ca.st_off[b], ns = ca.st_off[b + 1] - sb;  // <= 27 stencil cells
    if (threadIdx.x < 64) {
      // the stencil's cell ranges and their running offsets in staging order
      const int lane = threadIdx.x;
      if (lane == 0) sh_self = -1;
      int cell = -1, cb = 0, cn = 0;
      if (lane < ns) {
        cell = ca.st[sb + lane];
        cb = ca.start[cell];
        cn = ca.start[cell + 1] - cb;
      }
      int incl = cn;
      for (int o = 1; o < 32; o <<= 1) {
        const int v = __shfl_up(incl, o, 64);
        if (lane >= o) incl += v;
      }
      if (lane < ns) {
        s_base[lane] = cb;
        s_off[lane + 1] = incl;
        if (cell == b) sh_self = incl - cn;  // this cell's own atoms in the staging order
      }
      if (lane == 0) s_off[0] = 0;
      if (lane == (ns > 0 ? ns - 1 : 0)) {
        sh_nc = ns > 0 ? incl : 0;
        if (ns > 0 && incl > ca.seen) atomicMax(ca.flags + F_MAXST, incl);
      }
    }
    // owned atoms come first in a sorted bin
    int no = 0;
    for (int t0 = s0; t0 < e0; t0 += kBlock) {
      const int t = t0 + (int)threadIdx.x;
      no += __syncthreads_count(t < e0 && ca.items[t] < a.n);
    }
    __syncthreads();
    const int nc = sh_nc, self = sh_self;
    const bool staged = nc <= ca.cap && self >= 0;
    if (no > 0) {
      // lanes per atom: as many as fill the block (any count; the partial
      // forces are summed through LDS in lane order)
      const int L = no >= kBlock ? 1 : (kBlock / no < 64 ? kBlock / no : 64);
      const int per_pass = kBlock / L;
      const int slot = threadIdx.x / L, sub = threadIdx.x - slot * L;
      constexpr int U = 4;  // neighbour indices fetched together
      for (int a0 = 0; a0 < no; a0 += per_pass) {
        const int ai = a0 + slot;
        const bool act = slot < per_pass && ai < no;
        // the row's first indices are fetched before the stencil is staged:
        // rows hold cap entries, so reads below cap stay in the row
        const int i = act ? ca.items[s0 + ai] : 0;
        const long row = (long)i * a.cap;
        const int cnt = act ? a.nn[i] : 0;
        int loc[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int k = sub + u * L;
          loc[u] = (act && k < a.cap) ? (staged ? (int)ca.nll[row + k] : a.nl[row + k]) : 0;
        }
        if (a0 == 0) {
          if (staged) {
            for (int t = threadIdx.x; t < nc; t += kBlock) {
              int c = 0;
              while (s_off[c + 1] <= t) ++c;
              const int src = s_base[c] + t - s_off[c];
              lq[t] = ca.xqs[src];
              lt[t] = ca.tids[src];
              lj[t] = ca.items[src];
            }
          }
          __syncthreads();
        }
        T fx = 0, fy = 0, fz = 0;
        int ti = 0;
        if (act) {
          double4 pi4;
          int2 tii;
          if (staged) {
            pi4 = lq[self + ai];
            tii = lt[self + ai];
          } else {
            pi4 = a.xq[i];
            tii = a.tid[i];
          }
          ti = tii.x;
          const T qi = (T)pi4.w, keqi = (T)a.ke * qi;
          for (int k0 = sub; k0 < cnt; k0 += U * L) {
            if (k0 != sub) {
#pragma unroll
              for (int u = 0; u < U; ++u) {
                const int k = k0 + u * L;
                loc[u] = k < cnt ? (staged ? (int)ca.nll[row + k] : a.nl[row + k]) : 0;
              }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
              if (k0 + u * L >= cnt) break;
              int j;
              double4 pj;
              int2 tj;
              if (staged) {
                pj = lq[loc[u]];
                tj = lt[loc[u]];
                j = lj[loc[u]];
              } else {
                j = loc[u];
                pj = a.xq[j];
                tj = a.tid[j];
              }
              T dx, dy, dz;
              const T coef = pair_coef<T, LJ, ER, false>(
                  a, tab, pair_entry(j < i, ti, tj.x, a.nt), j > i && tii.y < tj.y, false, qi, keqi,
                  (T)pj.w, pi4, pj.x, pj.y, pj.z, dx, dy, dz, vir);
              fx = fma(coef, dx, fx);
              fy = fma(coef, dy, fy);
              fz = fma(coef, dz, fz);
            }
          }
        }
        s_f[0][threadIdx.x] = fx;
        s_f[1][threadIdx.x] = fy;
        s_f[2][threadIdx.x] = fz;
        __syncthreads();
        if (act && sub == 0) {
          fx = fy = fz = 0;
          for (int l = 0; l < L; ++l) {
            fx += s_f[0][threadIdx.x + l];
            fy += s_f[1][threadIdx.x + l];
            fz += s_f[2][threadIdx.x + l];
          }
          const double mi = a.minv[ti];
          if (a.accumulate) {
            a.ax[i] += (double)fx * mi;
            a.ay[i] += (double)fy * mi;
            a.az[i] += (double)fz * mi;
          } else {
            a.ax[i] = (double)fx * mi;
            a.ay[i] = (double)fy * mi;
            a.az[i] = (double)fz * mi;
          }
        }
        __syncthreads();
      }
    }
  }
  block_virial(vir, a.part + blockIdx.x);
}

// Packed copies for the pair gathers: (x, y, z, q) and (type, id).
__global__ void k_pack(int n, long cap_total, const double *x, const double *y, const double *z,
                       const double *q, const int *type, const int *id, const int *flags,
                       double4 *xq, int2 *tid, const int *binpos, double4 *xqs, int2 *tids,
                       int records)
{
  const long a = (long)blockIdx.x * kBlock + threadIdx.x;
  if (a >= (long)n + flags[F_NGHOST] || a >= cap_total) return;
  const double4 v = make_double4(x[a], y[a], z[a], q[a]);
  const int2 w = make_int2(type[a], id[a]);
  xq[a] = v;
  tid[a] = w;
  // the same in bin order, for the cell-staged pair kernel or as records for
  // the row kernel: only slots that existed at the last list build
  // have a bin position
  if (binpos && a < (long)n + flags[F_NGHOST_OLD]) {
    const int t = binpos[a];
    if (t >= 0 && t < cap_total) {
      xqs[t] = records ? slot_record(v, w, a >= n) : v;
      if (!records) tids[t] = w;
    }
  }
}

__global__ void k_reduce_part(int count, const double *part, double *out, int add)
{
  __shared__ double red[kBlock];
  double s = 0;
  for (int i = threadIdx.x; i < count; i += kBlock) s += part[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = kBlock / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = add ? *out + red[0] : red[0];
}

int reduce_partials(cav_ctx *c, int count, int slot, bool add)
{
  if (count > c->npart) return fail(c, CAV_ERR_STATE, "partial-sum buffer smaller than the grid");
  k_reduce_part<<<1, kBlock, 0, c->stream>>>(count, c->part, c->scal + slot, add ? 1 : 0);
  CAV_HIP(hipGetLastError());
  return CAV_OK;
}

static PairArgs pair_args(cav_ctx *c)
{
  PairArgs a;
  a.accumulate = 0;
  a.n = c->n;
  a.nt = c->nt;
  a.cap = c->nl_cap;
  a.x = c->x;
  a.y = c->y;
  a.z = c->z;
  a.q = c->q;
  a.minv = c->d_minv;
  a.type = c->type;
  a.id = c->id;
  a.mol = c->mol;
  a.nl = c->nl;
  a.nn = c->nn;
  a.order = c->order;
  a.xq = c->xq;
  a.tid = c->tid;
  const int nt2 = c->nt * c->nt;
  a.c12 = c->d_eps;           // laid out as [c12 | c6 | cshift] blocks, see upload
  a.c6 = c->d_eps + nt2;
  a.cshift = c->d_eps + 2 * nt2;
  a.lj_rc2 = c->lj_rc * c->lj_rc;
  a.al = ewald_alpha(c->er_alpha);
  a.ke = c->er_ke;
  a.two_a_rpi = 2 * c->er_alpha * CAV_PIS_INV;
  a.lambda = c->d_lambda;
  a.ax = c->ax;
  a.ay = c->ay;
  a.az = c->az;
  a.part = c->part;
  a.nlb = nullptr;
  a.xqs = nullptr;
  a.litems = nullptr;
  a.qtype = nullptr;
  return a;
}

static int pair_grid(const cav_ctx *c, int lpa = kLPA)
{
  return (grid_for((long)c->n * lpa) + 7) / 8 * 8;
}

// Lanes per atom of the row pair kernel (through slots and through indices
// alike, so that both sum in one order): more where the chip has room, since a
// lane's serial groups of gathers are then its time.  Measured with 8 / 16 / 32 lanes (us): 256 LJ atoms 8.5 / 6.2 / 5.1, 4000 9.1 /
// 6.5 / 6.0, 8000 ions (FP64) 14.0 / 13.5 / 11.8, 30011 (mixed) 19.3 / 19.4 /
// 24.0, 65536 (FP64) 101 / 112 / 118.
static int pair_lanes(const cav_ctx *c) { return c->n <= 16384 ? 32 : kLPA; }

int pair_blocks(const cav_ctx *c) { return pair_grid(c, pair_lanes(c)); }

// LDS of the row kernel: the LJ tables and the charges per type
template <typename T>
static size_t pair_lds(const PairArgs &a, bool lj)
{
  return sizeof(T) * ((lj ? 3 * a.nt * a.nt : 0) + a.nt);
}

template <typename T, int ROWS, int LPA>
static void launch_pairs_tr(cav_ctx *c, const PairArgs &a, bool lj, bool er)
{
  const int g = pair_grid(c, LPA);
  const size_t lds = pair_lds<T>(a, lj);
  if (lj && er)
    k_pairs<T, true, true, false, ROWS, LPA><<<g, kBlock, lds, c->stream>>>(a);
  else if (lj)
    k_pairs<T, true, false, false, ROWS, LPA><<<g, kBlock, lds, c->stream>>>(a);
  else
    k_pairs<T, false, true, false, ROWS, LPA><<<g, kBlock, lds, c->stream>>>(a);
}

// with the per-molecule lambda (of Ewald_r), which needs the neighbour's index
template <typename T, int ROWS, int LPA>
static void launch_pairs_tl(cav_ctx *c, const PairArgs &a, bool lj)
{
  const int g = pair_grid(c, LPA);
  const size_t lds = pair_lds<T>(a, lj);
  if (lj)
    k_pairs<T, true, true, true, ROWS, LPA><<<g, kBlock, lds, c->stream>>>(a);
  else
    k_pairs<T, false, true, true, ROWS, LPA><<<g, kBlock, lds, c->stream>>>(a);
}

// rows as bin-order slots (a.nlb) or as atom indices, each its own kernel
template <typename T, int LPA>
static void launch_pairs_tn(cav_ctx *c, const PairArgs &a, bool lj, bool er, bool lam)
{
  if (er && lam && a.nlb)
    launch_pairs_tl<T, ROWS_SLOTS, LPA>(c, a, lj);
  else if (er && lam)
    launch_pairs_tl<T, ROWS_INDEX, LPA>(c, a, lj);
  else if (!a.nlb)
    launch_pairs_tr<T, ROWS_INDEX, LPA>(c, a, lj, er);
  else if (c->ids_ascend)
    launch_pairs_tr<T, ROWS_SLOTS_ASC, LPA>(c, a, lj, er);
  else
    launch_pairs_tr<T, ROWS_SLOTS, LPA>(c, a, lj, er);
}

template <typename T>
static void launch_pairs_t(cav_ctx *c, const PairArgs &a, bool lj, bool er, bool lam)
{
  if (pair_lanes(c) == 32)
    launch_pairs_tn<T, 32>(c, a, lj, er, lam);
  else
    launch_pairs_tn<T, kLPA>(c, a, lj, er, lam);
}

// The cell-staged kernel runs on request (CAV_PAIRS_CELLS) where it applies:
// the cell-built list (its entries' staging positions), no per-molecule
// lambda.  Otherwise, and by default, the row-gather kernel runs (faster on
// the ion workloads measured at N=262144, rho=0.3: 0.165 vs 0.232 ms mixed).
// The row kernel reads neighbours through the list build's bin-order slots
// when the current list carries them (CAV_PAIRS_AUTO; lists built from cells).
bool sorted_rows(const cav_ctx *c)
{
  return c->pair_kind == CAV_PAIRS_AUTO && !c->all_atom_test && c->nlb && c->nlb_built;
}

bool cell_staged(const cav_ctx *c)
{
  return c->pair_kind == CAV_PAIRS_CELLS && c->from_cells && c->build_cells && !c->all_atom_test &&
         !c->lambda_set && c->nll && c->nll_built;
}

static int cell_grid(const cav_ctx *c) { return (c->nbins + 7) / 8 * 8; }

template <typename T>
static void launch_pairs_cells_t(cav_ctx *c, const PairArgs &a, bool lj, bool er)
{
  CellPairArgs ca;
  ca.nbins = c->nbins;
  ca.start = c->lstart;
  ca.st_off = c->d_st_off;
  ca.st = c->d_st;
  ca.items = c->litems;
  ca.xqs = c->xqs;
  ca.tids = c->tids;
  ca.nll = c->nll;
  ca.flags = c->flags;
  // LDS tile: the largest stencil met so far (last synchronised flags), in
  // steps of 64 atoms; cells beyond it gather from global memory and raise it
  const int seen = c->h_flags ? c->h_flags[F_MAXST] : 0;
  ca.seen = seen;
  ca.cap = seen > 0 ? std::min(kPairCand, (seen + 63) / 64 * 64) : kPairCand;
  const size_t lds = (size_t)ca.cap * kPairLds + 3 * sizeof(T) * a.nt * a.nt;
  const int g = cell_grid(c);
  if (lj && er)
    k_pairs_cells<T, true, true><<<g, kBlock, lds, c->stream>>>(a, ca);
  else if (lj)
    k_pairs_cells<T, true, false><<<g, kBlock, lds, c->stream>>>(a, ca);
  else
    k_pairs_cells<T, false, true><<<g, kBlock, lds, c->stream>>>(a, ca);
}

// The list-based fields (force_field lj, Electrostatic_short_range) on the
// current list, one pass for the fields in use; `accumulate` false overwrites
// the accelerations and the virial (this pass is then the first force of the
// step); `pack` first refreshes the packed copies (when no fused pair pass has
// packed them this step).
int launch_pairs_list(cav_ctx *c, bool want_ljl, bool want_sr, bool accumulate, bool pack)
{
  const bool ljl = want_ljl && c->ljl_on, sr = want_sr && c->sr_on;
  if (!ljl && !sr) return CAV_OK;
  if (pack) CAV_TRY(launch_pack(c));
  CAV_TRY(launch_nl_fill(c));
  PairArgs a = pair_args(c);
  a.accumulate = accumulate ? 1 : 0;
  ListArgs b;
  b.ljl = c->d_ljl;
  b.ljl_ignore_intra = c->ljl_ignore_intra;
  b.ljl_jump = c->ljl_jump;
  b.ljl_jump_tol = c->ljl_jump_tol;
  b.sr_rc = c->sr_rc;
  b.sr_rc2 = c->sr_rc * c->sr_rc;
  b.sr_ke = c->sr_ke;
  b.sr_beta1 = c->sr_beta + 1.0;
  for (int d = 0; d < 3; ++d) b.sr_ext[d] = c->sr_ext[d];
  b.sr_lambda = c->sr_lambda_set ? c->d_sr_lambda : nullptr;
  const int g = pair_grid(c);
  if (g > c->npart) return fail(c, CAV_ERR_STATE, "partial-sum buffer smaller than the pair grid");
  timer_begin(c, c->t_pair);
  if (c->precision == CAV_FP64) {
    if (ljl && sr)
      k_pairs_list<double, true, true><<<g, kBlock, 0, c->stream>>>(a, b);
    else if (ljl)
      k_pairs_list<double, true, false><<<g, kBlock, 0, c->stream>>>(a, b);
    else
      k_pairs_list<double, false, true><<<g, kBlock, 0, c->stream>>>(a, b);
  } else {
    if (ljl && sr)
      k_pairs_list<float, true, true><<<g, kBlock, 0, c->stream>>>(a, b);
    else if (ljl)
      k_pairs_list<float, true, false><<<g, kBlock, 0, c->stream>>>(a, b);
    else
      k_pairs_list<float, false, true><<<g, kBlock, 0, c->stream>>>(a, b);
  }
  timer_end(c, c->t_pair);
  CAV_HIP(hipGetLastError());
  return reduce_partials(c, g, 0, accumulate);
}

// Repacks (x, y, z, q) and (type, id) of the current owned atoms and ghosts
// for readers of the packed copies other than the pair kernels (the adjoint).
int launch_pack(cav_ctx *c)
{
  const long tot = (long)c->n + c->gcap;
  k_pack<<<grid_for(tot), kBlock, 0, c->stream>>>(c->n, tot, c->x, c->y, c->z, c->q, c->type,
                                                 c->id, c->flags, c->xq, c->tid, nullptr, nullptr,
                                                 nullptr, 0);
  CAV_HIP(hipGetLastError());
  return CAV_OK;
}

int launch_pairs(cav_ctx *c, bool want_lj, bool want_er, bool accumulate, bool packed, bool reduce)
{
  const bool lj = want_lj && c->lj_on && !c->lj_cellwalk, er = want_er && c->er_on;
  if (!lj && !er) return CAV_OK;
  PairArgs a = pair_args(c);
  a.accumulate = accumulate ? 1 : 0;
  const long tot = (long)c->n + c->gcap;
  const bool cells = cell_staged(c);
  // every block writes one virial partial: the buffer must cover the grid
  if ((cells ? cell_grid(c) : pair_blocks(c)) > c->npart)
    return fail(c, CAV_ERR_STATE, "partial-sum buffer smaller than the pair grid");
  const bool bins = !cells && sorted_rows(c);
  if (bins) {
    a.nlb = c->nlb;
    a.xqs = c->xqs;
    a.litems = c->litems;
    a.qtype = c->d_qtype;
  } else {
    CAV_TRY(launch_nl_fill(c));
  }
  if (!packed || !bins)
    k_pack<<<grid_for(tot), kBlock, 0, c->stream>>>(c->n, tot, c->x, c->y, c->z, c->q, c->type,
                                                 c->id, c->flags, c->xq, c->tid,
                                                 cells || bins ? c->binpos : nullptr, c->xqs,
                                                 c->tids, bins);
  timer_begin(c, c->t_pair);
  if (cells) {
    if (c->precision == CAV_FP64)
      launch_pairs_cells_t<double>(c, a, lj, er);
    else
      launch_pairs_cells_t<float>(c, a, lj, er);
  } else if (c->precision == CAV_FP64) {
    launch_pairs_t<double>(c, a, lj, er, c->lambda_set);
  } else {
    launch_pairs_t<float>(c, a, lj, er, c->lambda_set);
  }
  timer_end(c, c->t_pair);
  CAV_HIP(hipGetLastError());
  if (!reduce) return CAV_OK;
  return reduce_partials(c, cells ? cell_grid(c) : pair_blocks(c), 0, accumulate);
}

__global__ void k_zero_acc(int n, double *ax, double *ay, double *az)
{
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) ax[i] = ay[i] = az[i] = 0.0;
}

__global__ void k_zero_scalar(double *p) { *p = 0.0; }

__global__ void k_fill_d(double *p, long n, double v)
{
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void kb_zero_own(const RepDev *rep, double *ax, double *ay, double *az)
{
  const RepDev &r = rep[blockIdx.y];
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= r.n) return;
  ax[r.obase + i] = ay[r.obase + i] = az[r.obase + i] = 0.0;
}

int launch_zero_acc(cav_ctx *c)
{
  k_zero_acc<<<grid_for(c->n), kBlock, 0, c->stream>>>(c->n, c->ax, c->ay, c->az);
  k_zero_scalar<<<1, 1, 0, c->stream>>>(c->scal);
  CAV_HIP(hipGetLastError());
  return CAV_OK;
}

// --------------------------------------------------------------- cell walks --

struct CellArgs {
  int n;
  const double *x, *y, *z, *q;
  const int *type, *bin_of, *st_off, *st, *start, *items;
  const double4 *cpos;  // (x, y, z, index and slot) in bin order
  double lox, loy, loz, cinv;
  int nbx, nby, nbz;
};

__device__ __forceinline__ int cell_of(const CellArgs &c, double px, double py, double pz)
{
  int ix = (int)floor(xmul(xsub(px, c.lox), c.cinv));
  int iy = (int)floor(xmul(xsub(py, c.loy), c.cinv));
  int iz = (int)floor(xmul(xsub(pz, c.loz), c.cinv));
  ix = ix < 0 ? 0 : (ix >= c.nbx ? c.nbx - 1 : ix);
  iy = iy < 0 ? 0 : (iy >= c.nby ? c.nby - 1 : iy);
  iz = iz < 0 ? 0 : (iz >= c.nbz ? c.nbz - 1 : iz);
  return ix + c.nbx * iy + c.nbx * c.nby * iz;
}

static CellArgs cell_args(cav_ctx *c)
{
  CellArgs a;
  a.n = c->n;
  a.x = c->x;
  a.y = c->y;
  a.z = c->z;
  a.q = c->q;
  a.type = c->type;
  a.bin_of = c->bin_of;
  a.st_off = c->d_st_off;
  a.st = c->d_st;
  a.start = c->bin_start;
  a.items = c->bin_items;
  a.cpos = c->cpos;
  a.lox = c->lo[0];
  a.loy = c->lo[1];
  a.loz = c->lo[2];
  a.cinv = c->cinv;
  a.nbx = c->nb[0];
  a.nby = c->nb[1];
  a.nbz = c->nb[2];
  return a;
}

// Lj_cell_list::calculate_acceleration (lj_cell_list.cpp:85-175) as a gather:
// every owned j != i and every ghost in the 27 cells, skip dr^2 > rc^2.  Adds
// into the acceleration (the pair kernel, if any, has written it first).
__global__ void k_lj_cellwalk(CellArgs c, int nt, const double *c12, const double *c6,
                              const double *cshift, double rc2, const double *minv, double *ax,
                              double *ay, double *az)
{
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= c.n) return;
  const double xi = c.x[i], yi = c.y[i], zi = c.z[i];
  const int ti = c.type[i];
  const int b = c.bin_of[i];
  double fx = 0, fy = 0, fz = 0;
  for (int s = c.st_off[b]; s < c.st_off[b + 1]; ++s) {
    const int cell = c.st[s];
    for (int t = c.start[cell]; t < c.start[cell + 1]; ++t) {
      const int j = c.items[t];
      if (j == i) continue;
      const double dx = xsub(c.x[j], xi), dy = xsub(c.y[j], yi), dz = xsub(c.z[j], zi);
      const double r2 = dot_rn_p(dx, dy, dz);
      if (r2 > rc2) continue;
      const int tj = c.type[j];
      const int p = (j < c.n && j < i) ? tj * nt + ti : ti * nt + tj;
      const double ri2 = 1.0 / r2, ri4 = ri2 * ri2, ri8 = ri4 * ri4;
      const double coef = -c12[p] * (ri8 * ri4 * ri2) + c6[p] * ri8 + cshift[p];
      fx += coef * dx;
      fy += coef * dy;
      fz += coef * dz;
    }
  }
  const double mi = minv[ti];
  ax[i] += fx * mi;
  ay[i] += fy * mi;
  az[i] += fz * mi;
}

int launch_lj_cellwalk(cav_ctx *c)
{
  const int nt2 = c->nt * c->nt;
  k_lj_cellwalk<<<grid_for(c->n), kBlock, 0, c->stream>>>(
      cell_args(c), c->nt, c->d_eps, c->d_eps + nt2, c->d_eps + 2 * nt2, c->lj_rc * c->lj_rc,
      c->d_minv, c->ax, c->ay, c->az);
  CAV_HIP(hipGetLastError());
  return CAV_OK;
}

// The cell walk's candidates: the 27-cell stencil of cell b flattened in order
// (each cell in bin order).  Lanes 0..ns-1 load their cell's range at once; the
// running offsets go to the wave's LDS (s_base, s_off).  Returns their number.
__device__ __forceinline__ int walk_ranges(const CellArgs &c, int b, int *s_base, int *s_off)
{
  const int lane = threadIdx.x & 63;
  const int sb = c.st_off[b], ns = c.st_off[b + 1] - sb;  // 1..27 cells
  int cb = 0, cn = 0;
  if (lane < ns) {
    const int cell = c.st[sb + lane];
    cb = c.start[cell];
    cn = c.start[cell + 1] - cb;
  }
  int incl = cn;
  for (int o = 1; o < 32; o <<= 1) {
    const int v = __shfl_up(incl, o, 64);
    if (lane >= o) incl += v;
  }
  if (lane < ns) {
    s_base[lane] = cb;
    s_off[lane + 1] = incl;
  }
  if (lane == 0) s_off[0] = 0;
  return __shfl(incl, ns - 1, 64);
}

// Candidate g of the flattened stencil as (x, y, z, q); `cell` walks forward
// with g (start at 0, ascending g).
__device__ __forceinline__ double4 walk_cand(const CellArgs &c, const int *s_base, const int *s_off,
                                             int g, int &cell)
{
  while (s_off[cell + 1] <= g) ++cell;
  double4 v = c.cpos[s_base[cell] + g - s_off[cell]];
  v.w = c.q[(int)(__double_as_longlong(v.w) & 0xffffffffll)];  // low word: the atom
  return v;
}

// Electrostatic_ewald_r::potential/field at a point (electrostatic_ewald_r/
// potential.cpp:30-86, field.cpp:31-96): every owned or ghost atom in the 27
// cells around the point's bin, no cutoff, exact-zero separation skipped.
// One wave per point, its lanes over the candidates, summed by a fixed shuffle
// tree.  The FP64 erfc and exp bound it; with one lane per point a lane walked
// all of its candidates by itself and a launch held np / 64 waves: 1000 points
// among 100 ions took 818 us, now 14 us.
__global__ __launch_bounds__(kBlock) void k_point_r(CellArgs c, int np, const double *pts,
                                                    EwaldAlpha al, double ke, double *field,
                                                    double *pot)
{
  __shared__ int s_base_[kBlock / 64][32], s_off_[kBlock / 64][33];
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int p = blockIdx.x * (kBlock / 64) + wv;
  if (p >= np) return;
  const double px = pts[3 * p], py = pts[3 * p + 1], pz = pts[3 * p + 2];
  int *s_base = s_base_[wv], *s_off = s_off_[wv];
  const int total = walk_ranges(c, cell_of(c, px, py, pz), s_base, s_off);
  __syncwarp();
  const double two_a_rpi = 2 * al.alpha * CAV_PIS_INV;
  double phi = 0, ex = 0, ey = 0, ez = 0;
  int cell = 0;
  for (int g = lane; g < total; g += 64) {
    const double4 v = walk_cand(c, s_base, s_off, g, cell);
    const double dx = px - v.x, dy = py - v.y, dz = pz - v.z;
    if (dx == 0 && dy == 0 && dz == 0) continue;
    const double d2 = dx * dx + dy * dy + dz * dz;
    double e, ec, ri2;
    ewald_real(d2, al, e, ec, ri2);
    const bool none = d2 >= 1e290;  // infinitely far: both terms vanish
    phi += none ? 0.0 : v.w * ec;
    const double sr = none ? 0.0 : fma(two_a_rpi, e, ec) * ri2;
    ex += v.w * sr * dx;
    ey += v.w * sr * dy;
    ez += v.w * sr * dz;
  }
  for (int o = 32; o > 0; o >>= 1) {
    phi += __shfl_xor(phi, o, 64);
    ex += __shfl_xor(ex, o, 64);
    ey += __shfl_xor(ey, o, 64);
    ez += __shfl_xor(ez, o, 64);
  }
  if (lane == 0) {
    pot[p] = phi * ke;
    field[3 * p] = ex * ke;
    field[3 * p + 1] = ey * ke;
    field[3 * p + 2] = ez * ke;
  }
}

static int point_part_r(cav_ctx *c, int np, const double *pts, double *field, double *pot)
{
  // the points are read from pinned host memory and the sums written there,
  // both once per point
  const bool staged = stage_room(c->stage, 7 * (size_t)np);
  double *d = c->stage.dev;
  if (staged)
    std::memcpy(c->stage.host, pts, sizeof(double) * 3 * np);
  else {
    CAV_TRY(point_room(c, 7 * (size_t)np, 0));
    d = c->pt_dev;
    CAV_HIP(hipMemcpyAsync(d, pts, sizeof(double) * 3 * np, hipMemcpyHostToDevice, c->stream));
  }
  double *df = d + 3 * (size_t)np, *dp = d + 6 * (size_t)np;
  if (np > 0)
    k_point_r<<<(np + kBlock / 64 - 1) / (kBlock / 64), kBlock, 0, c->stream>>>(
        cell_args(c), np, d, ewald_alpha(c->er_alpha), c->er_ke, df, dp);
  CAV_HIP(hipGetLastError());
  if (!staged && field)
    CAV_HIP(hipMemcpyAsync(field, df, sizeof(double) * 3 * np, hipMemcpyDeviceToHost, c->stream));
  if (!staged && pot)
    CAV_HIP(hipMemcpyAsync(pot, dp, sizeof(double) * np, hipMemcpyDeviceToHost, c->stream));
  CAV_HIP(hipStreamSynchronize(c->stream));
  if (staged && field) std::memcpy(field, c->stage.host + 3 * (size_t)np, sizeof(double) * 3 * np);
  if (staged && pot) std::memcpy(pot, c->stage.host + 6 * (size_t)np, sizeof(double) * np);
  return CAV_OK;
}

// The points in parts that fit the staging memory.
int point_field_r(cav_ctx *c, int np, const double *pts, double *field, double *pot)
{
  const int per = (int)(kStageMax / (7 * sizeof(double)));
  for (int p0 = 0; p0 == 0 || p0 < np; p0 += per)
    CAV_TRY(point_part_r(c, std::min(per, np - p0), pts + 3 * (size_t)p0,
                         field ? field + 3 * (size_t)p0 : nullptr, pot ? pot + p0 : nullptr));
  return CAV_OK;
}

// Stencil candidates staged per pass of the real-space energy (16 KB of LDS).
constexpr int kWalkCand = 512;

// Electrostatic_ewald_r::energy (electrostatic_ewald_r/energy.cpp:30-51): the
// potential of the cell walk at every owned atom times its charge.  One
// workgroup per cell: its stencil's candidates (x, y, z, q) are staged in LDS
// once for the cell's owned atoms, which the four waves take in turn, lanes
// over the candidates.  The FP64 erfc of every (atom, candidate) bounds it
// (about 500 an atom at rho = 0.3); one lane per atom, each walking its
// stencil through scattered loads, took 3395 us at N = 100003, this 395 and with
// the terms of cav_math.hpp 267 us.
__global__ __launch_bounds__(kBlock) void k_energy_r(CellArgs c, EwaldAlpha al, double *part)
{
  __shared__ double4 cand[kWalkCand];
  __shared__ int s_base[32], s_off[33];
  __shared__ double red[kBlock / 64];
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int b = blockIdx.x;
  const int s0 = c.start[b], e0 = c.start[b + 1];
  int no = 0;  // owned atoms come first in a sorted bin
  for (int t = s0; t < e0; t += 64)
    no += __popcll(__ballot(t + lane < e0 && c.items[t + lane] < c.n));
  double e = 0;
  if (no > 0) {
    // every wave forms the ranges (the values are the same)
    const int total = walk_ranges(c, b, s_base, s_off);
    __syncthreads();
    for (int m0 = 0; m0 < total; m0 += kWalkCand) {
      const int m = min(kWalkCand, total - m0);
      int cell = 0;
      for (int t = threadIdx.x; t < m; t += kBlock)
        cand[t] = walk_cand(c, s_base, s_off, m0 + t, cell);
      __syncthreads();
      for (int o = wv; o < no; o += kBlock / 64) {
        const int i = c.items[s0 + o];
        const double xi = c.x[i], yi = c.y[i], zi = c.z[i];
        double phi = 0;
        for (int t = lane; t < m; t += 64) {
          const double4 v = cand[t];
          const double dx = xi - v.x, dy = yi - v.y, dz = zi - v.z;
          if (dx == 0 && dy == 0 && dz == 0) continue;
          const double d2 = dx * dx + dy * dy + dz * dz;
          double e, ec, ri2;
          ewald_real(d2, al, e, ec, ri2);
          phi += d2 >= 1e290 ? 0.0 : v.w * ec;  // infinitely far: nothing
        }
        e += c.q[i] * phi;
      }
      __syncthreads();
    }
  }
  for (int o = 32; o > 0; o >>= 1) e += __shfl_xor(e, o, 64);
  if (lane == 0) red[wv] = e;
  __syncthreads();
  if (threadIdx.x == 0) part[b] = (red[0] + red[1]) + (red[2] + red[3]);
}

// Leaves twice the energy over k_electrostatic in scal[2] (energy.cpp:50 and
// potential.cpp:85).
int launch_energy_r(cav_ctx *c)
{
  if (c->nbins > c->npart) return fail(c, CAV_ERR_STATE, "partial-sum buffer smaller than the cell grid");
  k_energy_r<<<c->nbins, kBlock, 0, c->stream>>>(cell_args(c), ewald_alpha(c->er_alpha), c->part);
  CAV_HIP(hipGetLastError());
  return reduce_partials(c, c->nbins, 2);
}

// Shifted-force LJ energy over the full rows: each (i,j) entry carries half of
// U(r) = 4e[(s/r)^12 - (s/r)^6] + r^2 cshift/2 - (same at rc); every pair is
// seen from both ends (owned pairs twice in the full rows, periodic pairs once
// from each owned end through its ghost image).  kLPA lanes per atom and the
// packed (x, y, z, q), (type, id), as the pair kernel, four entries' loads
// issued together; the rows are read as the list build wrote them (`items`:
// bin-order slots to be looked up there, or null for atom indices).  Gather
// latency bounds it: 242 us at N = 100003 with one lane per atom, and 52 us
// to fill the index rows first; now 74 us, no fill.
__global__ __launch_bounds__(kBlock) void k_energy_lj(PairArgs a, const int *rows, const int *items,
                                                      const double *u12, const double *u6,
                                                      const double *uc, double *part)
{
  const long gid = (long)blockIdx.x * kBlock + threadIdx.x;
  const int t = (int)(gid / kLPA), sub = (int)(gid % kLPA);
  double e = 0;
  if (t < a.n) {
    const int i = a.order[t];
    const double4 pi = a.xq[i];
    const int ti = a.tid[i].x, cnt = a.nn[i];
    const int *row = rows + (long)i * a.cap;
    constexpr int U = 4;
    for (int k0 = sub; k0 < cnt; k0 += U * kLPA) {
      int j[U], tj[U];
      double4 pj[U];
#pragma unroll
      for (int u = 0; u < U; ++u) j[u] = k0 + u * kLPA < cnt ? row[k0 + u * kLPA] : -1;
      if (items) {
#pragma unroll
        for (int u = 0; u < U; ++u) j[u] = j[u] < 0 ? -1 : items[j[u]];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int jj = j[u] < 0 ? i : j[u];
        pj[u] = a.xq[jj];
        tj[u] = a.tid[jj].x;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const double r2 = dot_rn_p(pj[u].x - pi.x, pj[u].y - pi.y, pj[u].z - pi.z);
        if (j[u] < 0 || r2 > a.lj_rc2) continue;
        const int p = (j[u] < a.n && j[u] < i) ? tj[u] * a.nt + ti : ti * a.nt + tj[u];
        const double ri2 = 1.0 / r2, ri6 = ri2 * ri2 * ri2;
        e += 0.5 * (u12[p] * ri6 * ri6 - u6[p] * ri6 + 0.5 * a.cshift[p] * r2 - uc[p]);
      }
    }
  }
  __shared__ double red[kBlock / 64];
  for (int o = 32; o > 0; o >>= 1) e += __shfl_xor(e, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = e;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// Leaves the energy in scal[1].
int launch_energy_lj(cav_ctx *c)
{
  const bool slots = sorted_rows(c);
  if (!slots) CAV_TRY(launch_nl_fill(c));
  CAV_TRY(launch_pack(c));
  const int nt2 = c->nt * c->nt, g = pair_grid(c);
  if (g > c->npart) return fail(c, CAV_ERR_STATE, "partial-sum buffer smaller than the pair grid");
  k_energy_lj<<<g, kBlock, 0, c->stream>>>(pair_args(c), slots ? c->nlb : c->nl,
                                           slots ? c->litems : nullptr, c->d_eps + 3 * nt2,
                                           c->d_eps + 4 * nt2, c->d_eps + 5 * nt2, c->part);
  CAV_HIP(hipGetLastError());
  return reduce_partials(c, g, 1);
}


// ---------------------------------------------------------- batched replicas --

template <typename T>
static void batch_pairs_t(cav_batch *b, const PairArgs &a, dim3 g)
{
  const size_t lds = pair_lds<T>(a, b->lj_on);
  if (b->lj_on && b->er_on)
    k_pairs<T, true, true, false, ROWS_SLOTS_ASC><<<g, kBlock, lds, b->stream>>>(a);
  else if (b->lj_on)
    k_pairs<T, true, false, false, ROWS_SLOTS_ASC><<<g, kBlock, lds, b->stream>>>(a);
  else
    k_pairs<T, false, true, false, ROWS_SLOTS_ASC><<<g, kBlock, lds, b->stream>>>(a);
}

// LJ + Ewald_r accelerations of every replica (overwriting), virial partials
// per replica; the packed copies are those of batch_neighbor.
int batch_pairs(cav_batch *b)
{
  const dim3 g = batch_grid(b, b->pair_blocks);
  if (!b->lj_on && !b->er_on) {
    kb_zero_own<<<dim3(grid_for(b->maxn), b->B), kBlock, 0, b->stream>>>(b->d_rep, b->ax, b->ay,
                                                                        b->az);
    k_fill_d<<<grid_for((long)b->B * b->pair_blocks), kBlock, 0, b->stream>>>(
        b->part, (long)b->B * b->pair_blocks, 0.0);
  } else {
    PairArgs a;
    a.n = 0;
    a.nt = b->nt;
    a.cap = b->cap;
    a.x = a.y = a.z = a.q = nullptr;
    a.minv = b->d_minv;
    a.type = a.id = a.mol = nullptr;
    a.nl = nullptr;
    a.nn = b->nn;
    a.order = b->order;
    a.xq = b->xq;
    a.tid = b->tid;
    const int nt2 = b->nt * b->nt;
    a.c12 = b->d_lj;
    a.c6 = b->d_lj + nt2;
    a.cshift = b->d_lj + 2 * nt2;
    a.lj_rc2 = b->lj_rc * b->lj_rc;
    a.al = ewald_alpha(b->er_alpha);
    a.ke = b->er_ke;
    a.two_a_rpi = 2 * b->er_alpha * CAV_PIS_INV;
    a.lambda = nullptr;
    a.ax = b->ax;
    a.ay = b->ay;
    a.az = b->az;
    a.part = b->part;
    a.accumulate = 0;
    a.reps = batch_reps(b);
    a.nlb = b->nlb;
    a.xqs = b->xqs;
    a.litems = b->litems;
    a.qtype = b->d_charge;
    if (b->precision == CAV_FP64)
      batch_pairs_t<double>(b, a, g);
    else
      batch_pairs_t<float>(b, a, g);
  }
  BAT_HIP(hipGetLastError());
  return CAV_OK;
}

}  // namespace cav
