// Ghost images, cell binning, rebuild test and Verlet-list construction on
// gfx950.  Every kernel that depends on the per-step rebuild decision reads the
// device flag and returns early, so a step never waits for the host.
#include <algorithm>

#include "cav_internal.hpp"

namespace cav {

// ------------------------------------------------------------------ scans --

// Exclusive scan of one value per thread over a block of BS threads: wave64
// prefix sums with DPP-backed shuffles, then the wave totals through LDS.
template <int BS = kBlock>
__device__ __forceinline__ int block_exclusive_scan(int v, int *total)
{
  __shared__ int wsum[BS / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    int t = __shfl_up(inc, o, 64);
    if (lane >= o) inc += t;
  }
  if (lane == 63) wsum[wave] = inc;
  __syncthreads();
  int base = 0, tot = 0;
#pragma unroll
  for (int w = 0; w < BS / 64; ++w) {
    if (w < wave) base += wsum[w];
    tot += wsum[w];
  }
  __syncthreads();
  if (total) *total = tot;
  return base + inc - v;
}

// Per-block sums of `count(i)`; the functor recomputes the per-item count.
template <class F>
__global__ void k_block_sums(long nitems, F count, int *blk, const int *cond)
{
  if (cond && !*cond) return;
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  int v = i < nitems ? count(i) : 0;
  int tot;
  block_exclusive_scan(v, &tot);
  if (threadIdx.x == 0) blk[blockIdx.x] = tot;
}

// Exclusive scan of the block sums in one block; writes the grand total.  Each
// thread sums a contiguous run of ceil(nblk / 256) entries, one block scan
// combines the runs, and each thread then writes its run's prefixes: one
// pass with two barriers instead of one block scan per 256 entries.
// stop (or nullptr): nothing is scanned once it is set.  The sums are then
// those of an earlier launch, scanned already.
__global__ void k_scan_blocks(int nblk, int *blk, int *total, const int *cond, const int *stop)
{
  if (cond && !*cond) return;
  if (stop && *stop) return;
  const int per = (nblk + kBlock - 1) / kBlock;
  const int b0 = threadIdx.x * per, b1 = min(nblk, b0 + per);
  int s = 0;
  for (int i = b0; i < b1; ++i) s += blk[i];
  int tot;
  int ex = block_exclusive_scan(s, &tot);
  for (int i = b0; i < b1; ++i) {
    const int v = blk[i];
    blk[i] = ex;
    ex += v;
  }
  if (threadIdx.x == 0) *total = tot;
}

// ----------------------------------------------------------------- ghosts --

struct GhostRule {
  const double *x, *y, *z;
  double xl, xu, yl, yu, zl, zu;
  int bx, by, bz;
  __device__ __forceinline__ void sides(double px, double py, double pz, int &sx, int &sy,
                                        int &sz) const
  {
    // exchange_ghost_single_md_domain.cpp:70-101: strict tests, times the bc flag
    sx = (px < xl ? -1 : (px > xu ? 1 : 0)) * bx;
    sy = (py < yl ? -1 : (py > yu ? 1 : 0)) * by;
    sz = (pz < zl ? -1 : (pz > zu ? 1 : 0)) * bz;
  }
  __device__ __forceinline__ void sides(long i, int &sx, int &sy, int &sz) const
  {
    sides(x[i], y[i], z[i], sx, sy, sz);
  }
  static __device__ __forceinline__ int images(int sx, int sy, int sz)
  {
    const int a = sx != 0, b = sy != 0, c = sz != 0;
    return a + b + c + (a & b) + (a & c) + (b & c) + (a & b & c);
  }
  __device__ __forceinline__ int operator()(long i) const
  {
    int sx, sy, sz;
    sides(i, sx, sy, sz);
    return images(sx, sy, sz);
  }
};

static GhostRule ghost_rule(const cav_ctx *c)
{
  GhostRule r;
  r.x = c->x;
  r.y = c->y;
  r.z = c->z;
  r.xl = c->lo[0] + c->ghost_cutoff;
  r.xu = c->hi[0] - c->ghost_cutoff;
  r.yl = c->lo[1] + c->ghost_cutoff;
  r.yu = c->hi[1] - c->ghost_cutoff;
  r.zl = c->lo[2] + c->ghost_cutoff;
  r.zu = c->hi[2] - c->ghost_cutoff;
  r.bx = c->bc[0];
  r.by = c->bc[1];
  r.bz = c->bc[2];
  return r;
}

// ------------------------------------------------------------ rebuild test --

// Lane `src`'s double, as a scalar.
__device__ __forceinline__ double lane_d(double v, int src)
{
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), src);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), src);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// The w word of a bin-ordered candidate (cpos): the atom index in the low 32
// bits and its bin-order slot in the high 32 bits, so the list build can
// record either.
__device__ __forceinline__ double cpos_tag(int j, long t)
{
  return __longlong_as_double((long long)((unsigned long long)(unsigned)t << 32 | (unsigned)j));
}
__device__ __forceinline__ int cpos_index(double w) { return (int)(__double_as_longlong(w) & 0xffffffffll); }
__device__ __forceinline__ int cpos_slot(double w) { return (int)(__double_as_longlong(w) >> 32); }

// A double that is the same in every lane, moved to scalar registers.
__device__ __forceinline__ double uniform_d(double v)
{
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readfirstlane((int)(b & 0xffffffffll));
  const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

__device__ __forceinline__ double dot_rn(double a, double b, double c)
{
  // Vector::operator* as the reference evaluates it: (a*a + b*b) + c*c, every
  // product and sum rounded on its own (hipcc contracts to FMA by default).
#pragma clang fp contract(off)
  return (a * a + b * b) + c * c;
}

// Neighborlist::update_is_needed (neighborlist.cpp:91-139): size change, or any
// owned/ghost displacement^2 (ghosts compared by index) above the threshold.
__global__ void k_rebuild_check(int n, long cap_total, const double *x, const double *y,
                                const double *z, const double *xo, const double *yo,
                                const double *zo, double thr_sq, int rebuild_test, int *flags)
{
  if (flags[F_REBUILD]) return;
  const int G = flags[F_NGHOST], Gold = flags[F_NGHOST_OLD];
  if (rebuild_test || G != Gold) {
    if (blockIdx.x == 0 && threadIdx.x == 0) flags[F_REBUILD] = 1;
    return;
  }
  const long a = (long)blockIdx.x * kBlock + threadIdx.x;
  if (a >= (long)n + G || a >= cap_total) return;
  const double dx = xsub(x[a], xo[a]), dy = xsub(y[a], yo[a]), dz = xsub(z[a], zo[a]);
  if (dot_rn(dx, dy, dz) > thr_sq) flags[F_REBUILD] = 1;
}

int launch_rebuild_check(cav_ctx *c)
{
  const long tot = (long)c->n + c->gcap;
  k_rebuild_check<<<grid_for(tot), kBlock, 0, c->stream>>>(c->n, tot, c->x, c->y, c->z, c->xo,
                                                          c->yo, c->zo, c->thr_sq,
                                                          c->rebuild_test, c->flags);
  CAV_HIP(hipGetLastError());
  return CAV_OK;
}

// ------------------------------------------------------------------- cells --

struct BinRule {
  double lox, loy, loz, cinv;
  int nbx, nby, nbz;
  int shift;  // 0: the reference grid; 1: the grid with a ghost layer past every face
  // binlist_index + neigh_bin_index (neighborlist.cpp:408-436): floor, clamp,
  // x-fastest linear index.  With the ghost layer the index is the
  // reference's plus one and the grid has two more cells per axis: ghosts
  // then lie in their own cells instead of clamped into the edge cells, and
  // those farther than one cell from the box, which no owned atom reaches,
  // share the outermost layer.
  __device__ __forceinline__ int operator()(double px, double py, double pz) const
  {
    int ix = (int)floor(xmul(xsub(px, lox), cinv)) + shift;
    int iy = (int)floor(xmul(xsub(py, loy), cinv)) + shift;
    int iz = (int)floor(xmul(xsub(pz, loz), cinv)) + shift;
    ix = ix < 0 ? 0 : (ix >= nbx ? nbx - 1 : ix);
    iy = iy < 0 ? 0 : (iy >= nby ? nby - 1 : iy);
    iz = iz < 0 ? 0 : (iz >= nbz ? nbz - 1 : iz);
    return ix + nbx * iy + nbx * nby * iz;
  }
};

static BinRule bin_rule(const cav_ctx *c, bool ghost_layer)
{
  BinRule b;
  b.lox = c->lo[0];
  b.loy = c->lo[1];
  b.loz = c->lo[2];
  b.cinv = c->cinv;
  b.shift = ghost_layer ? 1 : 0;
  b.nbx = c->nb[0] + 2 * b.shift;
  b.nby = c->nb[1] + 2 * b.shift;
  b.nbz = c->nb[2] + 2 * b.shift;
  return b;
}

__global__ void k_zero_int(int *p, long n, const int *cond)
{
  if (cond && !*cond) return;
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) p[i] = 0;
}

// Atoms are binned in the bin order of the last list build (`border`, a
// permutation of its n + G_old slots; atoms past them in index order; entries
// of atoms that no longer exist skipped), so lanes next to each other mostly
// fall into one bin and a wave adds one count per run of equal bins instead
// of one per atom.  The bins' contents are the same in any order: the fill
// below uses the same order and every bin is sorted by index afterwards.
__device__ __forceinline__ long bin_order_atom(long t, long tot, long told, const int *border)
{
  const long a = t < told ? (long)border[t] : t;
  return a >= 0 && a < tot ? a : -1;
}

// Runs of equal bins (b >= 0) among consecutive lanes: the length of the run
// this lane heads (0 if it heads none); `hm` returns the wave's run heads.
__device__ __forceinline__ int bin_run(int b, unsigned long long &hm)
{
  const int lane = threadIdx.x & 63;
  const int pb = __shfl_up(b, 1, 64);
  const bool brk = lane == 0 || b != pb;
  const unsigned long long bm = __ballot(brk);
  hm = __ballot(brk && b >= 0);
  if (!(brk && b >= 0)) return 0;
  const unsigned long long above = bm & ~((2ull << lane) - 1ull);
  return (above ? __ffsll((long long)above) - 1 : 64) - lane;
}

__global__ void k_bin_count(int n, long cap_total, BinRule rule, const double *x, const double *y,
                            const double *z, int *bin_of, int *bin_cnt, const int *flags,
                            const int *cond, const int *border)
{
  if (cond && !*cond) return;
  const long t = (long)blockIdx.x * kBlock + threadIdx.x;
  const long tot = (long)n + flags[F_NGHOST];
  const long told = flags[F_NGHOST_OLD] < 0 ? 0 : (long)n + flags[F_NGHOST_OLD];
  const long a = t < cap_total && t < (tot > told ? tot : told) ? bin_order_atom(t, tot, told, border) : -1;
  const int b = a >= 0 ? rule(x[a], y[a], z[a]) : -1;
  if (a >= 0) bin_of[a] = b;
  unsigned long long hm;
  const int len = bin_run(b, hm);
  if (len) atomicAdd(bin_cnt + b, len);
}

struct CountOf {
  const int *cnt;
  __device__ __forceinline__ int operator()(long i) const { return cnt[i]; }
};

__global__ void k_bin_start(int nbins, const int *cnt, const int *blk, int *start, const int *cond)
{
  if (cond && !*cond) return;
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  const int v = i < nbins ? cnt[i] : 0;
  const int off = block_exclusive_scan(v, nullptr) + blk[blockIdx.x];
  if (i < nbins) start[i] = off;
  if (i == nbins - 1) start[nbins] = off + v;
}

__global__ void k_bin_fill(int n, long cap_total, const int *bin_of, const int *start, int *cur,
                           int *items, const int *flags, const int *cond, const int *border)
{
  if (cond && !*cond) return;
  const long t = (long)blockIdx.x * kBlock + threadIdx.x;
  const long tot = (long)n + flags[F_NGHOST];
  const long told = flags[F_NGHOST_OLD] < 0 ? 0 : (long)n + flags[F_NGHOST_OLD];
  const long a = t < cap_total && t < (tot > told ? tot : told) ? bin_order_atom(t, tot, told, border) : -1;
  const int b = a >= 0 ? bin_of[a] : -1;
  unsigned long long hm;
  const int len = bin_run(b, hm);
  int base = 0;
  if (len) base = atomicAdd(cur + b, len);
  // every lane of a run takes the next slot after its head's
  const int lane = threadIdx.x & 63;
  const unsigned long long mine = hm & ((2ull << lane) - 1ull);
  const int head = mine ? 63 - __clzll((long long)mine) : lane;
  base = __shfl(base, head, 64);
  if (b >= 0) items[start[b] + base + (lane - head)] = (int)a;
}

// Insertion order of update_cell_list (owned ascending, then ghosts n+g
// ascending, neighborlist.cpp:457-471) is ascending index order: every bin is
// sorted after the (atomic, unordered) fill.
// One bin per wave (kSortWaves bins per workgroup, no block barrier): a bin of
// at most 64 atoms is sorted by rank (each lane counts the smaller indices of
// the others through shuffles; indices are distinct), a larger one with a
// bitonic network in the wave's LDS, and beyond kSortWaveMax atoms by lane 0.
constexpr int kSortWaves = 4, kSortWaveMax = 2048;

__device__ void sort_bin_wave(int s, int e, int *items, int *v)
{
  const int lane = threadIdx.x & 63;
  const int m = e - s;
  if (m <= 1) return;
  if (m <= 64) {
    const int x = lane < m ? items[s + lane] : 0x7fffffff;
    int rank = 0;
    for (int k = 0; k < m; ++k) rank += __shfl(x, k, 64) < x ? 1 : 0;
    if (lane < m) items[s + rank] = x;
    return;
  }
  if (m <= kSortWaveMax) {
    int p2 = 128;
    while (p2 < m) p2 <<= 1;
    for (int t = lane; t < p2; t += 64) v[t] = t < m ? items[s + t] : 0x7fffffff;
    __syncwarp();
    const int half = p2 >> 1;
    for (int k = 2; k <= p2; k <<= 1) {
      for (int j = k >> 1; j > 0; j >>= 1) {
        for (int t = lane; t < half; t += 64) {
          const int lo = ((t & ~(j - 1)) << 1) | (t & (j - 1));
          const int hi = lo | j;
          const int a = v[lo], c = v[hi];
          if ((a > c) == ((lo & k) == 0)) {
            v[lo] = c;
            v[hi] = a;
          }
        }
        __syncwarp();
      }
    }
    for (int t = lane; t < m; t += 64) items[s + t] = v[t];
    return;
  }
  if (lane != 0) return;
  for (int i = s + 1; i < e; ++i) {
    const int val = items[i];
    int j = i - 1;
    while (j >= s && items[j] > val) {
      items[j + 1] = items[j];
      --j;
    }
    items[j + 1] = val;
  }
}

__global__ __launch_bounds__(64 * kSortWaves) void k_bin_sort(int nbins, const int *start, int *items,
                                                              const int *cond)
{
  __shared__ int v_[kSortWaves][kSortWaveMax];
  if (cond && !*cond) return;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = blockIdx.x * kSortWaves + wv;
  if (b >= nbins) return;
  sort_bin_wave(start[b], start[b + 1], items, v_[wv]);
}

// (x, y, z, index and slot) in bin order, for contiguous candidate staging in
// the list build; on the list build's own binning (list_cond set) also the
// bin order the list keeps: slot -> atom (litems) and atom -> slot (binpos)
__global__ void k_cell_pack(long cap_total, int n, const int *items, const double *x, const double *y,
                            const double *z, double4 *cpos, const int *flags, const int *cond,
                            int *litems, int *binpos, const int *list_cond)
{
  if (cond && !*cond) return;
  const long t = (long)blockIdx.x * kBlock + threadIdx.x;
  if (t >= (long)n + flags[F_NGHOST] || t >= cap_total) return;
  const int j = items[t];
  cpos[t] = make_double4(x[j], y[j], z[j], cpos_tag(j, t));
  if (litems && *list_cond) {
    litems[t] = j;
    binpos[j] = (int)t;
  }
}

// Owned atoms in cell order: stable compaction of bin_items (ghost entries
// dropped).  Consecutive lanes then walk overlapping stencils.
__global__ void k_order_scatter(long cap_total, int n, const int *items, const int *blk, int *order,
                                const int *flags, const int *cond)
{
  if (cond && !*cond) return;
  const long t = (long)blockIdx.x * kBlock + threadIdx.x;
  const long tot = (long)n + flags[F_NGHOST];
  const int a = (t < tot && t < cap_total) ? items[t] : n;
  const int f = a < n ? 1 : 0;
  const int off = block_exclusive_scan(f, nullptr) + blk[blockIdx.x];
  if (f) order[off] = a;
}

struct OwnedFlagBounded {
  const int *items;
  const int *flags;
  int n;
  __device__ __forceinline__ int operator()(long t) const
  {
    return (t < (long)n + flags[F_NGHOST] && items[t] < n) ? 1 : 0;
  }
};

int launch_bins(cav_ctx *c, bool conditional, bool for_list)
{
  const int *cond = conditional ? c->flags + F_REBUILD : nullptr;
  // every list build keeps its bin order (the bin-order pair gathers and the
  // cell-staged kernel read it, and the next binning visits atoms in it)
  const bool keep = for_list;
  const long tot = (long)c->n + c->gcap;
  const bool xg = for_list && list_on_ghost_grid(c);
  const BinRule rule = bin_rule(c, xg);
  const int nbins = xg ? c->xnbins : c->nbins;
  k_zero_int<<<grid_for(nbins), kBlock, 0, c->stream>>>(c->bin_cnt, nbins, cond);
  k_bin_count<<<grid_for(tot), kBlock, 0, c->stream>>>(c->n, tot, rule, c->x, c->y, c->z,
                                                      c->bin_of, c->bin_cnt, c->flags, cond,
                                                      c->litems);
  const int nb = grid_for(nbins);
  CountOf cnt{c->bin_cnt};
  k_block_sums<<<nb, kBlock, 0, c->stream>>>(nbins, cnt, c->scan_tmp, cond);
  k_scan_blocks<<<1, kBlock, 0, c->stream>>>(nb, c->scan_tmp, c->flags + F_COUNT - 1, cond, nullptr);
  k_bin_start<<<nb, kBlock, 0, c->stream>>>(nbins, c->bin_cnt, c->scan_tmp, c->bin_start, cond);
  k_zero_int<<<grid_for(nbins), kBlock, 0, c->stream>>>(c->bin_cnt, nbins, cond);
  k_bin_fill<<<grid_for(tot), kBlock, 0, c->stream>>>(c->n, tot, c->bin_of, c->bin_start,
                                                     c->bin_cnt, c->bin_items, c->flags, cond,
                                                     c->litems);
  k_bin_sort<<<(nbins + kSortWaves - 1) / kSortWaves, 64 * kSortWaves, 0, c->stream>>>(
      nbins, c->bin_start, c->bin_items, cond);
  k_cell_pack<<<grid_for(tot), kBlock, 0, c->stream>>>(tot, c->n, c->bin_items, c->x, c->y, c->z,
                                                      c->cpos, c->flags, cond,
                                                      keep ? c->litems : nullptr,
                                                      keep ? c->binpos : nullptr,
                                                      c->flags + F_REBUILD);
  const int nbo = grid_for(tot);
  OwnedFlagBounded of{c->bin_items, c->flags, c->n};
  k_block_sums<<<nbo, kBlock, 0, c->stream>>>(tot, of, c->ord_blk, cond);
  k_scan_blocks<<<1, kBlock, 0, c->stream>>>(nbo, c->ord_blk, c->flags + F_COUNT - 2, cond, nullptr);
  k_order_scatter<<<nbo, kBlock, 0, c->stream>>>(tot, c->n, c->bin_items, c->ord_blk, c->order,
                                                 c->flags, cond);
  CAV_HIP(hipGetLastError());
  return CAV_OK;
}

// ------------------------------------------------------ a step's exchange --
//
// A step's short-range part up to the Verlet rows is four launches, whatever
// the size: k_move (drift or wrap, per-block ghost counts, displacement test of
// the owned atoms), k_ghosts (images, rebuild decision, cell counts and
// buckets), k_cells (cell starts, sorted cells and everything in bin order) and
// the list build.  As one kernel per scan, fill, sort and copy it was eighteen,
// of 2-4 us each plus the gap before it: this alone took a step of 256 LJ atoms
// from 141 to 72 us (now 39), of 8000 ions (FP64, kmax 8) from 209 to 119 (now
// 90); at N = 262144, where the gaps hide beside Ewald_k, it changed nothing.

typedef unsigned long long u64t;

// Sums of two values over the BS threads of a block, in every thread.
template <int BS>
__device__ __forceinline__ void block_sum2(int &a, int &b)
{
  __shared__ int s[2][BS / 64];
  for (int o = 32; o > 0; o >>= 1) {
    a += __shfl_xor(a, o, 64);
    b += __shfl_xor(b, o, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    s[0][threadIdx.x >> 6] = a;
    s[1][threadIdx.x >> 6] = b;
  }
  __syncthreads();
  a = b = 0;
#pragma unroll
  for (int w = 0; w < BS / 64; ++w) {
    a += s[0][w];
    b += s[1][w];
  }
}

// Batched replicas run the kernels of the exchange with each workgroup on one
// replica (rep_block): it shifts its arrays to the replica's slots (base), owned atoms
// (obase) and cells (cbase) and takes the box, ghost and cell rules from it.
__device__ __forceinline__ GhostRule ghost_rule_of(const RepDev &r, double gc)
{
  GhostRule g;
  g.x = g.y = g.z = nullptr;
  g.xl = r.lo[0] + gc;
  g.xu = r.hi[0] - gc;
  g.yl = r.lo[1] + gc;
  g.yu = r.hi[1] - gc;
  g.zl = r.lo[2] + gc;
  g.zu = r.hi[2] - gc;
  g.bx = g.by = g.bz = 1;
  return g;
}

// A replica's cells: the grid with the ghost layer (r.nb counts it).
__device__ __forceinline__ BinRule bin_rule_of(const RepDev &r, double cinv)
{
  BinRule b;
  b.lox = r.lo[0];
  b.loy = r.lo[1];
  b.loz = r.lo[2];
  b.cinv = cinv;
  b.shift = 1;
  b.nbx = r.nb[0];
  b.nby = r.nb[1];
  b.nbz = r.nb[2];
  return b;
}

struct MoveArgs {
  int n;
  double dt;
  double lo[3], hi[3], L[3];
  int bc[3];
  double *x, *y, *z;
  const double *vx, *vy, *vz, *ax, *ay, *az;
  double *aox, *aoy, *aoz, *snap;
  const double *xo, *yo, *zo;  // positions at the last list build, or nullptr
  double thr_sq;
  int *flags, *blk;
  u64t *cnt;  // cell counters to clear, or nullptr
  int nbins;
  long stride;  // of the snapshot's planes
  RepGrid reps;  // REP: the replicas, and their ghost cutoff
  double gc;
};

// DRIFT: integrate_velocity_verlet's drift (md_simulator.cpp:584-594), every
// operation rounded as the reference's expression is: r += (v*dt +
// ((0.5*a)*dt)*dt); the step snapshot of positions, velocities and
// accelerations ([x | y | z | vx | vy | vz | ax | ay | az], n each) is written
// from the values it reads.  Then, for setup and recalculate too, the wrap of
// exchange_owned (domain.cpp:418-468) and the number of the block's images.
// Once F_STOP is set (a step before this one failed) nothing moves and the
// snapshot stays.  HBM bound: 216 B an atom.
template <bool DRIFT, int BS, bool REP>
__global__ __launch_bounds__(BS) void k_move(MoveArgs a, GhostRule rule)
{
  int blk = blockIdx.x, blocks = gridDim.x;
  if constexpr (REP) {
    const int rr = rep_block(a.reps, blk, blocks);
    if (rr < 0) return;
    const RepDev &r = a.reps.rep[rr];
    a.blk += (long)rr * blocks;
    blocks = (r.n + BS - 1) / BS;
    if (blk >= blocks) return;
    a.n = r.n;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      a.lo[d] = r.lo[d];
      a.hi[d] = r.hi[d];
      a.L[d] = r.L[d];
      a.bc[d] = 1;
    }
    a.x += r.base, a.y += r.base, a.z += r.base;
    if (a.xo) a.xo += r.base, a.yo += r.base, a.zo += r.base;
    if constexpr (DRIFT) {
      a.vx += r.obase, a.vy += r.obase, a.vz += r.obase;
      a.ax += r.obase, a.ay += r.obase, a.az += r.obase;
      a.snap += r.obase;
    }
    a.flags += 16 * rr;
    a.cnt += r.cbase;
    a.nbins = r.nbins;
    rule = ghost_rule_of(r, a.gc);
  }
  const int i = blk * BS + threadIdx.x;
  const int at = i < a.n ? i : 0;
  const int stop = a.flags[F_STOP];
  const double old[3] = {a.x[at], a.y[at], a.z[at]};
  double acc[3], v[3], last[3];
  if constexpr (DRIFT) {
    acc[0] = a.ax[at], acc[1] = a.ay[at], acc[2] = a.az[at];
    v[0] = a.vx[at], v[1] = a.vy[at], v[2] = a.vz[at];
  }
  if (a.xo) last[0] = a.xo[at], last[1] = a.yo[at], last[2] = a.zo[at];
  if (DRIFT && stop) return;
  if (a.cnt)
    for (int k = i; k < a.nbins; k += blocks * BS) a.cnt[k] = 0;
  int cnt = 0, moved = 0;
  if (i < a.n) {
    double *p[3] = {a.x + i, a.y + i, a.z + i};
    double r[3] = {old[0], old[1], old[2]};
    if constexpr (DRIFT) {
      if (isnan(acc[0]) || isnan(acc[1]) || isnan(acc[2])) a.flags[F_NAN] = 1;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        a.snap[d * a.stride + i] = r[d];
        a.snap[(3 + d) * a.stride + i] = v[d];
        a.snap[(6 + d) * a.stride + i] = acc[d];
        const double h = xmul(xmul(xmul(0.5, acc[d]), a.dt), a.dt);
        r[d] = xadd(r[d], xadd(xmul(v[d], a.dt), h));
      }
      if constexpr (!REP) {  // a batch reads the snapshot's planes
        a.aox[i] = acc[0];
        a.aoy[i] = acc[1];
        a.aoz[i] = acc[2];
      }
    }
    bool wrapped = false;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      if (a.bc[d] == 1) {
        if (r[d] < a.lo[d]) {
          r[d] = xadd(r[d], a.L[d]);
          wrapped = true;
        } else if (r[d] > a.hi[d]) {
          r[d] = xsub(r[d], a.L[d]);
          wrapped = true;
        }
      }
      *p[d] = r[d];
    }
    if (wrapped) {
      a.flags[F_WRAPPED] = 1;
      a.flags[F_REBUILD] = 1;
    }
    int sx, sy, sz;
    rule.sides(r[0], r[1], r[2], sx, sy, sz);
    cnt = GhostRule::images(sx, sy, sz);
    if (a.xo) {
      const double dx = xsub(r[0], last[0]), dy = xsub(r[1], last[1]), dz = xsub(r[2], last[2]);
      moved = dot_rn(dx, dy, dz) > a.thr_sq;
    }
  }
  if (moved) a.flags[F_REBUILD] = 1;
  int none = 0;
  block_sum2<BS>(cnt, none);
  if (threadIdx.x == 0) a.blk[blk] = cnt;
}

struct GhostArgs {
  int n, nblk, scanned;  // scanned: blk already holds exclusive sums, F_NGHOST the total
  double L[3];
  const int *blk;
  double *x, *y, *z;
  int *type, *id, *mol, *gsrc;
  double *q;
  const double *xo, *yo, *zo;  // or nullptr: no rebuild decision
  double thr_sq;
  int rebuild_test;
  int *flags;
  double4 *xq;  // packed copies, or nullptr
  int2 *tid;
  u64t *cnt;    // cells (owned count in the high word), or nullptr
  int *bucket;
  int cap;
  RepGrid reps;  // REP: the replicas, their ghost cutoff and cell width
  double gc, cinv;
};

// The images of owned atom i at ghost slots n + g, g ascending with i, in the
// order x, y, z, xy, xz, yz, xyz (exchange_ghost_single_md_domain.cpp:167-215).
// Each block adds up the counts of the blocks before it itself (no scan
// launch).  With the total known, the rest of Neighborlist::update_is_needed
// (neighborlist.cpp:91-139; the owned displacements were tested by the move):
// the number of ghosts, and each ghost's displacement.  Every slot is also
// packed for the gathers and put into its cell's bucket, whether the list is
// rebuilt or not: the decision is not known yet, and the counting is cheaper
// than a launch of its own.
template <int BS, bool REP>
__global__ __launch_bounds__(BS) void k_ghosts(GhostArgs a, GhostRule rule, BinRule bins)
{
  int gcap = 0, blk = blockIdx.x;
  if constexpr (REP) {
    int blocks;
    const int rr = rep_block(a.reps, blk, blocks);
    if (rr < 0) return;
    const RepDev &r = a.reps.rep[rr];
    a.n = r.n;
    a.nblk = (r.n + BS - 1) / BS;
    if (blk >= a.nblk) return;
    a.blk += (long)rr * blocks;
    a.flags += 16 * rr;
    gcap = r.gcap;
    a.L[0] = r.L[0], a.L[1] = r.L[1], a.L[2] = r.L[2];
    a.x += r.base, a.y += r.base, a.z += r.base;
    a.type += r.base;
    a.id += r.base;
    a.q += r.base;
    if (a.xo) a.xo += r.base, a.yo += r.base, a.zo += r.base;
    a.xq += r.base;
    a.tid += r.base;
    a.cnt += r.cbase;
    a.bucket += r.bbase;
    a.cap = r.bcap;
    rule = ghost_rule_of(r, a.gc);
    bins = bin_rule_of(r, a.cinv);
  }
  // every load that depends on nothing first: at small sizes the kernel is a
  // chain of such latencies
  const int i = blk * BS + threadIdx.x;
  const bool live = i < a.n;
  const int at = live ? i : 0;
  const double px = a.x[at], py = a.y[at], pz = a.z[at], qq = a.q[at];
  const int t = a.type[at], d = a.id[at], m = REP ? 0 : a.mol[at];
  const int stop = a.flags[F_STOP], old = a.flags[F_NGHOST_OLD];
  int before, total;
  if (a.scanned) {
    before = a.blk[blk];
    total = a.flags[F_NGHOST];
  } else {
    before = total = 0;
    for (int k = threadIdx.x; k < a.nblk; k += BS) {
      const int v = a.blk[k];
      total += v;
      if (k < blk) before += v;
    }
    block_sum2<BS>(before, total);
  }
  if (stop) return;
  int sx = 0, sy = 0, sz = 0, cnt = 0;
  if (live) {
    rule.sides(px, py, pz, sx, sy, sz);
    cnt = GhostRule::images(sx, sy, sz);
  }
  const int off = before + block_exclusive_scan<BS>(cnt, nullptr);
  // a batch gives each replica the ghost slots it expects: images past them
  // are left out and the step is taken again with more
  const bool over = REP && total > gcap;
  if (over) {
    total = gcap;
    if (i == 0) a.flags[F_GOVER] = 1;
  }
  bool test = false;
  if (a.xo) {
    const bool differs = a.rebuild_test || total != old;
    test = !differs;
    if (differs && i == 0) a.flags[F_REBUILD] = 1;
  }
  if (i == 0 && !a.scanned) a.flags[F_NGHOST] = total;
  if (!live) return;
  const double gx = px - sx * a.L[0], gy = py - sy * a.L[1], gz = pz - sz * a.L[2];
  // slot 0 is the atom itself, 1..7 its images in order (the axes they shift as
  // bits: x, y, z, xy, xz, yz, xyz).  The counters' answers are asked for
  // first, in variables of their own (an array's elements are copied together,
  // which waits for each), so that up to eight atomics are in flight at once:
  // one after the other they were most of this kernel's time at small sizes.
  const bool mx = sx != 0, my = sy != 0, mz = sz != 0;
  int img = (mx ? 1 : 0) | (my ? 2 : 0) | (mz ? 4 : 0) | (mx && my ? 8 : 0) | (mx && mz ? 16 : 0) |
            (my && mz ? 32 : 0) | (mx && my && mz ? 64 : 0);
  if (over)
    while (img && off + __popc(img) > gcap) img &= ~(1 << (31 - __clz(img)));
  auto cell_of = [&](int ax) { return bins(ax & 1 ? gx : px, ax & 2 ? gy : py, ax & 4 ? gz : pz); };
  u64t r0, r1, r2, r3, r4, r5, r6, r7;
  if (a.cnt) {
    r0 = atomicAdd(a.cnt + cell_of(0), 1ull << 32 | 1ull);
    if (img & 1) r1 = atomicAdd(a.cnt + cell_of(1), 1ull);
    if (img & 2) r2 = atomicAdd(a.cnt + cell_of(2), 1ull);
    if (img & 4) r3 = atomicAdd(a.cnt + cell_of(4), 1ull);
    if (img & 8) r4 = atomicAdd(a.cnt + cell_of(3), 1ull);
    if (img & 16) r5 = atomicAdd(a.cnt + cell_of(5), 1ull);
    if (img & 32) r6 = atomicAdd(a.cnt + cell_of(6), 1ull);
    if (img & 64) r7 = atomicAdd(a.cnt + cell_of(7), 1ull);
  }
  int g = off;
  auto put = [&](int ax) {
    const double u = ax & 1 ? gx : px, v = ax & 2 ? gy : py, w = ax & 4 ? gz : pz;
    long s = i;
    if (ax > 0) {
      s = (long)a.n + g;
      if (test) {
        const double dx = xsub(u, a.xo[s]), dy = xsub(v, a.yo[s]), dz = xsub(w, a.zo[s]);
        if (dot_rn(dx, dy, dz) > a.thr_sq) a.flags[F_REBUILD] = 1;
      }
      if constexpr (!REP) {  // (of a batch's images only the packed copies are read)
        a.x[s] = u;
        a.y[s] = v;
        a.z[s] = w;
        a.type[s] = t;
        a.id[s] = d;
        a.mol[s] = m;
        a.q[s] = qq;
        a.gsrc[g] = i;
      }
      ++g;
    }
    if (a.xq) {
      a.xq[s] = make_double4(u, v, w, qq);
      a.tid[s] = make_int2(t, d);
    }
  };
  put(0);
  if (img & 1) put(1);
  if (img & 2) put(2);
  if (img & 4) put(4);
  if (img & 8) put(3);
  if (img & 16) put(5);
  if (img & 32) put(6);
  if (img & 64) put(7);
  if (!a.cnt) return;
  auto keep = [&](long s, int ax, u64t r) {
    const int b = cell_of(ax), rank = (int)(unsigned)r;
    if (rank < a.cap) a.bucket[(long)b * a.cap + rank] = (int)s;
  };
  long s = (long)a.n + off;
  keep(i, 0, r0);
  if (img & 1) keep(s++, 1, r1);
  if (img & 2) keep(s++, 2, r2);
  if (img & 4) keep(s++, 4, r3);
  if (img & 8) keep(s++, 3, r4);
  if (img & 16) keep(s++, 5, r5);
  if (img & 32) keep(s++, 6, r6);
  if (img & 64) keep(s++, 7, r7);
}

struct CellBuild {
  int n, nbins, bpb, cap;
  const u64t *cnt;
  const int *bucket;
  const double4 *xq;
  const int2 *tid;
  int *start, *items, *order, *binpos, *litems;
  double4 *xqs;  // slot_record
  double *xo, *yo, *zo;
  int *flags;
  RepGrid reps;  // REP: the replicas, their cell width
  double cinv;
  const u64t *first;  // counters before each workgroup's cells, or nullptr: added up here
};

// Threads of a cell workgroup.  A batch, whose replicas have few cells each, takes
// four waves: sixteen wait for a whole compute unit beside Ewald_k's passes (256
// replicas: 208 us, four waves of two cells 116; alone 97 and 79).
constexpr int kCellBlock = 1024, kBatchCellBlock = 256;

// Cells of a list build, one wave per cell, bpb cells per workgroup: cell
// starts (a workgroup adds up the counters of the cells before its own),
// the cell's slots sorted by index (update_cell_list's insertion order is
// owned ascending, then ghosts ascending, neighborlist.cpp:457-471), and in
// that order the slot -> atom and atom -> slot maps, the owned atoms, the list
// build's candidates and the packed copies; pos_old as well
// (neighborlist.cpp:302-303).  Without a rebuild only the packed copies are
// refreshed, in the order of the last one.
template <bool REP, int CB>
__global__ __launch_bounds__(CB) void k_cells(CellBuild a, BinRule bins)
{
  int blk = blockIdx.x, blocks = gridDim.x;
  if constexpr (REP) {
    const int rr = rep_block(a.reps, blk, blocks);
    if (rr < 0) return;
    const RepDev &r = a.reps.rep[rr];
    a.n = r.n;
    a.nbins = r.nbins;
    if (a.first) a.first += (long)rr * blocks;
    blocks = (r.nbins + a.bpb - 1) / a.bpb;
    if (blk >= blocks) return;
    a.cnt += r.cbase;
    a.bucket += r.bbase;
    a.cap = r.bcap;
    a.xq += r.base, a.tid += r.base;
    a.start += r.cbase + rr;  // one closing entry a replica
    a.items += r.base, a.litems += r.base;
    a.order += r.obase;
    a.xqs += r.base;
    a.xo += r.base, a.yo += r.base, a.zo += r.base;
    a.flags += 16 * rr;
    bins = bin_rule_of(r, a.cinv);
  }
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = a.flags[F_NGHOST], stop = a.flags[F_STOP], rebuild = a.flags[F_REBUILD];
  const int b0 = blk * a.bpb;
  // counters before the workgroup's cells, its own, and the slots of each
  // wave's first cell (whatever the bucket holds past its count): asked for
  // together, before the flags are known
  u64t s = 0;
  if (REP && a.first) {
    if (threadIdx.x == 0) s = a.first[blk];
  } else {
#pragma unroll 4
    for (int k = threadIdx.x; k < b0; k += CB) s += a.cnt[k];
  }
  const u64t own = lane < a.bpb && b0 + lane < a.nbins ? a.cnt[b0 + lane] : 0;
  const int early = lane < a.cap && wv < a.bpb && b0 + wv < a.nbins
                        ? a.bucket[(long)(b0 + wv) * a.cap + lane] : 0;
  const long tot = (long)a.n + G;
  if (stop) return;
  if (!rebuild) {
    for (long t = (long)blk * CB + threadIdx.x; t < tot;
         t += (long)blocks * CB) {
      const int j = a.litems[t];
      a.xqs[t] = slot_record(a.xq[j], a.tid[j], j >= a.n);
    }
    return;
  }
  if (blk == 0 && threadIdx.x == 0) a.flags[F_NGHOST_OLD] = G;
  __shared__ u64t part[CB / 64];
  __shared__ u64t first[65];  // per cell: slots before it, owned atoms before it
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if (lane == 0) part[wv] = s;
  __syncthreads();
  if (wv == 0) {
    u64t base = lane < CB / 64 ? part[lane] : 0;
    for (int o = 8; o > 0; o >>= 1) base += __shfl_xor(base, o, 16);
    base = __shfl(base, 0, 64);
    const u64t v = own;
    u64t inc = v;
    for (int o = 1; o < 64; o <<= 1) {
      const u64t u = __shfl_up(inc, o, 64);
      if (lane >= o) inc += u;
    }
    first[lane] = base + inc - v;
    if (lane == 63) first[64] = base + inc;
    if (lane < a.bpb && b0 + lane < a.nbins) a.start[b0 + lane] = (int)(base + inc - v);
    if (lane < a.bpb && b0 + lane == a.nbins - 1) a.start[a.nbins] = (int)(base + inc);
  }
  __syncthreads();
  for (int w = wv; w < a.bpb && b0 + w < a.nbins; w += CB / 64) {
    const int b = b0 + w;
    const long s0 = (long)(unsigned)first[w];
    const int o0 = (int)(first[w] >> 32);
    const int m = (int)((unsigned)first[w + 1] - (unsigned)first[w]);
    if (m == 0) continue;
    const int *mine = a.bucket + (long)b * a.cap;
    int j0 = 0x7fffffff, rank = 0;
    if (m <= 64 && m <= a.cap) {
      // one slot per lane, ranked by the smaller indices of the others
      if (lane < m) j0 = w == wv ? early : mine[lane];
      for (int k = 0; k < m; ++k) rank += __builtin_amdgcn_readlane(j0, k) < j0 ? 1 : 0;
    } else {
      // large cells through memory: the unsorted slots (those past the bucket's
      // capacity are found again by their cell), then each one's rank
      if (m > a.cap) {
        if (lane == 0) atomicMax(a.flags + F_MAXCELL, m);  // the host makes the buckets larger
        int at = 0;
        for (long t0 = 0; t0 < tot; t0 += 64) {
          bool in = false;
          if (t0 + lane < tot) {
            const double4 v = a.xq[t0 + lane];
            in = bins(v.x, v.y, v.z) == b;
          }
          const u64t mask = __ballot(in);
          if (in) a.items[s0 + at + __popcll(mask & ((1ull << lane) - 1ull))] = (int)(t0 + lane);
          at += __popcll(mask);
        }
      } else {
        for (int k = lane; k < m; k += 64) a.items[s0 + k] = mine[k];
      }
      __threadfence_block();
      for (int k = lane; k < m; k += 64) {
        const int j = a.items[s0 + k];
        int r = 0;
        for (int u = 0; u < m; ++u) r += a.items[s0 + u] < j ? 1 : 0;
        a.litems[s0 + r] = j;
      }
      __threadfence_block();
    }
    for (int k = lane; k < m; k += 64) {
      int j = j0, r = rank;
      if (m > 64 || m > a.cap) {
        r = k;
        j = a.litems[s0 + k];
      }
      const long t = s0 + r;
      const double4 v = a.xq[j];
      const int2 u = a.tid[j];
      a.litems[t] = j;
      if constexpr (!REP) a.binpos[j] = (int)t;
      if (j < a.n) a.order[o0 + r] = j;  // owned atoms come first in a cell
      a.xqs[t] = slot_record(v, u, j >= a.n);
      a.xo[j] = v.x;
      a.yo[j] = v.y;
      a.zo[j] = v.z;
    }
  }
}

// The four-launch exchange covers lists built on the ghost-layer grid for the
// bin-order pair kernel (the default).  A workgroup of k_cells reads the
// counters of all cells before its own, so grids past 65536 cells (about a
// million atoms at rho = 0.3) keep the scans; so do grids so empty that the
// buckets would take more room than the atoms' slots.
bool fused_cells(const cav_ctx *c)
{
  return c->nl_on && c->bucket && c->pair_kind == CAV_PAIRS_AUTO && list_on_ghost_grid(c) && c->nlb;
}

int cells_alloc(cav_ctx *c)
{
  if (c->bucket) (void)hipFree(c->bucket);
  if (c->cell_cnt) (void)hipFree(c->cell_cnt);
  c->bucket = nullptr;
  c->cell_cnt = nullptr;
  k_zero_int<<<1, kBlock, 0, c->stream>>>(c->flags + F_MAXCELL, 1, nullptr);
  if (!c->nl_on || c->n == 0 || c->xnbins > 65536) return CAV_OK;
  // twice the mean cell and some, in whole half waves
  const double cell = c->rce * c->rce * c->rce, vol = c->L[0] * c->L[1] * c->L[2];
  const long want = (long)(2.0 * cell * (c->n / vol)) + 32;
  const long cap = std::min(1024L, (want + 31) / 32 * 32);
  if (cap * c->xnbins > 32L * ((long)c->n + c->gcap) + 65536) return CAV_OK;
  CAV_HIP(hipMalloc(&c->bucket, sizeof(int) * cap * c->xnbins));
  CAV_HIP(hipMalloc(&c->cell_cnt, sizeof(u64t) * c->xnbins));
  c->bucket_cap = (int)cap;
  return CAV_OK;
}

// A quarter more than the fullest cell, in whole half waves.
static long crowd_cap(int most) { return ((long)most + most / 4 + 31) / 32 * 32; }

// Buckets are sized for the mean cell.  A wave of k_cells whose cell has more
// slots looks through all atoms for them: in a droplet of 30000 atoms (cutoff
// 5, 150 a cell, the mean 9) 717 us a build, from larger buckets 180.  So once
// cells were met past their room, with the flags read back and the stream
// idle, the buckets grow to the fullest, as long as they stay within 64 MB or
// what the slots themselves take.
int cells_fit(cav_ctx *c)
{
  const int most = c->h_flags[F_MAXCELL];
  if (!c->bucket || most <= c->bucket_cap) return CAV_OK;
  const long cap = crowd_cap(most);
  if (cap * c->xnbins > std::max(16L << 20, 32L * ((long)c->n + c->gcap))) return CAV_OK;
  (void)hipSetDevice(c->device);
  int *larger = nullptr;
  if (hipMalloc(&larger, sizeof(int) * cap * c->xnbins) != hipSuccess) {
    (void)hipGetLastError();  // the present ones do
    return CAV_OK;
  }
  (void)hipFree(c->bucket);
  c->bucket = larger;
  c->bucket_cap = (int)cap;
  return CAV_OK;
}

// Threads per workgroup of the move and the ghosts (the image counts are per
// workgroup of both): one wave for few atoms, so that the images' scattered
// stores (up to eighty an atom) spread over more CUs.  The ghosts
// of 256 atoms 14.2 -> 8.5 us, of 4000 11.5 -> 9.3, of 8000 12.2 -> 10.2; 30011
// 12.3 -> 13.3, which keeps 256.
static int move_block(const cav_ctx *c) { return c->n <= 16384 ? 64 : kBlock; }

// Owned atoms moved (drift of dt, or only wrapped) and the images counted;
// `decide`: with the rebuild test.
int launch_move(cav_ctx *c, bool drift, double dt, bool decide)
{
  MoveArgs a;
  a.n = c->n;
  a.dt = dt;
  for (int d = 0; d < 3; ++d) {
    a.lo[d] = c->lo[d];
    a.hi[d] = c->hi[d];
    a.L[d] = c->L[d];
    a.bc[d] = c->bc[d];
  }
  a.x = c->x;
  a.y = c->y;
  a.z = c->z;
  a.vx = c->vx;
  a.vy = c->vy;
  a.vz = c->vz;
  a.ax = c->ax;
  a.ay = c->ay;
  a.az = c->az;
  a.aox = c->aox;
  a.aoy = c->aoy;
  a.aoz = c->aoz;
  a.snap = c->snap;
  a.xo = decide && c->nl_on ? c->xo : nullptr;
  a.yo = c->yo;
  a.zo = c->zo;
  a.thr_sq = c->thr_sq;
  a.flags = c->flags;
  a.blk = c->blk;
  a.cnt = fused_cells(c) ? c->cell_cnt : nullptr;
  a.nbins = c->xnbins;
  const int bs = move_block(c), nb = grid_for(c->n, bs);
  a.stride = c->n;
  const auto kern = bs == 64 ? (drift ? k_move<true, 64, false> : k_move<false, 64, false>)
                             : (drift ? k_move<true, kBlock, false> : k_move<false, kBlock, false>);
  kern<<<nb, bs, 0, c->stream>>>(a, ghost_rule(c));
  CAV_HIP(hipGetLastError());
  return CAV_OK;
}

// Images of the moved atoms, and the rebuild decision; after launch_move.
int launch_ghosts(cav_ctx *c, bool decide)
{
  const int bs = move_block(c), nb = grid_for(c->n, bs);
  GhostArgs a;
  a.n = c->n;
  a.nblk = nb;
  // each block reads every block's count: past a million atoms one scan does
  a.scanned = nb > 4096;
  for (int d = 0; d < 3; ++d) a.L[d] = c->L[d];
  a.blk = c->blk;
  a.x = c->x;
  a.y = c->y;
  a.z = c->z;
  a.type = c->type;
  a.id = c->id;
  a.mol = c->mol;
  a.gsrc = c->gsrc;
  a.q = c->q;
  a.xo = decide && c->nl_on ? c->xo : nullptr;
  a.yo = c->yo;
  a.zo = c->zo;
  a.thr_sq = c->thr_sq;
  a.rebuild_test = c->rebuild_test;
  a.flags = c->flags;
  const bool fused = fused_cells(c);
  a.xq = fused ? c->xq : nullptr;
  a.tid = c->tid;
  a.cnt = fused ? c->cell_cnt : nullptr;
  a.bucket = c->bucket;
  a.cap = c->bucket_cap;
  if (a.scanned)
    k_scan_blocks<<<1, kBlock, 0, c->stream>>>(nb, c->blk, c->flags + F_NGHOST, nullptr,
                                               c->flags + F_STOP);
  const auto kern = bs == 64 ? k_ghosts<64, false> : k_ghosts<kBlock, false>;
  kern<<<nb, bs, 0, c->stream>>>(a, ghost_rule(c), bin_rule(c, true));
  CAV_HIP(hipGetLastError());
  return CAV_OK;
}

// Cells and bin-order copies of the images launch_ghosts made.
int launch_cells(cav_ctx *c)
{
  CellBuild a;
  a.n = c->n;
  a.nbins = c->xnbins;
  // one cell per wave where the chip has room, else four (fewer workgroups
  // that add up the counters before theirs)
  a.bpb = c->xnbins <= 4096 ? 16 : 64;
  a.cap = c->bucket_cap;
  a.cnt = c->cell_cnt;
  a.bucket = c->bucket;
  a.xq = c->xq;
  a.tid = c->tid;
  a.start = c->bin_start;
  a.items = c->bin_items;
  a.order = c->order;
  a.binpos = c->binpos;
  a.litems = c->litems;
  a.xqs = c->xqs;
  a.xo = c->xo;
  a.yo = c->yo;
  a.zo = c->zo;
  a.flags = c->flags;
  a.first = nullptr;
  k_cells<false, kCellBlock><<<(c->xnbins + a.bpb - 1) / a.bpb, kCellBlock, 0, c->stream>>>(a, bin_rule(c, true));
  CAV_HIP(hipGetLastError());
  return CAV_OK;
}

// ------------------------------------------------------------- Verlet list --

// Stencil candidates staged in LDS per pass (8 KB of a wave's LDS at 256):
// fewer candidates per pass, more waves per CU, but more passes over the owned
// atoms.  Measured with 128 / 192 / 256 / 384 (us): 262144 ions 226 / 225 / 219
// / 253 beside Ewald_k, 256 replicas 434 / 395 / 384 / 418.
#ifndef CAV_LIST_CAND
#define CAV_LIST_CAND 256
#endif
constexpr int kCand = CAV_LIST_CAND;

// Full Verlet rows: for owned i every owned j != i and every ghost within
// cutoff_extra (strict, dr = pos_i - pos_j rounded as the reference rounds it,
// neighborlist.cpp:531-566).  The reference's half list is the subset with
// owned j > i plus every ghost; both directions are kept so that forces are
// gathered per atom without atomics.  Rows are row-major: nl[i*cap + k].
// With nlb the entries are (also) written as bin-order slots; with nl null
// only the slots are written and F_NL_STALE tells the readers of the index
// rows to fill them first (launch_nl_fill).
//
// One wave per cell: the candidates of the cell's de-duplicated stencil are
// staged in LDS (in stencil order, each cell in bin order), then the cell's
// owned atoms are tested kAPI at a time against 64 candidates per iteration
// (each staged candidate is read once for kAPI independent tests).  Candidates
// come from the cell-ordered packed copy (x, y, z, index) written after the
// bin sort, so staging reads are contiguous per stencil cell; passing
// lanes append in lane order through a ballot and a prefix popcount, so rows
// are written coalesced and in a deterministic order.
//
// Instruction issue bounds it (counters over a launch at N=262144: 20.0 vector
// and 13.1 scalar instructions for each test of 64 pairs, of which the exact
// FP64 distance needs nine; 22.6 and 13.0 before this form).  So the owned atoms
// come by scalar loads, the bounds check of a buffer store stands for the tests
// of a full row and of an idle lane, the atom itself is looked for only in the
// pass that holds it, and a stage's cells are found by bisection with all its
// loads in flight.
// In order: N=262144 144 -> 121 us, 256 replicas (540000 atoms at rho 0.2 to
// 0.8) 444 -> 332 us.
constexpr int kAPI = 4;  // owned atoms tested per staged candidate

// Cells per workgroup, one wave each (measured at N=262144: 1 -> 0.307 ms,
// 2 -> 0.318, 4 -> 0.323, 8 -> 0.374; the build is not occupancy bound).
// Cells go to workgroups in plain order: giving each XCD a contiguous run of
// cells (as the pair kernel does with atoms) cut the fetched bytes from 90 to
// 34 MB per build but made it slower, 0.251 -> 0.288 ms.
#ifndef CAV_LIST_WPB
#define CAV_LIST_WPB 1
#endif
constexpr int kListWaves = CAV_LIST_WPB;

static int list_grid(long cells) { return (int)((cells + kListWaves - 1) / kListWaves); }

// One atom's row as buffers of cap entries: a store past the end is dropped by
// the bounds check, so neither a full row nor a lane with nothing to store
// (offset -1) needs a branch of its own.
template <bool NL, bool NLL, bool NLB>
struct Rows {
  __amdgpu_buffer_rsrc_t nl, nll, nlb;
  __device__ __forceinline__ void set(int *pl, unsigned short *pll, int *plb, long at, int cap)
  {
    constexpr int raw = 0x00027000;  // untyped 32-bit data
    if constexpr (NL) nl = __builtin_amdgcn_make_buffer_rsrc(pl + at, 0, 4 * cap, raw);
    if constexpr (NLL) nll = __builtin_amdgcn_make_buffer_rsrc(pll + at, 0, 2 * cap, raw);
    if constexpr (NLB) nlb = __builtin_amdgcn_make_buffer_rsrc(plb + at, 0, 4 * cap, raw);
  }
  // entry e4 / 4 of the row: candidate (tag) at staging position pos
  __device__ __forceinline__ void put(int e4, double tag, int pos) const
  {
    if constexpr (NL) __builtin_amdgcn_raw_buffer_store_b32(cpos_index(tag), nl, e4, 0, 0);
    if constexpr (NLL)
      __builtin_amdgcn_raw_buffer_store_b16((unsigned short)pos, nll, e4 >> 1, 0, 0);
    if constexpr (NLB) __builtin_amdgcn_raw_buffer_store_b32(cpos_slot(tag), nlb, e4, 0, 0);
  }
};

// An owned atom against one candidate per lane; SELF: lane `self`, if there is
// one, holds the atom itself, which is left out.  c4: 4 per entry of the row.
template <bool SELF, class R>
__device__ __forceinline__ void list_test(double px, double py, double pz, const double4 &q,
                                          double rce2, int lane, int self, int pos, const R &row,
                                          int &c4)
{
  const double dx = xsub(px, q.x), dy = xsub(py, q.y), dz = xsub(pz, q.z);
  bool pass = dot_rn(dx, dy, dz) < rce2;
  if constexpr (SELF) pass = pass && lane != self;
  // the compare's lanes as a scalar mask
  const u64t mask = __builtin_amdgcn_ballot_w64(pass);
  if (mask) {
    // the lane's rank among the passing lanes, after the row's entries so far
    const unsigned pre = __builtin_amdgcn_mbcnt_hi(
        (unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
    row.put(pass ? c4 + 4 * (int)pre : -1, q.w, pos);
    c4 += 4 * (int)__popcll(mask);
  }
}

// The row outputs a build writes (index rows nl, staging positions nll,
// bin-order slots nlb) are template flags, so the append path of the inner
// loop carries only the stores the launch needs.
//
// PACKED: candidates come from the bin-ordered records that the pair kernel
// gathers, with `items` the slots' atoms; else from a copy made for the list
// (x, y, z, index and slot).
template <bool NL, bool NLL, bool NLB, bool PACKED>
__global__ __launch_bounds__(64 * kListWaves) void k_list_wave(int n, int nwaves, int nbx, int nby, int nbz,
                                                  int cap, double rce2, const double4 *cpos,
                                                  const int *st_off, const int *st,
                                                  const int *start, const int *items, int *nl,
                                                  int *nn, int *flags, const int *cond,
                                                  const RepDev *rep, const int2 *waves,
                                                  unsigned short *nll, int *nlb, int split)
{
  // Each wave builds the rows of one cell on its own (wave-local LDS, no
  // block barrier).  The wave index is read as a scalar so that everything
  // derived from the cell stays in scalar registers.
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int w = (int)((long)blockIdx.x * kListWaves + wv);
  if (w >= nwaves) return;
  const int lane = threadIdx.x & 63;
  int b = w;
  bool shell = false;
  if (waves) {  // batched replicas: arrays shifted to the wave's
    const int2 v = waves[w];
    const RepDev &r = rep[v.y];
    n = r.n;
    flags += 16 * v.y;
    cond = flags + F_REBUILD;
    shell = v.x < 0;
    b = shell ? -1 - v.x : v.x;
    nbx = r.nb[0], nby = r.nb[1], nbz = r.nb[2];
    cpos += r.base;
    items += r.base;
    start += r.cbase + v.y;  // every replica's cell starts carry one closing entry
    st_off += r.cbase;
    nn += r.obase;
    nlb += (long)r.obase * cap;
  } else if (nbx) {
    const int ix = nbx - 2, iy = nby - 2, ni = ix * iy * (nbz - 2);
    shell = w >= ni;
    const int y = w / ix;
    b = shell ? 64 * (w - ni) : w - y * ix + 1 + nbx * (y % iy + 1 + nby * (y / iy + 1));
  }
  if (cond && !*cond) return;
  // with `split` waves per cell (blockIdx.y), this one takes every split-th
  // group of kAPI owned atoms
  const int part = blockIdx.y;
  if (!waves && w == 0 && part == 0 && threadIdx.x == 0) flags[F_NL_STALE] = NL ? 0 : 1;
  // staged candidates (x, y, z, index and slot) in the cell's stencil order; a stage is
  // padded to a multiple of 64 with far-away entries so every lane tests one
  __shared__ double4 sc_[kListWaves][kCand];
  double4 *sc = sc_[wv];
  __shared__ int s_off_[kListWaves][32], s_shift_[kListWaves][32];
  int *s_off = s_off_[wv], *s_shift = s_shift_[wv];
  u64t todo = 1;
  if (shell) {  // the cells among the next 64 that are of the layer and hold an owned atom
    const int c = b + lane, cx = c % nbx, cy = c / nbx % nby, cz = c / (nbx * nby);
    bool has = c < nbx * nby * nbz && (cx == 0 || cx == nbx - 1 || cy == 0 || cy == nby - 1 ||
                                       cz == 0 || cz == nbz - 1);
    if (has) {
      const int first = start[c];
      has = first < start[c + 1] && items[first] < n;  // owned atoms come first in a sorted bin
    }
    todo = __ballot(has);
  }
  for (int b0 = b; todo; todo &= todo - 1) {
    b = b0 + __ffsll(todo) - 1;
    // the stencil's cell ranges, loaded by lanes 0..ns-1 at once, and the
    // cell's own atoms: two chains of loads, side by side
    const int s0 = start[b], e0 = start[b + 1];
    const int sb = st_off[b], ns = st_off[b + 1] - sb;  // <= 27 stencil cells
    int cell = -1, cb = 0, cn = 0;
    if (lane < ns) {
      cell = st[sb + lane];
      cb = start[cell];
      cn = start[cell + 1] - cb;
    }
    int no = 0;  // owned atoms come first in a sorted bin
    for (int t = s0; t < e0; t += 64) {
      const int v = (t + lane < e0) ? items[t + lane] : n;
      no += __popcll(__ballot(v < n));
    }
    if (no <= kAPI * part) continue;
    // running offsets of the ranges in staging order (stencil cells in order,
    // each in bin order), and what takes a staging position to its slot
    int incl = cn;
    for (int o = 1; o < 32; o <<= 1) {
      const int v = __shfl_up(incl, o, 64);
      if (lane >= o) incl += v;
    }
    const int total = __builtin_amdgcn_readlane(incl, 31);  // lanes past ns add nothing
    if (lane < 32) {
      s_off[lane] = incl - cn;
      s_shift[lane] = cb - (incl - cn);
    }
    // staging position of the cell's first atom: where a row's own atom is left out
    const int centre = __ffsll(__ballot(cell == b)) - 1;
    const int own0 = __builtin_amdgcn_readlane(incl - cn, centre);
    __syncwarp();
    for (int og = 0; og < no; og += 64) {
      const int gsize = (no - og) < 64 ? (no - og) : 64;
      int cnt = 0;  // lane t: the row count of owned atom og + t
      for (int mbase = 0; mbase < total; mbase += kCand) {
        // stage candidates mbase .. mbase+m-1 of the flattened stencil: each
        // lane finds the cells of its kCand/64 by bisection and issues their
        // loads together
        const int m = (total - mbase) < kCand ? (total - mbase) : kCand;
        const int mpad = (m + 63) & ~63;
        int at[kCand / 64];
        double4 cv[kCand / 64];
#pragma unroll
        for (int q = 0; q < kCand / 64; ++q) at[q] = 0;
#pragma unroll
        for (int step = 16; step > 0; step >>= 1)
#pragma unroll
          for (int q = 0; q < kCand / 64; ++q)
            if (s_off[at[q] + step] <= mbase + 64 * q + lane) at[q] += step;
#pragma unroll
        for (int q = 0; q < kCand / 64; ++q) {
          const int g = mbase + 64 * q + lane;
          at[q] = g < total ? s_shift[at[q]] + g : s0;
        }
#pragma unroll
        for (int q = 0; q < kCand / 64; ++q) cv[q] = cpos[at[q]];
#pragma unroll
        for (int q = 0; q < kCand / 64; ++q) {
          cv[q].x = 64 * q + lane < m ? cv[q].x : 1e300;
          if constexpr (PACKED) cv[q].w = cpos_tag(-1, at[q]);
          sc[64 * q + lane] = cv[q];
        }
        __syncwarp();
        for (int o0 = kAPI * part; o0 < gsize; o0 += kAPI * split) {
          // the kAPI owned atoms are the same for every lane: positions (by
          // scalar loads), rows and row lengths in scalar registers.  Empty
          // places of the group and padding sit at x = -+1e300: their squared
          // distance to anything is +inf, so they never pass the cutoff test
          double px[kAPI], py[kAPI], pz[kAPI];
          Rows<NL, NLL, NLB> row[kAPI];
#pragma unroll
          for (int u = 0; u < kAPI; ++u) {
            const int src = o0 + u;  // < 64: o0 is a multiple of kAPI below 64
            // (past the group: some other slot's values, or the arrays' padding)
            typedef const __attribute__((address_space(4))) double *scalar_d;
            const long at = (long)s0 + og + src;
            const scalar_d own = (scalar_d)(cpos + at);
            px[u] = own[0];
            py[u] = own[1];
            pz[u] = own[2];
            int i = PACKED ? ((const __attribute__((address_space(4))) int *)items)[at]
                           : cpos_index(own[3]);
            if (src >= gsize) {
              px[u] = -1e300;
              i = 0;
            }
            row[u].set(nl, nll, nlb, (long)i * cap, cap);
          }
          // the row lengths, 4 per entry (an array would be copied as a whole)
          static_assert(kAPI == 4, "four atoms a group");
          int c0 = 4 * __builtin_amdgcn_readlane(cnt, o0), c1 = 4 * __builtin_amdgcn_readlane(cnt, o0 + 1),
              c2 = 4 * __builtin_amdgcn_readlane(cnt, o0 + 2), c3 = 4 * __builtin_amdgcn_readlane(cnt, o0 + 3);
          // the group's own places in the staging order, where no lane passes
          const int self0 = own0 + og + o0 - mbase;
          for (int cc = 0; cc < mpad; cc += 64) {
            const int idx = cc + lane;
            const double4 q = sc[idx];
            if ((unsigned)(self0 - cc + kAPI - 1) < 64u + kAPI - 1) {
              const int self = self0 - cc;
              list_test<true>(px[0], py[0], pz[0], q, rce2, lane, self, mbase + idx, row[0], c0);
              list_test<true>(px[1], py[1], pz[1], q, rce2, lane, self + 1, mbase + idx, row[1], c1);
              list_test<true>(px[2], py[2], pz[2], q, rce2, lane, self + 2, mbase + idx, row[2], c2);
              list_test<true>(px[3], py[3], pz[3], q, rce2, lane, self + 3, mbase + idx, row[3], c3);
            } else {
              list_test<false>(px[0], py[0], pz[0], q, rce2, lane, 0, mbase + idx, row[0], c0);
              list_test<false>(px[1], py[1], pz[1], q, rce2, lane, 0, mbase + idx, row[1], c1);
              list_test<false>(px[2], py[2], pz[2], q, rce2, lane, 0, mbase + idx, row[2], c2);
              list_test<false>(px[3], py[3], pz[3], q, rce2, lane, 0, mbase + idx, row[3], c3);
            }
          }
          cnt = lane == o0 ? c0 >> 2 : lane == o0 + 1 ? c1 >> 2 : lane == o0 + 2 ? c2 >> 2
              : lane == o0 + 3 ? c3 >> 2 : cnt;
        }
        __syncwarp();
      }
      if (lane < gsize && lane / kAPI % split == part) {
        const int i = items[s0 + og + lane];
        nn[i] = cnt < cap ? cnt : cap;
        // the longest row is needed only to regrow the list after an overflow:
        // one device-wide atomic per overflowing row, none otherwise
        if (cnt > cap) {
          flags[F_OVERFLOW] = 1;
          atomicMax(flags + F_MAXNB, cnt);
        }
      }
    }
  }
}

// k_list_wave for the outputs that are not null (index rows, staging
// positions, bin-order slots: the combinations the single system and the
// batched replicas use)
static void launch_list_wave(hipStream_t st, int n, int nbins, const int *xnb, int cap, double rce2,
                             const double4 *cpos, const int *st_off, const int *stc,
                             const int *start, const int *items, int *nl, int *nn, int *flags,
                             const int *cond, const RepDev *rep, const int2 *waves, int nwaves,
                             unsigned short *nll, int *nlb, bool packed)
{
  // Waves per cell: small grids leave CUs idle, and a wave's chain over its
  // atoms' groups is then the kernel's time; every wave stages the candidates
  // for itself, so a full chip keeps one.  Measured with 1 / 2 / 3 / 6 waves
  // (us): 125 cells 24 / 16 / 13 / 11, 1000 cells 34 / 23 / 20 / 17, 2744 cells
  // 45 / 34 / 33 / 34, 8000 cells 77 / 76 / 84 / 104.
  const int split = std::max(1, std::min(6, 8192 / nbins));
  // One wave per cell, or on a grid with a ghost layer (xnb: its cells per
  // axis) one per inner cell and one per 64 of all cells for what owned atoms
  // the layer holds (positions on the upper face)
  int bx = 0, by = 0, bz = 0;
  if (!waves) {
    nwaves = nbins;
    if (xnb) {
      bx = xnb[0] + 2, by = xnb[1] + 2, bz = xnb[2] + 2;
      nwaves = xnb[0] * xnb[1] * xnb[2] + (nbins + 63) / 64;
    }
  }
  const dim3 g(list_grid(nwaves), split), blk(64 * kListWaves);
#define CAV_LISTW(A, B, C, D)                                                                    \
  k_list_wave<A, B, C, D><<<g, blk, 0, st>>>(n, nwaves, bx, by, bz, cap, rce2, cpos,             \
                                             st_off, stc, start, items, nl, nn, flags, cond, rep, \
                                             waves, nll, nlb, split)
  if (nlb && packed)
    CAV_LISTW(false, false, true, true);
  else if (nlb)
    CAV_LISTW(false, false, true, false);
  else if (nll)
    CAV_LISTW(true, true, false, false);
  else
    CAV_LISTW(true, false, false, false);
#undef CAV_LISTW
}

// all_atom_test_function (neighborlist.cpp:161-191): every owned j != i and
// every ghost, no distance test.
__global__ void k_list_all(int n, int cap, int *nl, int *nn, int *flags, const int *cond)
{
  if (cond && !*cond) return;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const int tot = n + flags[F_NGHOST];
  int cnt = 0;
  for (int j = 0; j < tot; ++j) {
    if (j == i) continue;
    if (cnt < cap) nl[(long)i * cap + cnt] = j;
    ++cnt;
  }
  nn[i] = cnt < cap ? cnt : cap;
  if (cnt > cap) {
    flags[F_OVERFLOW] = 1;
    atomicMax(flags + F_MAXNB, cnt);
  }
}

// The cells the list was built from, kept for the cell-staged pair kernel:
// later re-binnings (the LJ cell walk, energy and point queries) rewrite
// bin_start/bin_items, while the list's staging positions refer to these.
// binpos is the inverse permutation (slot -> position in bin order).
__global__ void k_list_bins(int n, int nbins, long cap_total, const int *start, const int *items,
                            int *lstart, int *litems, int *binpos, const int *flags, const int *cond)
{
  if (cond && !*cond) return;
  const long t = (long)blockIdx.x * kBlock + threadIdx.x;
  if (t <= nbins) lstart[t] = start[t];
  if (t < (long)n + flags[F_NGHOST] && t < cap_total) {
    const int a = items[t];
    litems[t] = a;
    binpos[a] = (int)t;
  }
}

int launch_list(cav_ctx *c, bool conditional, bool packed)
{
  const int *cond = conditional ? c->flags + F_REBUILD : nullptr;
  // staging positions (and the cells they refer to) only for the cell-staged
  // pair kernel; a build that writes them makes them valid for its list, one
  // that does not invalidates them (known at once for an unconditional build,
  // after the flags are read back for a conditional one)
  const bool with_nll = c->pair_kind == CAV_PAIRS_CELLS && c->nll && !c->all_atom_test;
  c->nll_pending = with_nll;
  if (!conditional) c->nll_built = with_nll;
  // bin-order slots of the entries, for the row kernel's gathers from the
  // bin-ordered copies: valid on the same terms
  const bool with_nlb = c->pair_kind == CAV_PAIRS_AUTO && c->nlb && !c->all_atom_test;
  // the grid the list build's binning used (launch_bins with for_list)
  const bool xg = list_on_ghost_grid(c);
  c->nlb_pending = with_nlb;
  if (!conditional) c->nlb_built = with_nlb;
  if (c->all_atom_test)
    k_list_all<<<grid_for(c->n), kBlock, 0, c->stream>>>(c->n, c->nl_cap, c->nl, c->nn, c->flags,
                                                        cond);
  else
    launch_list_wave(c->stream, c->n, xg ? c->xnbins : c->nbins, xg ? c->nb : nullptr, c->nl_cap,
                     c->rce2, packed ? c->xqs : c->cpos,
                     xg ? c->d_xst_off : c->d_st_off, xg ? c->d_xst : c->d_st, c->bin_start,
                     packed ? c->litems : c->bin_items, with_nlb ? nullptr : c->nl, c->nn, c->flags, cond, nullptr,
                     nullptr, 0, with_nll ? c->nll : nullptr, with_nlb ? c->nlb : nullptr, packed);
  // (the bin order itself, litems and binpos, was kept by the list build's
  // binning; the cell-staged kernel also needs the cell starts)
  if (with_nll) {
    const long tot = (long)c->n + c->gcap;
    k_list_bins<<<grid_for(tot > c->nbins + 1 ? tot : c->nbins + 1), kBlock, 0, c->stream>>>(
        c->n, c->nbins, tot, c->bin_start, c->bin_items, c->lstart, c->litems, c->binpos, c->flags,
        cond);
  }
  CAV_HIP(hipGetLastError());
  return CAV_OK;
}

// Index rows from the bin-order slots of the last list build, when that build
// wrote the slots only (F_NL_STALE); the flag is cleared by a kernel of its own
// after every entry is written.
__global__ void k_nl_fill(long entries, int cap, long slots, const int *nlb, const int *litems,
                          const int *nn, int *nl, const int *flags)
{
  if (!flags[F_NL_STALE]) return;
  const long e = (long)blockIdx.x * kBlock + threadIdx.x;
  if (e >= entries || e % cap >= nn[e / cap]) return;
  const int t = nlb[e];
  if (t >= 0 && t < slots) nl[e] = litems[t];
}

__global__ void k_nl_fresh(int *flags) { flags[F_NL_STALE] = 0; }

int launch_nl_fill(cav_ctx *c)
{
  if (!c->nlb || !c->nl || c->all_atom_test) return CAV_OK;
  const long entries = (long)c->n * c->nl_cap;
  k_nl_fill<<<grid_for(entries), kBlock, 0, c->stream>>>(entries, c->nl_cap, (long)c->n + c->gcap,
                                                          c->nlb, c->litems, c->nn, c->nl,
                                                          c->flags);
  k_nl_fresh<<<1, 1, 0, c->stream>>>(c->flags);
  CAV_HIP(hipGetLastError());
  return CAV_OK;
}

// pos_old = pos, ghost_pos_old = ghost pos (neighborlist.cpp:302-303,568-569).
__global__ void k_save_old(int n, long cap_total, const double *x, const double *y, const double *z,
                           double *xo, double *yo, double *zo, int *flags, const int *cond)
{
  if (cond && !*cond) return;
  const long a = (long)blockIdx.x * kBlock + threadIdx.x;
  const int G = flags[F_NGHOST];
  if (a == 0) flags[F_NGHOST_OLD] = G;
  if (a >= (long)n + G || a >= cap_total) return;
  xo[a] = x[a];
  yo[a] = y[a];
  zo[a] = z[a];
}

int launch_save_old(cav_ctx *c, bool conditional)
{
  if (c->all_atom_test) return CAV_OK;  // the reference returns before saving
  const int *cond = conditional ? c->flags + F_REBUILD : nullptr;
  const long tot = (long)c->n + c->gcap;
  k_save_old<<<grid_for(tot), kBlock, 0, c->stream>>>(c->n, tot, c->x, c->y, c->z, c->xo, c->yo,
                                                     c->zo, c->flags, cond);
  CAV_HIP(hipGetLastError());
  return CAV_OK;
}

// ---------------------------------------------------------- batched replicas --
//
// The same exchange for every replica of a cav_batch at once, in the same
// kernels: each workgroup works on one replica (RepGrid: the grid row, or dealt
// to an XCD), whose decisions (ghost count, rebuild) live in its own 16 flag
// words.  256 replicas (540000 atoms, 1.5 million with their images), a step's
// exchange without the list: 455 us as thirteen kernels of its own, now 220.

// Counters before every bpb-th cell of a replica, for grids on which each
// workgroup of k_cells adding them up itself would read too much.
__global__ __launch_bounds__(kCellBlock) void kb_cell_first(const RepDev *rep, int bpb, int blocks,
                                                            const u64t *cnt, u64t *first)
{
  const RepDev &r = rep[blockIdx.x];
  cnt += r.cbase;
  first += (long)blockIdx.x * blocks;
  const int nb = (r.nbins + bpb - 1) / bpb, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  __shared__ u64t part[kCellBlock / 64];
  u64t carry = 0;
  for (int k0 = 0; k0 < nb; k0 += kCellBlock) {
    const int k = k0 + threadIdx.x;
    u64t v = 0;
    if (k < nb)
      for (int c = k * bpb; c < min(r.nbins, (k + 1) * bpb); ++c) v += cnt[c];
    u64t inc = v;
    for (int o = 1; o < 64; o <<= 1) {
      const u64t u = __shfl_up(inc, o, 64);
      if (lane >= o) inc += u;
    }
    if (lane == 63) part[wv] = inc;
    __syncthreads();
    u64t before = carry;
    for (int q = 0; q < kCellBlock / 64; ++q) {
      if (q < wv) before += part[q];
      carry += part[q];
    }
    if (k < nb) first[k] = before + inc - v;
    __syncthreads();
  }
}

// Threads per workgroup of the move and the images: one wave, whose scattered
// stores and atomics wait for no other (256 replicas: images 152 -> 131 us
// against four waves); large replicas keep four, since each workgroup adds up
// the counts of all of its replica's.
static int batch_block(const cav_batch *b) { return b->maxn <= 65536 ? 64 : kBlock; }

// Cells per workgroup of k_cells: two a wave; on large grids sixteen (fewer
// workgroups that add up the counters before theirs)
static int cells_per_block(const cav_batch *b) { return b->maxcells > 4096 ? 64 : 8; }

int batch_cells_alloc(cav_batch *b)
{
  b->maxcells = 0;
  size_t room = 0;
  for (RepDev &r : b->reps) {
    b->maxcells = std::max(b->maxcells, r.nbins);
    // twice the replica's mean cell and some, in whole half waves, as the
    // single system: the room stays in proportion to its cells and atoms
    const double want = 2.0 * b->rce * b->rce * b->rce * r.n / (r.L[0] * r.L[1] * r.L[2]) + 32;
    r.bcap = (int)(std::min(1024.0, want + 31) / 32) * 32;
    r.bcap = std::max(r.bcap, b->hreps[&r - b->reps.data()].bcap);
    r.bbase = (long)room;
    room += (size_t)r.bcap * r.nbins;
  }
  b->scan_blocks = grid_for(b->maxn, batch_block(b));
  const int blocks = (b->maxcells + cells_per_block(b) - 1) / cells_per_block(b);
  void **bufs[] = {(void **)&b->cell_cnt, (void **)&b->bucket, (void **)&b->cell_first,
                   (void **)&b->gblk};
  const size_t bytes[] = {sizeof(u64t) * b->ncells, sizeof(int) * room,
                          b->maxcells > 65536 ? sizeof(u64t) * (size_t)blocks * b->B : 0,
                          sizeof(int) * (size_t)b->B * b->scan_blocks};
  for (int k = 0; k < 4; ++k) {
    if (*bufs[k]) (void)hipFree(*bufs[k]);
    *bufs[k] = nullptr;
    if (bytes[k]) BAT_HIP(hipMalloc(bufs[k], bytes[k]));
  }
  return CAV_OK;
}

// cells_fit for every replica of a batch, each within a megabyte or what its
// slots take.  `grown`: kernel arguments have changed.
int batch_cells_fit(cav_batch *b, bool *grown)
{
  *grown = false;
  for (int k = 0; k < b->B; ++k) {
    RepDev &r = b->reps[k];
    const int most = b->h_flags[16 * k + F_MAXCELL];
    const long cap = crowd_cap(most);
    if (most <= r.bcap || cap * r.nbins > std::max(1L << 18, 32L * ((long)r.n + r.gcap))) continue;
    b->hreps[k].bcap = (int)cap;  // (a new layout keeps it)
    *grown = true;
  }
  if (!*grown) return CAV_OK;
  CAV_TRY(batch_cells_alloc(b));
  BAT_HIP(hipMemcpyAsync(b->d_rep, b->reps.data(), sizeof(RepDev) * b->B, hipMemcpyHostToDevice, b->stream));
  BAT_HIP(hipStreamSynchronize(b->stream));
  return CAV_OK;
}

// Owned atoms of every replica drifted (its Ewald_k then starts beside the
// rest) or only wrapped, images, the rebuild
// decision (`drift` false: every list is rebuilt, F_REBUILD is already set),
// cells, packed copies and Verlet rows.
int batch_neighbor(cav_batch *b, bool drift, double dt)
{
  const int bs = batch_block(b);
  const dim3 own_grid = batch_grid(b, b->scan_blocks);
  MoveArgs m;
  m.n = 0;
  m.dt = dt;
  m.x = b->x;
  m.y = b->y;
  m.z = b->z;
  m.vx = b->vx;
  m.vy = b->vy;
  m.vz = b->vz;
  m.ax = b->ax;
  m.ay = b->ay;
  m.az = b->az;
  m.aox = m.aoy = m.aoz = nullptr;
  m.snap = b->snap;
  m.xo = drift ? b->xo : nullptr;
  m.yo = b->yo;
  m.zo = b->zo;
  m.thr_sq = b->thr_sq;
  m.flags = b->flags;
  m.blk = b->gblk;
  m.cnt = b->cell_cnt;
  m.nbins = 0;
  m.stride = b->nown;
  m.reps = batch_reps(b);
  m.gc = b->ghost_cutoff;
  const auto move = bs == 64 ? (drift ? k_move<true, 64, true> : k_move<false, 64, true>)
                             : (drift ? k_move<true, kBlock, true> : k_move<false, kBlock, true>);
  move<<<own_grid, bs, 0, b->stream>>>(m, GhostRule{});
  BAT_HIP(hipGetLastError());
  if (drift && b->ek_on) CAV_TRY(batch_ewald_k_fork(b));
  GhostArgs g;
  g.n = g.nblk = 0;
  g.scanned = 0;
  g.blk = b->gblk;
  g.x = b->x;
  g.y = b->y;
  g.z = b->z;
  g.type = b->type;
  g.id = b->id;
  g.mol = g.gsrc = nullptr;
  g.q = b->q;
  g.xo = drift ? b->xo : nullptr;
  g.yo = b->yo;
  g.zo = b->zo;
  g.thr_sq = b->thr_sq;
  g.rebuild_test = 0;
  g.flags = b->flags;
  g.xq = b->xq;
  g.tid = b->tid;
  g.cnt = b->cell_cnt;
  g.bucket = b->bucket;
  g.cap = 0;
  g.reps = batch_reps(b);
  g.gc = b->ghost_cutoff;
  g.cinv = b->cinv;
  const auto ghosts = bs == 64 ? k_ghosts<64, true> : k_ghosts<kBlock, true>;
  ghosts<<<own_grid, bs, 0, b->stream>>>(g, GhostRule{}, BinRule{});
  CellBuild a;
  a.n = a.nbins = 0;
  a.bpb = cells_per_block(b);
  a.cap = 0;
  a.cnt = b->cell_cnt;
  a.bucket = b->bucket;
  a.xq = b->xq;
  a.tid = b->tid;
  a.start = b->bin_start;
  a.items = b->bin_items;
  a.order = b->order;
  a.binpos = nullptr;
  a.litems = b->litems;
  a.xqs = b->xqs;
  a.xo = b->xo;
  a.yo = b->yo;
  a.zo = b->zo;
  a.flags = b->flags;
  a.reps = batch_reps(b);
  a.cinv = b->cinv;
  a.first = b->cell_first;
  const int blocks = (b->maxcells + a.bpb - 1) / a.bpb;
  if (a.first)
    kb_cell_first<<<b->B, kCellBlock, 0, b->stream>>>(b->d_rep, a.bpb, blocks, b->cell_cnt,
                                                      b->cell_first);
  k_cells<true, kBatchCellBlock><<<batch_grid(b, blocks), kBatchCellBlock, 0, b->stream>>>(a, BinRule{});
  launch_list_wave(b->stream, 0, b->ncells, nullptr, b->cap, b->rce2, b->xqs, b->st_off, b->st,
                   b->bin_start, b->litems, nullptr, b->nn, b->flags, nullptr, b->d_rep, b->waves,
                   b->nwaves, nullptr, b->nlb, true);
  BAT_HIP(hipGetLastError());
  return CAV_OK;
}

}  // namespace cav
