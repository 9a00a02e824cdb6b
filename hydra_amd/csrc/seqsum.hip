// seqsum.hip -- the exact value of a left-to-right floating-point sum.
//
// gfortran evaluates SUM(a) and the explicit accumulation loops of the
// reference (contours.f90:330-336, evolution.f90:553) as
// s = ((a(1) + a(2)) + a(3)) + ..., each addition rounded.  Those sums feed
// the state (the PV mean removed by con2grid, the rms vorticity inside the
// integrating factors), and a one-ulp change there alters surgery decisions
// within a hundred steps, so the GPU must produce the very same double.
//
// Method (speculate, then verify every accepted step):
//   * Translation property.  While the partial sums stay inside one binade
//     [2^E, 2^(E+1)) of one sign, every addition rounds on the grid
//     u = 2^(E-52) and s_(j+1) = s_j + RN_u(x_j): a run adds the same D to
//     any start on the grid whose run stays inside, provided the starts
//     agree mod 2u (exact ties round to even).  Simulating the run from g
//     and from g+u gives both translations D0, D1.
//   * Classes.  A run that crosses binades is a translation per residue
//     class of its start: for a start S = G_c + Delta, G_c = g + c u (u the
//     grid of g's binade, c < M) and Delta a multiple of M u = 2 u_max (u_max
//     the coarsest grid the run visits), every rounding of the run from S
//     happens on the grid it happens on from G_c, displaced by Delta, as
//     long as every partial sum stays in its binade: it ends exactly at
//     E_c + Delta.  A table holds E_c and the admissible Delta interval of
//     each class.
//   * Chunks of 64 values are simulated in parallel from a guessed start
//     (prefix of the chunk totals); windows of 16 chunks that
//     stay in one binade fold into a composite by row scans; the other
//     windows get a table, 64 classes walked at once, one to a lane: over
//     each chunk by its translation where it has one, value by value where
//     it changes binade.  The four windows of a workgroup then make the
//     segment's table the same way, and above kTop segments sixteen tables
//     at a time make the next level's.
//   * The chain takes the top level's tables in order: the class from the
//     low mantissa bits of S - g, a range check, S = E_c + Delta.  A start
//     that its table does not cover descends to the entry's parts, at last
//     to windows summed in order.
// Every accepted translation is exact by construction and every rejected
// piece is summed in order, so the result is the sequential sum bit for bit.
//
// What bounds it: latency -- a workgroup is one wavefront with a serial walk
// of 64 values (about 2 us), and the chain's lookups (about 0.1 us each) are
// serial; a dependent FP64 add takes 2.3 ns from registers, 4.3 ns from LDS
// on gfx950.  A sum whose producer has made the chunk totals takes (before:
// windows of 1024 values with 8 classes in four launches)
//   2^20 values  31 us segments + 12 fold + 8 chain   (118)
//   2^18         25 + 13                               (61)
//   2^16         22 + 9                                (53)
//   2^10         11 in one launch                      (38)
#include <atomic>
#include <mutex>

#include "hyd_internal.h"

namespace hyd {

static constexpr int kChunk = 64;    // values per chunk
static constexpr int kWin = 16;      // chunks per window
static constexpr int kWins = 4;      // windows per segment (one workgroup)
static constexpr int kSegVals = kChunk * kWin * kWins;
static constexpr int kClasses = 64;  // classes of a table, one to a lane
static constexpr int kFold = 16;     // entries folded into one of the next level
static constexpr int kTop = 64;      // most entries of the level that the chain takes
static constexpr int kChainWaves = 16;
static constexpr int kGroup = kTop / kChainWaves;  // entries of one of its wavefronts
static constexpr int kMaxLevels = 6;
static constexpr int64_t kSeqOwnTotals = 512 * (int64_t)kSegVals;

// A table: M classes (0: none; -1: the entry's sum starts at the very
// beginning, c[0].e is its exact end), emax the coarsest binade its runs visit.
// Class c: its start G_c, the end E_c from there, the displacements.
struct __align__(16) SeqClass {
  double s, e, lo, hi;
};
struct __align__(16) SeqTab {
  double g;
  int32_t M, emax;
  SeqClass c[kClasses];
};

// A window of chunks that stays in one binade, folded: a start S in g's
// binade, p grid steps (mod 2) from g and inside [lo_p, hi_p], ends at
// S + d_p.
struct SeqComp {
  double g, d0, d1, lo0, hi0, lo1, hi1;
  int32_t ok, eb;
};

__device__ __forceinline__ int binade(double x) {
  return (int)((__double_as_longlong(x) >> 52) & 0x7ff);
}

__device__ __forceinline__ double pow2_field(int eb) {  // 2^(eb-1023)
  return __longlong_as_double((int64_t)eb << 52);
}

// Is a run from start x (binade eb, same sign as g) strictly inside the
// binade with a 4-ulp margin, given extremes [lo,hi] relative to g?
__device__ __forceinline__ bool run_inside(double x, int eb, double lo, double hi) {
  const double bl = pow2_field(eb), bh = pow2_field(eb + 1), m = 4.0 * bl * 0x1p-52;
  const double ax = fabs(x);
  const double rlo = (x < 0.0) ? -hi : lo;
  const double rhi = (x < 0.0) ? -lo : hi;
  return ax + rlo > bl + m && ax + rhi < bh - m;
}

// ---- wavefront primitives -------------------------------------------------
template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) {
  return __builtin_amdgcn_mov_dpp(v, CTRL, 0xf, 0xf, false);
}
template <int CTRL>
__device__ __forceinline__ double dpp_d(double x) {
  const int lo = dpp_i<CTRL>(__double2loint(x));
  const int hi = dpp_i<CTRL>(__double2hiint(x));
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

// Inclusive scans inside each DPP row of 16 lanes.
__device__ __forceinline__ double row_incl_add(double v) {
  const int rl = lane_id() & 15;
  double t;
  t = dpp_d<0x111>(v); if (rl >= 1) v = t + v;
  t = dpp_d<0x112>(v); if (rl >= 2) v = t + v;
  t = dpp_d<0x114>(v); if (rl >= 4) v = t + v;
  t = dpp_d<0x118>(v); if (rl >= 8) v = t + v;
  return v;
}

// GF(2) affine maps p -> k ? p ^ c : c packed as (k << 1) | c; "then" applies
// the earlier map t first.
__device__ __forceinline__ int map_then(int t, int v) {
  const int kv = v >> 1, cv = v & 1, kt = t >> 1, ct = t & 1;
  return ((kv & kt) << 1) | (kv ? (ct ^ cv) : cv);
}
__device__ __forceinline__ int row_incl_map(int v) {
  const int rl = lane_id() & 15;
  int t;
  t = dpp_i<0x111>(v); if (rl >= 1) v = map_then(t, v);
  t = dpp_i<0x112>(v); if (rl >= 2) v = map_then(t, v);
  t = dpp_i<0x114>(v); if (rl >= 4) v = map_then(t, v);
  t = dpp_i<0x118>(v); if (rl >= 8) v = map_then(t, v);
  return v;
}

__device__ __forceinline__ int segkey(double x) {
  return (int)((uint64_t)__double_as_longlong(x) >> 52);  // sign and exponent
}
// Binades whose grid and its inverse are ordinary numbers; sums below or
// above are left to the in-order path.
__device__ __forceinline__ bool binade_ok(int eb) { return eb >= 64 && eb <= 2045; }

__device__ __forceinline__ int parity_of(double num, double uinv) {
  // num is an exact multiple of u = 1/uinv (a power of two), |num/u| < 2^53
  return (int)((long long)(num * uinv) & 1);
}

// Wavefront sum in every lane and inclusive scan (any order: for guesses).
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) v += __shfl_xor(v, o);
  return v;
}
__device__ __forceinline__ double wave_incl_add(double v) {
  const int l = lane_id(), rl = l & 15;
  double t;
  t = dpp_d<0x111>(v); if (rl >= 1) v = t + v;
  t = dpp_d<0x112>(v); if (rl >= 2) v = t + v;
  t = dpp_d<0x114>(v); if (rl >= 4) v = t + v;
  t = dpp_d<0x118>(v); if (rl >= 8) v = t + v;
  t = dpp_d<0x142>(v); if ((l & 31) >= 16) v = t + v;
  t = dpp_d<0x143>(v); if (l >= 32) v = t + v;
  return v;
}

// ---- classes ----------------------------------------------------------------
// A lane's walk from one class start: the value, and the interval of
// displacements that leave every partial sum so far in its binade.
struct Walk {
  double S, dlo, dhi;
  int emax;
  bool ok;
};

// Partial sums between mn and mx (one binade and sign): displacements keep
// them inside it with 4 ulps to spare; sums nearer to its ends than that, or
// outside the ordinary range, admit none.
__device__ __forceinline__ void keep_binade(double mn, double mx, Walk &w) {
  const int eb = binade(mn);
  w.emax = max(w.emax, eb);
  const double bl = pow2_field(eb), bh = pow2_field(eb + 1), m = pow2_field(max(eb - 50, 1));
  const double L = mn > 0.0 ? bl + m : -bh + m, U = mn > 0.0 ? bh - m : -bl - m;
  if (!binade_ok(eb) || mn < L || mx > U) {
    w.dlo = fmax(w.dlo, 0.0);
    w.dhi = fmin(w.dhi, 0.0);
    return;
  }
  w.dlo = fmax(w.dlo, L - mn);
  w.dhi = fmin(w.dhi, U - mx);
}

// A chunk's 64 values added in order (values beyond the array are zeros,
// which change nothing), eight at a time: the sums of a group that all share
// the binade so far only extend its extremes.
__device__ __forceinline__ void ordered_chunk(const double *v, Walk &w) {
  double S = w.S, mn = 0.0, mx = 0.0;
  int key = -1;
  for (int j0 = 0; j0 < kChunk; j0 += 8) {
    double x[8];
#pragma unroll
    for (int j = 0; j < 8; j++) x[j] = v[j0 + j];
    double y[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      S = S + x[j];
      y[j] = S;
    }
    const double lo = fmin(fmin(fmin(y[0], y[1]), fmin(y[2], y[3])),
                           fmin(fmin(y[4], y[5]), fmin(y[6], y[7])));
    const double hi = fmax(fmax(fmax(y[0], y[1]), fmax(y[2], y[3])),
                           fmax(fmax(y[4], y[5]), fmax(y[6], y[7])));
    if (segkey(lo) == key && segkey(hi) == key) {
      mn = fmin(mn, lo);
      mx = fmax(mx, hi);
    } else {
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int k = segkey(y[j]);
        if (k != key) {
          if (key >= 0) keep_binade(mn, mx, w);
          key = k;
          mn = mx = y[j];
        } else {
          mn = fmin(mn, y[j]);
          mx = fmax(mx, y[j]);
        }
      }
    }
  }
  keep_binade(mn, mx, w);
  w.S = S;
}

// Grid steps (mod 2) between two values of one binade: the mantissas' last
// bits.
__device__ __forceinline__ int parity_from(double S, double g) {
  return (__double2loint(S) ^ __double2loint(g)) & 1;
}

// A chunk's record: its guess g, the translations from g and g + u, and the
// open range of starts whose runs stay inside g's binade (with 4 ulps to
// spare; empty if the run from g itself leaves it).
struct ChunkRec {
  double g, d0, d1, lo, hi;
};

// The walk over a chunk: by its translation if its record covers S, else
// value by value.
__device__ __forceinline__ void walk_chunk(const ChunkRec &r, const double *v, Walk &w) {
  if (w.S > r.lo && w.S < r.hi) {
    w.dlo = fmax(w.dlo, r.lo - w.S);
    w.dhi = fmin(w.dhi, r.hi - w.S);
    w.emax = max(w.emax, binade(r.g));
    w.S = w.S + (parity_from(w.S, r.g) ? r.d1 : r.d0);
  } else {
    ordered_chunk(v, w);
  }
}

// The walk over a folded window.
__device__ __forceinline__ void walk_comp(const SeqComp &c, Walk &w) {
  const int p = parity_from(w.S, c.g);
  const double lo = p ? c.lo1 : c.lo0, hi = p ? c.hi1 : c.hi0;
  w.ok = w.ok && w.S >= lo && w.S <= hi;
  w.dlo = fmax(w.dlo, lo - w.S);
  w.dhi = fmin(w.dhi, hi - w.S);
  w.emax = max(w.emax, c.eb);
  w.S = w.S + (p ? c.d1 : c.d0);
}

// The class of start S in a table from g: grid steps away from zero, the
// difference of the mantissas.
__device__ __forceinline__ int class_of(double S, double g, int M) {
  const uint32_t dm = (uint32_t)__double2loint(S) - (uint32_t)__double2loint(g);
  return (int)(dm & (uint32_t)(max(M, 1) - 1));
}

// The walk over an entry that has a table (M classes at cls).
__device__ __forceinline__ void walk_classes(const SeqClass *cls, double g, int M, int emax,
                                             Walk &w) {
  w.ok = w.ok && M > 0 && segkey(w.S) == segkey(g);
  const SeqClass c = cls[class_of(w.S, g, M)];
  const double delta = w.S - c.s;  // exact: one binade
  w.ok = w.ok && delta >= c.lo && delta <= c.hi;
  w.dlo = fmax(w.dlo, c.lo - delta);
  w.dhi = fmin(w.dhi, c.hi - delta);
  w.emax = max(w.emax, emax);
  w.S = c.e + delta;
}
__device__ __forceinline__ void walk_tab(const SeqTab &t, Walk &w) {
  walk_classes(t.c, t.g, t.M, t.emax, w);
}

// The same from one start, every lane alike; false if the table does not
// cover it.
__device__ __forceinline__ bool take_tab(const SeqTab &t, double &S) {
  Walk w;
  w.S = S;
  w.ok = true;
  w.dlo = w.dhi = 0.0;
  w.emax = 0;
  walk_tab(t, w);
  if (!__ballot(w.ok)) return false;
  S = w.S;
  return true;
}

// Lane c's class start of a table that begins at g: c grid steps away from
// zero, so that every class has g's binade unless it is left at once.
__device__ __forceinline__ Walk class_start(double g) {
  const int l = lane_id(), eb = binade(g);
  Walk w;
  w.ok = binade_ok(eb);
  const double u = w.ok ? pow2_field(eb - 52) : 0.0;
  w.S = g + (double)(g < 0.0 ? -l : l) * u;  // exact: fewer than 2^6 ulps
  w.ok = w.ok && segkey(w.S) == segkey(g);
  w.dlo = -0x1p1000;
  w.dhi = 0x1p1000;
  w.emax = eb;
  return w;
}

// The walks' results as the table of an entry; s0: the lane's start.
__device__ __forceinline__ void put_tab(SeqTab &t, double g, double s0, const Walk &w) {
  const int l = lane_id(), e0 = binade(g);
  int em = w.ok ? w.emax : e0;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) em = max(em, __shfl_xor(em, o));
  const int lgm = 1 + em - e0;
  int M = lgm <= 6 ? 1 << lgm : 0;
  if (__ballot(l < M && !w.ok)) M = 0;
  if (l < M) t.c[l] = {s0, w.S, w.dlo, w.dhi};
  if (l == 0) {
    t.g = g;
    t.M = M;
    t.emax = em;
  }
}
__device__ __forceinline__ void put_exact(SeqTab &t, double S) {
  if (lane_id() == 0) {
    t.g = 0.0;
    t.M = -1;
    t.emax = 0;
    t.c[0].e = S;
  }
}

// ---- chunk totals -------------------------------------------------------------
// tot[c] and blk[sg]: the totals of each chunk and segment in any order,
// for the guesses (a wavefront takes a chunk at a time, coalesced).
__global__ void __launch_bounds__(256) seq_totals(const double *__restrict__ a, int64_t n,
                                                  double *__restrict__ tot,
                                                  double *__restrict__ blk) {
  __shared__ double part[4];
  const int l = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t c0 = (int64_t)blockIdx.x * 64 + wv * 16;
  double v[16], s = 0.0;
#pragma unroll
  for (int j = 0; j < 16; j++) {
    const int64_t gi = (c0 + j) * kChunk + l;
    v[j] = gi < n ? a[gi] : 0.0;
  }
#pragma unroll
  for (int j = 0; j < 16; j++) {
    const double t = wave_sum(v[j]);
    s += t;
    if (l == 0 && (c0 + j) * kChunk < n) tot[c0 + j] = t;
  }
  if (l == 0) part[wv] = s;
  __syncthreads();
  if (threadIdx.x == 0) blk[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

// blk[k] <- the total of the segments before k (one workgroup; for sums of
// so many segments that each segment's own loop over them would dominate)
__global__ void __launch_bounds__(1024) seq_prefix(double *blk, int64_t nb) {
  __shared__ double part[1024];
  const int t = threadIdx.x;
  const int64_t per = (nb + 1023) / 1024, b = min(nb, per * t), e = min(nb, per * (t + 1));
  double s = 0.0;
  for (int64_t k = b; k < e; k++) s += blk[k];
  part[t] = s;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {
    const double p = t >= o ? part[t - o] : 0.0;
    __syncthreads();
    part[t] += p;
    __syncthreads();
  }
  s = t > 0 ? part[t - 1] : 0.0;
  for (int64_t k = b; k < e; k++) {
    const double v = blk[k];
    blk[k] = s;
    s += v;
  }
}

// ---- segments -------------------------------------------------------------------
// ONE: the sum is this one segment; its exact value goes to dout.
// The total before the segment comes from the chunk totals, or with blk from
// the prefix of the segments' totals.
// Wave 0 makes the chunks' records and folds the windows; wave k the table of
// window k if that did not fold.
template <bool ONE>
__global__ void __launch_bounds__(64 * kWins) seq_segments(const double *__restrict__ a, int64_t n,
                                                   const double *__restrict__ tot,
                                                   const double *__restrict__ blk,
                                                   SeqComp *__restrict__ comps,
                                                   SeqTab *__restrict__ tabs, double *dout) {
  __shared__ double tile[64][kChunk + 1];
  __shared__ ChunkRec rec[64];
  __shared__ SeqComp comp[kWins];
  __shared__ SeqTab wtab[kWins];
  __shared__ double before[kWins];
  const int t = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t sg = blockIdx.x, c0 = sg * 64, c = c0 + t, nch = (n + kChunk - 1) / kChunk;
  {
    constexpr int PER = kSegVals / (64 * kWins);
    double v[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) {
      const int64_t gi = sg * kSegVals + (j * kWins + wv) * 64 + t;
      v[j] = gi < n ? a[gi] : 0.0;
    }
    if (!ONE) {
      double s = 0.0;
      if (blk) {
        if (threadIdx.x == 0) s = blk[sg];
      } else {
        // sixteen totals a thread in flight
        for (int64_t k = threadIdx.x; k < c0; k += 16 * 64 * kWins) {
          double q[16];
#pragma unroll
          for (int j = 0; j < 16; j++) {
            const int64_t kj = k + j * 64 * kWins;
            q[j] = kj < c0 ? tot[kj] : 0.0;
          }
#pragma unroll
          for (int j = 0; j < 16; j++) s += q[j];
        }
      }
      s = wave_sum(s);
      if (t == 0) before[wv] = s;
    }
#pragma unroll
    for (int j = 0; j < PER; j++) tile[j * kWins + wv][t] = v[j];
  }
  const int nwin = (int)min((int64_t)kWins, (nch - c0 + kWin - 1) / kWin);
  double tc = !ONE && wv == 0 && c < nch ? tot[c] : 0.0;
  __syncthreads();
  if (wv == 0) {
  double off = 0.0;  // the total before this segment
  if (ONE) {
    const double *row = tile[t];
#pragma unroll 16
    for (int j = 0; j < kChunk; j++) tc += row[j];
  } else {
#pragma unroll
    for (int k = 0; k < kWins; k++) off += before[k];
  }
  // guess of the chunk's start, and of the one after it
  const double gnext = off + wave_incl_add(tc);
  double g = __shfl_up(gnext, 1);
  if (t == 0) g = off;
  // the runs from g and g + u, branch-free: the rounded partial sums bound
  // the exact ones within half an ulp, and in one binade the second run
  // stays 0 to 2 u above the first
  const int eb = binade(g), key = segkey(g);
  const bool eb_ok = binade_ok(eb);
  const double u = eb_ok ? pow2_field(eb - 52) : 0.0, ui = eb_ok ? pow2_field(2098 - eb) : 0.0;
  double f0 = g, f1 = g + u, mn = g, mx = g;
  bool in = eb_ok && segkey(f1) == key;
  const double *row = tile[t];
#pragma unroll
  for (int j0 = 0; j0 < kChunk; j0 += 8) {
    double x[8];
#pragma unroll
    for (int j = 0; j < 8; j++) x[j] = row[j0 + j];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      f0 = f0 + x[j];
      f1 = f1 + x[j];
      mn = fmin(mn, f0);
      mx = fmax(mx, f0);
    }
  }
  mx = mx + 2.0 * u;
  // extremes in g's binade: then so is every partial sum
  in = in && segkey(mn) == key && segkey(mx) == key && segkey(f1) == key;
  const double d0 = f0 - g, d1 = f1 - (g + u), rlo0 = mn - g, rhi0 = mx - g;
  const bool rok = in && run_inside(g, eb, rlo0, rhi0);
  {
    const double bl = eb_ok ? pow2_field(eb) : 0.0, m4 = 4.0 * u, bh = 2.0 * bl;
    ChunkRec R;
    R.g = g;
    R.d0 = d0;
    R.d1 = d1;
    R.lo = !rok ? 1.0 : (g > 0.0 ? bl + m4 : m4 - bh) - rlo0;
    R.hi = !rok ? 0.0 : (g > 0.0 ? bh - m4 : -bl - m4) - rhi0;
    rec[t] = R;
  }
  // windows: the 16 lanes of DPP row w fold window w, lane i taking member
  // i: start parities by a row scan of the members' maps, translations by
  // row scans (exact sums), intervals by row max/min
  const int wl = t / kWin, rl = t & 15;
  const int64_t w0 = c0 + (int64_t)wl * kWin;
  const int nm = w0 < nch ? (int)min((int64_t)kWin, nch - w0) : 0;
  const bool mem = rl < nm;
  const int src0 = wl * kWin;
  const double gA = __shfl(g, src0);
  const int kA = __shfl(key, src0);
  const double sig = gA < 0.0 ? -1.0 : 1.0;
  bool fold = mem ? rok && key == kA : true;
  int mapm = 2;  // identity
  double d0m = 0.0, d1m = 0.0, Li = -0x1p60, Ui = 0x1p60;
  if (mem && fold) {
    const double rlo = sig > 0.0 ? rlo0 : -rhi0, rhi = sig > 0.0 ? rhi0 : -rlo0;
    Li = ceil(5.0 - rlo * ui) + 1.0;
    Ui = floor(0x1p52 - 5.0 - rhi * ui) - 1.0;
    // parity towards the next member (a run that leaves the binade there
    // does not fold)
    const int am = rl + 1 < nm ? parity_of((g + d0) - gnext, ui) : 0;
    const int bm = parity_of(d1 - d0, ui);
    mapm = ((bm ? 0 : 1) << 1) | am;  // p -> bm ? am : p ^ am
    d0m = d0;
    d1m = d1;
  }
  const int incl = row_incl_map(mapm);
  int ex = dpp_i<0x111>(incl);
  if (rl == 0) ex = 2;
  const int pa = ex & 1, pb = (ex >> 1) ? (1 ^ (ex & 1)) : (ex & 1);
  const double ia = row_incl_add(mem ? (pa ? d1m : d0m) : 0.0);
  const double ib = row_incl_add(mem ? (pb ? d1m : d0m) : 0.0);
  double xa = dpp_d<0x111>(ia), xb = dpp_d<0x111>(ib);
  if (rl == 0) xa = xb = 0.0;
  // admissible start offsets: member i's start is G1 + delta + sig D / u
  double lo0 = -0x1p60, hi0 = 0x1p60, lo1 = -0x1p60, hi1 = 0x1p60;
  if (mem && fold) {
    const double G1 = (fabs(gA) - pow2_field(eb)) * ui;
    const double Oa = sig * xa * ui, Ob = sig * xb * ui;
    lo0 = Li - G1 - Oa;
    hi0 = Ui - G1 - Oa;
    lo1 = Li - G1 - Ob;
    hi1 = Ui - G1 - Ob;
    // partial translations stay well inside 2^53 u, so every sum is exact
    if (fabs(ia) * ui > 0x1p51 || fabs(ib) * ui > 0x1p51) fold = false;
  }
#pragma unroll
  for (int m = 1; m < kWin; m <<= 1) {
    lo0 = fmax(lo0, __shfl_xor(lo0, m));
    hi0 = fmin(hi0, __shfl_xor(hi0, m));
    lo1 = fmax(lo1, __shfl_xor(lo1, m));
    hi1 = fmin(hi1, __shfl_xor(hi1, m));
  }
  const uint64_t foldm = __ballot(fold);
  const int last = src0 + (nm > 0 ? nm - 1 : 0);  // its lane holds the totals
  const double Da = __shfl(ia, last), Db = __shfl(ib, last);
  if (rl == 0) {
    SeqComp C;
    C.g = gA;
    C.d0 = Da;
    C.d1 = Db;
    // from grid steps towards larger magnitude to starts (the steps' margins
    // cover the roundings here)
    C.lo0 = gA + (sig > 0.0 ? lo0 : -hi0) * u;
    C.hi0 = gA + (sig > 0.0 ? hi0 : -lo0) * u;
    C.lo1 = gA + (sig > 0.0 ? lo1 : -hi1) * u;
    C.hi1 = gA + (sig > 0.0 ? hi1 : -lo1) * u;
    C.ok = nm > 0 && ((foldm >> src0) & 0xffff) == 0xffff;
    C.eb = eb;
    comp[wl] = C;
    if (!ONE) comps[sg * kWins + wl] = C;
  }
  }
  __syncthreads();
  if (ONE || sg == 0) {
    if (wv != 0) return;
    // the first segment starts at exactly +0: every lane walks it
    Walk w;
    w.S = 0.0;
    w.dlo = -0x1p1000;
    w.dhi = 0x1p1000;
    w.emax = 0;
    for (int k = 0; k < nwin; k++) {
      Walk z = w;
      z.ok = comp[k].ok;
      if (z.ok) walk_comp(comp[k], z);
      if (z.ok) {
        w = z;
        continue;
      }
      const int m = (int)min((int64_t)kWin, nch - c0 - k * kWin);
      for (int i = k * kWin; i < k * kWin + m; i++)
        walk_chunk(rec[i], tile[i], w);
    }
    if (ONE) {
      if (t == 0) *dout = w.S;
    } else {
      put_exact(tabs[0], w.S);
    }
    return;
  }
  if (wv < nwin && !comp[wv].ok) {
    const double gk = rec[wv * kWin].g;
    Walk w = class_start(gk);
    const double s0 = w.S;
    const int m = (int)min((int64_t)kWin, nch - c0 - wv * kWin);
    for (int i = wv * kWin; i < wv * kWin + m && __ballot(w.ok); i++)
      walk_chunk(rec[i], tile[i], w);
    put_tab(wtab[wv], gk, s0, w);
  }
  __syncthreads();
  if (wv != 0) return;
  // the segment's table
  const double gs = rec[0].g;
  Walk w = class_start(gs);
  const double s0 = w.S;
  for (int k = 0; k < nwin; k++) {
    if (comp[k].ok) walk_comp(comp[k], w);
    else walk_tab(wtab[k], w);
  }
  put_tab(tabs[sg], gs, s0, w);
}

// Sixteen entries of a level to one of the next: a wavefront per entry.
__global__ void __launch_bounds__(64) seq_fold(const SeqTab *__restrict__ in, int64_t nin,
                                               SeqTab *__restrict__ out) {
  __shared__ SeqTab t[kFold];
  const int l = threadIdx.x;
  const int64_t i0 = (int64_t)blockIdx.x * kFold;
  const int m = (int)min((int64_t)kFold, nin - i0);
  // every class of every entry in flight at once (those beyond an entry's M
  // are not used)
  SeqClass c[kFold];
#pragma unroll
  for (int k = 0; k < kFold; k++) c[k] = in[i0 + min(k, m - 1)].c[l];
  if (l < m) {
    t[l].g = in[i0 + l].g;
    t[l].M = in[i0 + l].M;
    t[l].emax = in[i0 + l].emax;
  }
#pragma unroll
  for (int k = 0; k < kFold; k++)
    if (k < m) t[k].c[l] = c[k];
  __syncthreads();
  const bool first = blockIdx.x == 0;  // starts at the sum's beginning
  Walk w = class_start(t[0].g);
  if (first) {
    // entry 0's exact end, unless it did not fold itself (its c[0] is then
    // whatever an earlier sum left there)
    w.S = t[0].c[0].e;
    w.ok = t[0].M < 0;
  }
  const double s0 = w.S;
  for (int k = first ? 1 : 0; k < m; k++) walk_tab(t[k], w);
  if (first && w.ok) put_exact(out[0], w.S);
  else if (first) {
    if (l == 0) out[0].M = 0;
  } else {
    put_tab(out[blockIdx.x], t[0].g, s0, w);
  }
}

// ---- the chain --------------------------------------------------------------------
struct SeqLevels {
  const SeqTab *tab[kMaxLevels];
  int64_t n[kMaxLevels];
  int top;  // the level that the chain takes
};

// Orders the calling wavefront's LDS accesses.
__device__ __forceinline__ void seq_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  __builtin_amdgcn_wave_barrier();
}

// Window k of segment sg from S: folded, or its values added in order
// (staged through LDS, a dependent add of 4.3 ns each).
__device__ double resolve_window(const double *__restrict__ a, int64_t n, int64_t win,
                                 const SeqComp *__restrict__ comps, double S, double *lds) {
  const int l = lane_id();
  const SeqComp C = comps[win];
  const int p = parity_from(S, C.g);
  if (__ballot(C.ok && S >= (p ? C.lo1 : C.lo0) && S <= (p ? C.hi1 : C.hi0)))
    return S + (p ? C.d1 : C.d0);
  const int64_t b = win * (int64_t)(kWin * kChunk);
  seq_wave_sync();
  for (int j = l; j < kWin * kChunk; j += 64) lds[j] = b + j < n ? a[b + j] : 0.0;
  seq_wave_sync();
  for (int j0 = 0; j0 < kWin * kChunk; j0 += 16) {
    double x[16];
#pragma unroll
    for (int j = 0; j < 16; j++) x[j] = lds[j0 + j];
#pragma unroll
    for (int j = 0; j < 16; j++) S = S + x[j];
  }
  return S;
}

// Entry i of level lev from S, by its table or by its parts.
__device__ double resolve(const double *__restrict__ a, int64_t n, const SeqLevels &L, int lev,
                          int64_t i, const SeqComp *__restrict__ comps, double S, double *lds) {
  // the entries still to take, a depth-first descent: at most kFold - 1
  // siblings a level
  int64_t at[kMaxLevels], end[kMaxLevels];
  at[lev] = i;
  end[lev] = i + 1;
  int k = lev;
  for (;;) {
    while (k <= lev && at[k] >= end[k]) k++;
    if (k > lev) return S;
    const int64_t j = at[k]++;
    const SeqTab &t = L.tab[k][j];
    const int M = t.M;
    if (M < 0) {
      S = t.c[0].e;
      continue;
    }
    if (M > 0 && take_tab(t, S)) continue;
    if (k > 0) {
      k--;
      at[k] = j * kFold;
      end[k] = min(L.n[k], (j + 1) * kFold);
      continue;
    }
    const int64_t nwin = (n + kWin * kChunk - 1) / (kWin * kChunk);
    for (int64_t wn = j * kWins; wn < min(nwin, (j + 1) * kWins); wn++)
      S = resolve_window(a, n, wn, comps, S, lds);
  }
}

// The top level's entries in order.  Each of the workgroup's wavefronts folds
// its kGroup or fewer consecutive entries into one table (their classes
// brought into LDS first if they fit its share); wavefront 0 takes the
// sixteen tables.  A start that a table does not cover descends to the
// group's entries.
static constexpr int kShare = 192;  // classes in LDS per wavefront
struct ChainLds {
  SeqTab group[kChainWaves];
  SeqClass cls[kChainWaves][kShare];
  double vals[kWin * kChunk];
};
__global__ void __launch_bounds__(64 * kChainWaves) seq_chain(const double *__restrict__ a,
                                                              int64_t n, SeqLevels L,
                                                              const SeqComp *__restrict__ comps,
                                                              double *dout) {
  extern __shared__ __align__(16) unsigned char chain_raw[];
  ChainLds &C = *(ChainLds *)chain_raw;
  const int l = threadIdx.x & 63, wv = threadIdx.x >> 6, m = (int)L.n[L.top];
  const SeqTab *tab = L.tab[L.top];
  const int per = (m + kChainWaves - 1) / kChainWaves, k0 = wv * per, ke = min(m, k0 + per);
  if (k0 < m) {
    // lane i: the head of entry k0 + i
    const bool have = l < ke - k0;
    const int Mi = have ? tab[k0 + l].M : 0, ei = have ? tab[k0 + l].emax : 0;
    const double gi = have ? tab[k0 + l].g : 0.0;
    const int cnt = abs(Mi);
    int incl = cnt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int u = __shfl_up(incl, o);
      if (l >= o) incl += u;
    }
    const int first = incl - cnt;
    const bool fits = __shfl(incl, 63) <= kShare;
    if (fits) {
      SeqClass c[kGroup];
#pragma unroll
      for (int j = 0; j < kGroup; j++)
        if (l < __builtin_amdgcn_readlane(cnt, j)) c[j] = tab[k0 + j].c[l];
#pragma unroll
      for (int j = 0; j < kGroup; j++)
        if (l < __builtin_amdgcn_readlane(cnt, j))
          C.cls[wv][__builtin_amdgcn_readlane(first, j) + l] = c[j];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    __builtin_amdgcn_wave_barrier();
    const double g0 = readlane_f64(gi, 0);
    Walk w = class_start(g0);
    if (k0 == 0) {  // the sum's beginning: one exact start
      w.S = tab[0].c[0].e;
      w.ok = __builtin_amdgcn_readlane(Mi, 0) < 0;
    }
    const double s0 = w.S;
    for (int j = k0 == 0 ? 1 : 0; j < ke - k0; j++) {
      const int M = __builtin_amdgcn_readlane(Mi, j), em = __builtin_amdgcn_readlane(ei, j);
      const double g = readlane_f64(gi, j);
      if (fits) walk_classes(C.cls[wv] + __builtin_amdgcn_readlane(first, j), g, M, em, w);
      else walk_classes(tab[k0 + j].c, g, M, em, w);
    }
    if (k0 > 0) put_tab(C.group[wv], g0, s0, w);
    else if (w.ok) put_exact(C.group[0], w.S);
    else if (l == 0) C.group[0].M = 0;
  }
  __syncthreads();
  if (wv != 0) return;
  double S = 0.0;  // the reference's accumulator starts at +0
  for (int q = 0; q * per < m; q++) {
    const int M = C.group[q].M;
    if (M < 0) {
      S = C.group[q].c[0].e;
      continue;
    }
    if (M > 0 && take_tab(C.group[q], S)) continue;
    for (int k = q * per; k < min(m, (q + 1) * per); k++)
      S = resolve(a, n, L, L.top, k, comps, S, C.vals);
  }
  if (l == 0) *dout = S;
}

__global__ void seq_zero(double *out) {
  if (threadIdx.x == 0) *out = 0.0;
}

struct SeqLayout {
  int64_t nch, nseg, tot, blk, comps, tabs[kMaxLevels], n[kMaxLevels], bytes;
  int top;
};

static SeqLayout seq_layout(int64_t n) {
  SeqLayout L;
  L.nch = (n + kChunk - 1) / kChunk;
  L.nseg = (n + kSegVals - 1) / kSegVals;
  auto al = [](int64_t x) { return (x + 255) / 256 * 256; };
  L.tot = 0;
  L.blk = al(L.tot + 8 * L.nch);
  L.comps = al(L.blk + 8 * L.nseg);
  int64_t at = al(L.comps + (int64_t)sizeof(SeqComp) * kWins * L.nseg);
  // 2^31 nodes' worth of values (the largest array any caller has) needs
  // five levels
  int64_t m = L.nseg;
  for (L.top = 0;; L.top++) {
    L.n[L.top] = m;
    L.tabs[L.top] = at;
    at = al(at + (int64_t)sizeof(SeqTab) * m);
    if (m <= kTop || L.top == kMaxLevels - 1) break;
    m = (m + kFold - 1) / kFold;
  }
  L.bytes = at;
  return L;
}

// The launches of one sum over a work area laid out by seq_layout(n).
// totals: the chunk totals, where the array's producer has made them.
static int seqsum_launch(const double *a, int64_t n, double *dout, char *w, const SeqLayout &L,
                         hipStream_t s, const double *totals = nullptr) {
  if (n == 0) {
    hipLaunchKernelGGL(seq_zero, dim3(1), dim3(64), 0, s, dout);
    HYD_HIP(hipGetLastError());
    return HYD_OK;
  }
  if (L.nseg == 1) {
    hipLaunchKernelGGL(seq_segments<true>, dim3(1), dim3(64 * kWins), 0, s, a, n, nullptr,
                       nullptr, nullptr, nullptr, dout);
    HYD_HIP(hipGetLastError());
    return HYD_OK;
  }
  if (L.n[L.top] > kTop) {
    set_error("seqsum: array too long");
    return HYD_EARG;
  }
  double *tot = (double *)(w + L.tot);
  double *blk = (double *)(w + L.blk);
  SeqComp *comps = (SeqComp *)(w + L.comps);
  SeqLevels lv;
  lv.top = L.top;
  for (int k = 0; k <= L.top; k++) {
    lv.tab[k] = (const SeqTab *)(w + L.tabs[k]);
    lv.n[k] = L.n[k];
  }
  // up to 512 segments (kSeqOwnTotals) each one adds the chunk totals before
  // it (at most 128 loads a thread); beyond, a launch of the prefix is shorter
  const bool prefixed = n > kSeqOwnTotals;
  if (!totals || prefixed)
    hipLaunchKernelGGL(seq_totals, dim3((unsigned)L.nseg), dim3(256), 0, s, a, n, tot, blk);
  if (prefixed) hipLaunchKernelGGL(seq_prefix, dim3(1), dim3(1024), 0, s, blk, L.nseg);
  hipLaunchKernelGGL(seq_segments<false>, dim3((unsigned)L.nseg), dim3(64 * kWins), 0, s, a, n,
                     totals && !prefixed ? totals : tot, prefixed ? blk : nullptr, comps,
                     (SeqTab *)(w + L.tabs[0]), nullptr);
  for (int k = 1; k <= L.top; k++)
    hipLaunchKernelGGL(seq_fold, dim3((unsigned)L.n[k]), dim3(64), 0, s, lv.tab[k - 1], L.n[k - 1],
                       (SeqTab *)(w + L.tabs[k]));
  constexpr size_t shm = sizeof(ChainLds);
  static_assert(shm <= 160 * 1024, "the chain's LDS");
  static std::atomic<bool> raised{false};  // more than 64 KiB of LDS must be requested
  if (!raised.load(std::memory_order_acquire)) {
    HYD_HIP(hipFuncSetAttribute((const void *)seq_chain,
                                hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    raised.store(true, std::memory_order_release);
  }
  hipLaunchKernelGGL(seq_chain, dim3(1), dim3(64 * kChainWaves), shm, s, a, n, lv, comps, dout);
  HYD_HIP(hipGetLastError());
  return HYD_OK;
}

int seqsum(Ctx &c, const double *a, int64_t n, double *dout, const double *totals) {
  const SeqLayout L = seq_layout(n);
  if (L.nch > c.seq_cap || seq_layout((int64_t)c.seq_cap * kChunk).bytes < L.bytes) {
    set_error("seqsum: array longer than the context's work space");
    return HYD_ECAPACITY;
  }
  KTimer t(c, "seqsum", 8 * n);
  return seqsum_launch(a, n, dout, (char *)c.seq_work, L, c.s, totals);
}

// ---- the sequential sum without allocation ---------------------------------
// Work area in a file-scope device array: each GPU the library runs on holds
// its own copy (3.1 MiB used of 4 MiB for the largest sum, 2^22 values)
// until the process ends.  Host code never passes `scratch` itself to a
// kernel (in host code the name is a host-side stand-in): each device's
// address comes from hipGetSymbolAddress, taken once per device, with that
// device current, on the first call there.
static constexpr int64_t kNoAllocMaxN = (int64_t)1 << 22;
static constexpr int64_t kNoAllocBytes = (int64_t)4 << 20;
static __device__ __align__(256) char scratch[kNoAllocBytes];

static constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[kMaxDevices];

static int scratch_address(void **out) {
  int dev = 0;
  HYD_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) {
    set_error("sum_sequential_noalloc: device ordinal beyond the library's table");
    return HYD_EARG;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    HYD_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) {
      set_error("sum_sequential_noalloc: no device address for the work area");
      return HYD_EHIP;
    }
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return HYD_OK;
}

int64_t seqsum_work_chunks(int64_t n) { return (n + kChunk - 1) / kChunk; }

int64_t seqsum_work_bytes(int64_t n) { return seq_layout(n).bytes; }

}  // namespace hyd

extern "C" int hyd_sum_sequential_noalloc(const double *a, int64_t n, double *sum, void *stream) {
  using namespace hyd;
  if (n < 0 || n > kNoAllocMaxN) {
    set_error("sum_sequential_noalloc: length outside [0, 2^22]");
    return n < 0 ? HYD_EARG : HYD_ECAPACITY;
  }
  if (!sum || (n > 0 && !a)) {
    set_error("sum_sequential_noalloc: null device pointer");
    return HYD_EARG;
  }
  const SeqLayout L = seq_layout(n);
  if (L.bytes > kNoAllocBytes) {
    set_error("sum_sequential_noalloc: work area larger than the static scratch");
    return HYD_ECAPACITY;
  }
  void *w = nullptr;
  HYD_CHECK(scratch_address(&w));
  return seqsum_launch(a, n, sum, (char *)w, L, (hipStream_t)stream);
}
