// renode.hip -- node redistribution, contours.f90:687-933, for a batch of
// closed contours, one workgroup per contour.
//
// The per-node geometry (increments, cubic coefficients, corner test,
// curvature-based density) is evaluated lane-parallel in the reference's
// expression order.  The two sequential pieces -- the sum of the fractional
// node counts (contours.f90:799-802, whose nint decides how many nodes the
// contour keeps) and the accumulator walk that places the new nodes
// (813-930) -- run as wavefront-uniform chains: consecutive values are
// staged in LDS and every lane reads each one by broadcast, so the serial
// chain is the floating-point additions alone.  The walk is written per old
// node: acc + e(i) is the only rounded operation (acc - 1 is exact for acc
// >= 1), so acc = s - floor(s) after s = acc + e(i) is the reference's
// value after its floor(s) subtractions, and the nodes placed from old node
// i carry acc values s - 1, s - 2, ...; each lane recovers the s of its old
// node from LDS and emits its nodes in parallel.  Positions are then
// evaluated lane-parallel.
//
// Two launches: RN_COUNT computes the geometry, the sum and npr per contour
// (0 = delete) and keeps them; after an exclusive scan of npr, RN_PLACE
// scales, walks and writes the nodes.
#include "hyd_internal.h"

namespace hyd {

struct RenodeArgs {
  // input contours: nodes xd/yd, contour c has npd[c] nodes from off_in[c]
  const double *xd, *yd;
  const int64_t *off_in;
  const int32_t *npd;
  int32_t ncont;
  // scratch, indexed like the input nodes
  double *sdx, *sdy, *sa, *sb, *sc, *sd, *se, *su, *sv, *stm;
  int32_t *wi;     // walk: old node index per new node (indexed like output)
  double *wacc;    // walk: accumulator per new node
  // count pass results per contour, read by the place pass
  double *csum;
  int32_t *cnc, *cfirst;
  // output
  int32_t *npr;    // per contour
  const int64_t *off_out;
  double *xr, *yr;
  // constants
  double ellx, elly, hlxi, hlyi, oms, small, small3, dmsq, elf, dmi, densf;
};

#define F12 0.5
#define F13 (1.0 / 3.0)
#define F16 (1.0 / 6.0)

__device__ __forceinline__ double wrapc(double v, double L, double hli) {
  return v - L * (double)(int)(v * hli);
}

// Shared geometry of contours.f90:717-796 for contour c (all lanes).
__device__ void renode_geometry(const RenodeArgs &g, int64_t o, int n) {
  const int l = threadIdx.x, nt = blockDim.x;
  // increments, v, e
  for (int i = l; i < n; i += nt) {
    const int ia = i + 1 < n ? i + 1 : 0;
    const double xx = g.xd[o + ia] - g.xd[o + i];
    const double dx = wrapc(xx, g.ellx, g.hlxi);
    const double yy = g.yd[o + ia] - g.yd[o + i];
    const double dy = wrapc(yy, g.elly, g.hlyi);
    g.sdx[o + i] = dx;
    g.sdy[o + i] = dy;
    const double v = dx * dx + dy * dy;
    g.sv[o + i] = v;
    g.se[o + i] = sqrt(v);
  }
  __syncthreads();
  // u(i)=v(ib), a(i)=-dx(ib), c(i)=-dy(ib); corner test; b(i)
  for (int i = l; i < n; i += nt) {
    const int ib = i > 0 ? i - 1 : n - 1;
    const double u = g.sv[o + ib], a = -g.sdx[o + ib], c = -g.sdy[o + ib];
    const double dx = g.sdx[o + i], dy = g.sdy[o + i], v = g.sv[o + i];
    const bool corner = dx * a + dy * c > 0.0;
    double b;
    if (corner) {
      b = 0.0;
    } else {
      const double t1 = a * v - dx * u;
      const double t2 = c * v - dy * u;
      b = (dx * c - a * dy) / sqrt(t1 * t1 + t2 * t2 + g.small3);
    }
    g.sb[o + i] = b;
    g.sd[o + i] = corner ? 1.0 : 0.0;  // corner flag (d is reused below)
  }
  __syncthreads();
  // u=e*(b(ia)+b), c=e*(b(ia)-b); a,b,c cubic coefficients; curvature terms
  for (int i = l; i < n; i += nt) {
    const int ia = i + 1 < n ? i + 1 : 0;
    const double e = g.se[o + i], bi = g.sb[o + i], ba = g.sb[o + ia];
    double u = e * (ba + bi);
    double c = e * (ba - bi);
    g.sa[o + i] = F16 * c - F12 * u;
    const double bnew = F12 * (u - c);
    c = F13 * c;
    g.sc[o + i] = c;
    const double v = g.sv[o + i];
    const double ww = 1.0 / (v + g.dmsq);
    u = ww * sqrt(g.elf * v + u * u);
    g.su[o + i] = u;
    g.sv[o + i] = ww * e;
    // b is needed by the neighbour (ba) above: write it to a separate slot
    g.stm[o + i] = bnew;
  }
  __syncthreads();
  for (int i = l; i < n; i += nt) g.sb[o + i] = g.stm[o + i];
  __syncthreads();
  // d(i) = (u(ib)+u(i))/(v(ib)+v(i)+small), kept in stm
  for (int i = l; i < n; i += nt) {
    const int ib = i > 0 ? i - 1 : n - 1;
    g.stm[o + i] = (g.su[o + ib] + g.su[o + i]) / (g.sv[o + ib] + g.sv[o + i] + g.small);
  }
  __syncthreads();
  // u(i) = f12*(d(i)+d(ia)); e(i) = e(i)*min(dmi, densf*sqrt(u)+u)
  for (int i = l; i < n; i += nt) {
    const int ia = i + 1 < n ? i + 1 : 0;
    const double u = F12 * (g.stm[o + i] + g.stm[o + ia]);
    const double t = g.densf * sqrt(u) + u;
    g.se[o + i] = g.se[o + i] * (g.dmi < t ? g.dmi : t);
  }
  __syncthreads();
}

__device__ __forceinline__ double rl_d(double x, int l) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(x), l);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(x), l);
  return __hiloint2double(hi, lo);
}

// Orders the calling wavefront's LDS accesses (LDS serves one wavefront's
// accesses in issue order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// e of the q-th node of a walk that starts at node ibeg and wraps (q < n).
__device__ __forceinline__ double e_at(const double *se, int64_t o, int n, int ibeg, int q) {
  int i = ibeg + q;
  if (i >= n) i -= n;
  return se[o + i];
}

// The chains of long stretches take kRnBlock nodes at a time through LDS, the
// next ones in flight meanwhile.
static constexpr int kRnPer = 4, kRnBlock = 64 * kRnPer;
__device__ __forceinline__ void load_block(double (&v)[kRnPer], const double *se, int64_t o, int n,
                                           int ibeg, int q0, int len) {
  const int l = threadIdx.x & 63;
#pragma unroll
  for (int j = 0; j < kRnPer; j++) {
    const int q = q0 + 64 * j + l;
    v[j] = q < len ? e_at(se, o, n, ibeg, q % n) : 0.0;
  }
}

// Sequential sum of e over len nodes from ibeg (wrapping: next() order),
// contours.f90:799-802 and 880-884.  Wavefront-uniform (every lane returns
// the same value); lds holds kRnBlock doubles of the calling wavefront.
// Bound by the serial additions, 4.3 ns each from LDS.
__device__ double seq_sum_e(const double *se, int64_t o, int n, int ibeg, int len,
                            double *lds) {
  const int l = threadIdx.x & 63;
  double s = 0.0, v[kRnPer];
  load_block(v, se, o, n, ibeg, 0, len);
  for (int q0 = 0; q0 < len; q0 += kRnBlock) {
#pragma unroll
    for (int j = 0; j < kRnPer; j++) lds[64 * j + l] = v[j];
    if (q0 + kRnBlock < len) load_block(v, se, o, n, ibeg, q0 + kRnBlock, len);
    wave_sync();
    const int m = len - q0 < kRnBlock ? len - q0 : kRnBlock;
    int j = 0;
    for (; j + 64 <= m; j += 64) {
#pragma unroll
      for (int k = 0; k < 64; k++) s = s + lds[j + k];
    }
    for (; j < m; j++) s = s + lds[j];
    wave_sync();
  }
  return s;
}

// The accumulator walk (contours.f90:826-838, 858-868, 907-920) over the
// nodes ibeg, next(ibeg), ... for `want` new nodes, written to out slots
// oo+1 .. oo+want (old node index, acc after the subtraction).  acc starts
// at 0.  The scaled e of the len nodes sum to want + 1, so the walk ends
// among them: the roundings of its additions (len (want + 1) 2^-53 at most)
// do not make up for that one.  Wavefront-uniform; lds_e and lds_s hold
// kRnBlock doubles of the calling wavefront.
__device__ void walk_nodes(const RenodeArgs &g, int64_t o, int n, int ibeg, int len, int want,
                           int64_t oo, double *lds_e, double *lds_s) {
  const int l = threadIdx.x & 63;
  double acc = 0.0, v[kRnPer];
  int done = 0;
  load_block(v, g.se, o, n, ibeg, 0, len);
  int m;
  for (int q0 = 0; q0 < len && done < want; q0 += m) {
#pragma unroll
    for (int j = 0; j < kRnPer; j++) lds_e[64 * j + l] = v[j];
    m = len - q0 < kRnBlock ? len - q0 : kRnBlock;
    if (q0 + m < len) load_block(v, g.se, o, n, ibeg, q0 + m, len);
    wave_sync();
    // s - floor(s) is exact and s >= 0: the hardware's fraction
    int j = 0;
    for (; j + 16 <= m; j += 16) {
#pragma unroll
      for (int k = 0; k < 16; k++) {
        const double sj = acc + lds_e[j + k];
        lds_s[j + k] = sj;
        acc = __builtin_amdgcn_fract(sj);
      }
    }
    for (; j < m; j++) {
      const double sj = acc + lds_e[j];
      lds_s[j] = sj;
      acc = __builtin_amdgcn_fract(sj);
    }
    wave_sync();
    // old node q0+q places floor(s) new nodes, capped at the total wanted;
    // a lane takes kRnPer consecutive ones
    double sl[kRnPer];
    int k[kRnPer], mine = 0;
#pragma unroll
    for (int i = 0; i < kRnPer; i++) {
      const int q = kRnPer * l + i;
      sl[i] = q < m ? lds_s[q] : 0.0;
      k[i] = q < m ? (int)floor(sl[i]) : 0;
      mine += k[i];
    }
    int incl = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int t = __shfl_up(incl, d, 64);
      if (l >= d) incl += t;
    }
    int slot = done + incl - mine;  // 1-based new node after the first
    int i0 = ibeg + (q0 + kRnPer * l) % n;
    if (i0 >= n) i0 -= n;
#pragma unroll
    for (int i = 0; i < kRnPer; i++) {
      for (int r = 1; r <= k[i]; r++) {
        if (++slot > want) break;
        g.wi[oo + slot] = i0;
        g.wacc[oo + slot] = sl[i] - (double)r;
      }
      if (++i0 == n) i0 = 0;
    }
    done += __shfl(incl, 63, 64);
    wave_sync();
  }
  // (should slots ever be left, they get the last node, never an index
  // outside the contour)
  for (int slot = done + 1 + l; slot <= want; slot += 64) {
    int i = ibeg + len - 1;
    if (i >= n) i -= n;
    g.wi[oo + slot] = i;
    g.wacc[oo + slot] = 0.0;
  }
}

__device__ __forceinline__ int nint_d(double x) { return (int)llround(x); }

// Place one new node from old node i (0-based) and accumulator acc
// (contours.f90:833-838).
__device__ __forceinline__ void place(const RenodeArgs &g, int64_t o, int i, double acc,
                                      double &xo, double &yo) {
  const double e = g.se[o + i];
  const double p = 1.0 - acc / e;
  const double eta = p * (g.sa[o + i] + p * (g.sb[o + i] + p * g.sc[o + i]));
  const double xx = g.xd[o + i] + p * g.sdx[o + i] - eta * g.sdy[o + i];
  xo = g.oms * wrapc(xx, g.ellx, g.hlxi);
  const double yy = g.yd[o + i] + p * g.sdy[o + i] + eta * g.sdx[o + i];
  yo = g.oms * wrapc(yy, g.elly, g.hlyi);
}

// Exclusive prefix of v over the workgroup's 256 threads, and the total;
// lds holds 4 integers.
__device__ __forceinline__ int block_excl(int v, int *lds, int &total) {
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  int incl = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int t = __shfl_up(incl, d, 64);
    if (l >= d) incl += t;
  }
  __syncthreads();  // the previous call's reads
  if (l == 63) lds[w] = incl;
  __syncthreads();
  const int t0 = lds[0], t1 = lds[1], t2 = lds[2], t3 = lds[3];
  total = t0 + t1 + t2 + t3;
  return incl - v + (w > 0 ? t0 : 0) + (w > 1 ? t1 : 0) + (w > 2 ? t2 : 0);
}

// The stretches between corners (contours.f90:873-929) of a contour, kept
// from the count pass to the place pass in the scratch of u and v, which the
// geometry no longer needs (a contour has at most as many corners as nodes):
// stretch k starts at node beg(k), has len(k) nodes, its e sum to sum(k) and
// it gets np(k) nodes.
struct Stretches {
  int2 *u;      // .x the corner, .y the node count
  double *sum;
  int n, ncorn;
  __device__ Stretches(const RenodeArgs &g, int64_t o, int n_, int nc)
      : u((int2 *)(g.su + o)), sum(g.sv + o), n(n_), ncorn(nc) {}
  __device__ int beg(int k) const { return u[k].x; }
  __device__ int len(int k) const {
    const int e = u[k + 1 < ncorn ? k + 1 : 0].x, b = u[k].x;
    return e > b ? e - b : e + n - b;
  }
};
// A stretch of up to kShort nodes is one lane's, longer ones are a wavefront's.
// A recontoured field's contours have a corner every few nodes, thousands
// of them on the longest contours: recontouring a developed ng=64 flow took
// 5.9 + 3.1 ms in the two launches with one wavefront taking a contour's
// stretches in turn, and takes 0.8 + 1.7 ms; what remains is the longest
// contour's total, one chain of additions.
static constexpr int kShort = 64;

// One workgroup of 256 threads per contour: the lane-parallel phases use
// all of them, the sequential sums and walks run on a lane or a wavefront.
// RN_COUNT (PLACE = false): geometry, corners, sums, npr; RN_PLACE: the
// scaling, the walk and the node positions from the count pass's geometry.
template <bool PLACE>
__global__ void __launch_bounds__(256) renode_kernel(RenodeArgs g) {
  const int c = blockIdx.x;
  if (c >= g.ncont) return;
  const int n = g.npd[c];
  const int64_t o = g.off_in[c];
  const int t = threadIdx.x, l = t & 63, w = t >> 6, nt = blockDim.x;
  __shared__ double lds_e[4][kRnBlock], lds_s[PLACE ? 4 : 1][PLACE ? kRnBlock : 1];
  __shared__ int s_scan[4];
  __shared__ double s_sum;
  if (n <= 0) {
    if (!PLACE && t == 0) g.npr[c] = 0;
    return;
  }
  int ncorn = 0;
  if (!PLACE) {
    renode_geometry(g, o, n);
    // corners (d holds the flag), in order
    int2 *const corner = (int2 *)(g.su + o);
    for (int b0 = 0; b0 < n; b0 += 8 * nt) {
      int f[8], mine = 0, tot;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int i = b0 + 8 * t + j;
        f[j] = i < n && g.sd[o + i] != 0.0;
        mine += f[j];
      }
      int at = ncorn + block_excl(mine, s_scan, tot);
#pragma unroll
      for (int j = 0; j < 8; j++)
        if (f[j]) corner[at++].x = b0 + 8 * t + j;
      ncorn += tot;
    }
    // the total of e (contours.f90:799-809)
    if (w == 0) {
      const double sum = seq_sum_e(g.se, o, n, 0, n, lds_e[0]);
      if (l == 0) s_sum = sum;
    }
    __syncthreads();
    if (t == 0) {
      g.csum[c] = s_sum;
      g.cnc[c] = ncorn;
      g.cfirst[c] = ncorn ? corner[0].x : -1;
    }
  } else {
    ncorn = g.cnc[c];
  }
  const double sum = PLACE ? g.csum[c] : s_sum;
  const int npr = nint_d(sum) + 1;
  if (npr < 3) {
    if (!PLACE && t == 0) g.npr[c] = 0;
    return;
  }
  if (ncorn <= 1) {
    if (!PLACE) {
      if (t == 0) g.npr[c] = npr;
      return;
    }
    const double fac = (double)npr / sum;
    for (int i = t; i < n; i += nt) g.se[o + i] = fac * g.se[o + i];
    __syncthreads();
    const int64_t oo = g.off_out[c];
    const int start = ncorn == 0 ? 0 : g.cfirst[c];
    if (w == 0) {
      if (l == 0) {
        g.xr[oo] = g.xd[o + start];
        g.yr[oo] = g.yd[o + start];
      }
      // ncorn = 0 walks i = 1, 2, ...; ncorn = 1 starts at the corner and
      // wraps (contours.f90:826-868)
      walk_nodes(g, o, n, start, n, npr - 1, oo, lds_e[0], lds_s[0]);
    }
    __syncthreads();
    for (int im = 1 + t; im < npr; im += nt) {
      double xo, yo;
      place(g, o, g.wi[oo + im], g.wacc[oo + im], xo, yo);
      g.xr[oo + im] = xo;
      g.yr[oo + im] = yo;
    }
    return;
  }
  // several corners: renode each stretch between consecutive corners
  // (contours.f90:873-929)
  const Stretches st(g, o, n, ncorn);
  if (!PLACE) {
    // sums over the stretches (next() wraps)
    int mine = 0;
    auto keep = [&](int k, double sm) {
      const int np = sm > g.small ? nint_d(sm) + 1 : 0;
      st.sum[k] = sm;
      st.u[k].y = np;
      mine += np;
    };
    for (int k = t; k < ncorn; k += nt) {
      const int len = st.len(k);
      if (len > kShort) continue;
      const int ib = st.beg(k);
      double sm = 0.0;
      for (int q = 0; q < len; q += 8) {
        double e[8];
#pragma unroll
        for (int j = 0; j < 8; j++) e[j] = e_at(g.se, o, n, ib, q + j < len ? q + j : q);
#pragma unroll
        for (int j = 0; j < 8; j++)
          if (q + j < len) sm = sm + e[j];
      }
      keep(k, sm);
    }
    for (int k = w; k < ncorn; k += 4) {
      const int len = st.len(k);
      if (len <= kShort) continue;
      const double sm = seq_sum_e(g.se, o, n, st.beg(k), len, lds_e[w]);
      if (l == 0) keep(k, sm);
    }
    int tot;
    block_excl(mine, s_scan, tot);
    if (t == 0) g.npr[c] = tot;
    return;
  }
  const int64_t oo = g.off_out[c];
  // each stretch's first slot, in place of its node count
  int tot = 0;
  for (int k0 = 0; k0 < ncorn; k0 += nt) {
    const int k = k0 + t, np = k < ncorn ? st.u[k].y : 0;
    int add;
    const int at = tot + block_excl(np, s_scan, add);
    if (k < ncorn) st.u[k].y = np ? at : -1;
    tot += add;
  }
  __syncthreads();
  for (int k = t; k < ncorn; k += nt) {
    const int at = st.u[k].y, ib = st.beg(k), len = st.len(k);
    if (at < 0) continue;
    g.xr[oo + at] = g.xd[o + ib];
    g.yr[oo + at] = g.yd[o + ib];
    g.wi[oo + at] = -1;
    if (len > kShort) continue;
    const double sm = st.sum[k];
    const int np = nint_d(sm) + 1;
    const double fac = (double)np / sm;
    double acc = 0.0;
    int slot = at;  // the last one written
    for (int q = 0; q < len; q += 8) {
      double e[8];
#pragma unroll
      for (int j = 0; j < 8; j++) e[j] = e_at(g.se, o, n, ib, q + j < len ? q + j : q);
#pragma unroll
      for (int j = 0; j < 8; j++)
        if (q + j < len) {
          int i = ib + q + j;
          if (i >= n) i -= n;
          const double ei = fac * e[j], sj = acc + ei;
          g.se[o + i] = ei;
          acc = __builtin_amdgcn_fract(sj);
          const int kn = (int)floor(sj);
          for (int r = 1; r <= kn && slot + 1 < at + np; r++) {
            slot++;
            g.wi[oo + slot] = i;
            g.wacc[oo + slot] = sj - (double)r;
          }
        }
    }
    // (never reached, as in walk_nodes)
    for (slot++; slot < at + np; slot++) {
      g.wi[oo + slot] = ib;
      g.wacc[oo + slot] = 0.0;
    }
  }
  for (int k = w; k < ncorn; k += 4) {
    const int at = st.u[k].y, ib = st.beg(k), len = st.len(k);
    if (at < 0 || len <= kShort) continue;
    const double sm = st.sum[k];
    const int np = nint_d(sm) + 1;
    const double fac = (double)np / sm;
    for (int q0 = l; q0 < len; q0 += 64) {
      const int q = ib + q0 < n ? ib + q0 : ib + q0 - n;
      g.se[o + q] = fac * g.se[o + q];
    }
    __threadfence_block();  // the walk reads the scaled values (other lanes' stores)
    if (np > 1) walk_nodes(g, o, n, ib, len, np - 1, oo + at, lds_e[w], lds_s[w]);
  }
  __syncthreads();
  for (int im = t; im < tot; im += nt) {
    const int i = g.wi[oo + im];
    if (i < 0) continue;  // corner copied above
    double xo, yo;
    place(g, o, i, g.wacc[oo + im], xo, yo);
    g.xr[oo + im] = xo;
    g.yr[oo + im] = yo;
  }
}

}  // namespace hyd

namespace hyd {

// Renode a batch of contours: count, exclusive scan, place.  Returns
// HYD_ECAPACITY (with *ntot_out set) when the output would exceed cap_out.
int renode_batch(Ctx &c, const double *xd, const double *yd, const int64_t *off_in,
                 const int32_t *npd, int ncont, int64_t nin, double *xr, double *yr,
                 int64_t *off_out, int32_t *npr, int64_t *ntot_out, int64_t cap_out) {
  *ntot_out = 0;
  if (ncont <= 0) return HYD_OK;
  KTimer tm(c, "renode", 16 * nin * 3);
  RenodeArgs g;
  const Consts &k = c.c;
  g.xd = xd;
  g.yd = yd;
  g.off_in = off_in;
  g.npd = npd;
  g.ncont = ncont;
  const int64_t ns = std::max<int64_t>(nin, 1);
  double **scr[] = {&g.sdx, &g.sdy, &g.sa, &g.sb, &g.sc, &g.sd, &g.se, &g.su, &g.sv, &g.stm};
  static const char *names[] = {"rn_dx", "rn_dy", "rn_a", "rn_b", "rn_c",
                                "rn_d",  "rn_e",  "rn_u", "rn_v", "rn_t"};
  for (int t = 0; t < 10; t++) HYD_CHECK(dbuf(c, names[t], ns, scr[t]));
  g.npr = npr;
  g.off_out = off_out;
  g.xr = xr;
  g.yr = yr;
  g.ellx = k.ellx;
  g.elly = k.elly;
  g.hlxi = k.hlxi;
  g.hlyi = k.hlyi;
  g.oms = k.oms;
  g.small = k.small;
  g.small3 = k.small3;
  g.dmsq = k.dmsq;
  g.elf = k.elf;
  g.dmi = k.dmi;
  g.densf = k.densf;
  g.wi = nullptr;
  g.wacc = nullptr;
  HYD_CHECK(dbuf(c, "rn_csum", ncont, &g.csum));
  HYD_CHECK(dbuf(c, "rn_cnc", ncont, &g.cnc));
  HYD_CHECK(dbuf(c, "rn_cfirst", ncont, &g.cfirst));
  hipLaunchKernelGGL(renode_kernel<false>, dim3(ncont), dim3(256), 0, c.s, g);
  HYD_HIP(hipGetLastError());
  std::vector<int32_t> hn(ncont);
  HYD_HIP(hipMemcpyAsync(hn.data(), npr, 4 * ncont, hipMemcpyDeviceToHost, c.s));
  HYD_HIP(hipStreamSynchronize(c.s));
  std::vector<int64_t> ho(ncont);
  int64_t tot = 0;
  for (int j = 0; j < ncont; j++) {
    ho[j] = tot;
    tot += hn[j];
  }
  *ntot_out = tot;
  if (tot > cap_out) {
    set_error("renode: output exceeds buffer");
    return HYD_ECAPACITY;
  }
  HYD_HIP(hipMemcpyAsync(off_out, ho.data(), 8 * ncont, hipMemcpyHostToDevice, c.s));
  HYD_CHECK(dbuf(c, "rn_wi", std::max<int64_t>(tot, 1), &g.wi));
  HYD_CHECK(dbuf(c, "rn_wacc", std::max<int64_t>(tot, 1), &g.wacc));
  hipLaunchKernelGGL(renode_kernel<true>, dim3(ncont), dim3(256), 0, c.s, g);
  HYD_HIP(hipGetLastError());
  return HYD_OK;
}

}  // namespace hyd
