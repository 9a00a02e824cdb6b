// fft_kernel.h -- the stafft-faithful real FFT kernel (see fft.hip for the
// transforms built from it).
//
// A block transforms V vectors of length N.  stafft's factors (a 2 first if
// log2 N is odd, then 4s; in reverse order backward) are taken one or two at
// a time: the butterflies of two consecutive stages that share their values
// form a unit of up to 32 values, held in one thread's registers.  The units
// close because a stage pairs the rows k and lv - k, and the rows that such
// a pair writes (k + lv j and lv - k + lv j) are the pairs of the next
// stage.  So N = 1024 takes three passes over the values and two exchanges
// through LDS instead of five; the first pass reads global memory straight
// into registers and the last one writes from them.  Every butterfly is
// stafft's own, in its expression order without contraction, hence the
// results are stafft's bit for bit whatever the blocking.
//
// What bounds it: memory at large grids (a pass of four 1024^2 FP64 fields
// moves 67 MB in 18-20 us, 3.5 TB/s, and in 21 beside the other stream's
// kernels; a stage at a time through LDS it took 23-25), latency at small ones.  All of a thread's (up to 32) global loads
// are issued before the first use.  FP32 gains most: its passes at 2048^2
// were bound by the LDS exchanges.
#pragma once
#include <hip/hip_ext.h>

#include <atomic>
#include <type_traits>

#include "hyd_internal.h"

namespace hyd {

// Up to kMaxF fields of the same shape and direction per launch
// (blockIdx.y selects the field); each field has its own input, output,
// fused derivative and scaling.
static constexpr int kMaxF = 4;
static constexpr int kMaxV = 16;  // vectors per block: a power of two

struct FftArgs {
  const void *in[kMaxF];    // TI
  void *out[kMaxF];         // TO
  const double *dk[kMaxF];  // filtered wavenumbers for a fused derivative
  int pre[kMaxF];           // 0 none, 1 derivative across vectors, 2 along elements
  double post[kMaxF];       // normalisation (and sign) folded into the store
  const void *trig;         // T, 2n: cos then -sin (stafft.f90:103-122)
  const double *sub;        // forward: subtract *sub / subdiv from every input value
  double subdiv;
  int m;                    // vectors
};

// ---- butterflies ------------------------------------------------------------
// One radix-4 butterfly of a stage, forward (forrdx4, stafft.f90:890-997) and
// backward (revrdx4, 1463-1571): of the rows k and lv-k, of row 0, and of the
// middle row lv/2.

template <class T>
struct Tw {  // the three twiddles of row k
  T c1, s1, c2, s2, c3, s3;
};
// stage lv of the table: cos/-sin of its three multiples, lv entries each,
// from entry N - 4 lv on
template <int N, class T>
__device__ __forceinline__ Tw<T> twiddle(const T *__restrict__ trig, int lv, int k) {
  const T *cs = trig + (N - 4 * lv) + k, *sn = cs + N;
  return {cs[0], sn[0], cs[lv], sn[lv], cs[2 * lv], sn[2 * lv]};
}

template <class T>
__device__ __forceinline__ void f4_pair(T a0k, T a1k, T a2k, T a3k, T a0kc, T a1kc, T a2kc, T a3kc,
                                        const Tw<T> &w, T &bk0, T &bk1, T &bk2, T &bk3, T &bc0,
                                        T &bc1, T &bc2, T &bc3) {
  const T x1p = w.c1 * a1k - w.s1 * a1kc;
  const T y1p = w.c1 * a1kc + w.s1 * a1k;
  const T x2p = w.c2 * a2k - w.s2 * a2kc;
  const T y2p = w.c2 * a2kc + w.s2 * a2k;
  const T x3p = w.c3 * a3k - w.s3 * a3kc;
  const T y3p = w.c3 * a3kc + w.s3 * a3k;
  const T t1r = a0k + x2p;
  const T t1i = a0kc + y2p;
  const T t2r = x1p + x3p;
  const T t2i = y1p + y3p;
  const T t3r = a0k - x2p;
  const T t3i = a0kc - y2p;
  const T t4r = x3p - x1p;
  const T t4i = y1p - y3p;
  bk0 = t1r + t2r;
  bc0 = t3r - t4i;
  bk1 = t3r + t4i;
  bc1 = t1r - t2r;
  bk2 = t2i - t1i;
  bc2 = t3i + t4r;
  bk3 = t4r - t3i;
  bc3 = t1i + t2i;
}
template <class T>
__device__ __forceinline__ void f4_zero(T a0, T a1, T a2, T a3, T &b0, T &b1, T &b2, T &b3) {
  const T t1r = a0 + a2;
  const T t2r = a1 + a3;
  b0 = t1r + t2r;
  b1 = a0 - a2;
  b2 = t1r - t2r;
  b3 = a3 - a1;
}
template <class T>
__device__ __forceinline__ void f4_mid(T a0, T a1, T a2, T a3, T &b0, T &b1, T &b2, T &b3) {
  const T rtf12 = (T)0.7071067811865475244008443621048490392848359376884740365883398689953662;
  const T q1 = rtf12 * (a1 - a3);
  const T q2 = rtf12 * (a1 + a3);
  b0 = a0 + q1;
  b1 = a0 - q1;
  b2 = a2 - q2;
  b3 = -a2 - q2;
}
template <class T>
__device__ __forceinline__ void r4_pair(T ak0, T ak1, T ak2, T ak3, T akc0, T akc1, T akc2, T akc3,
                                        const Tw<T> &w, T &bk0, T &bk1, T &bk2, T &bk3, T &bc0,
                                        T &bc1, T &bc2, T &bc3) {
  const T t1r = ak0 + akc1;
  const T t1i = akc3 - ak2;
  const T t2r = ak1 + akc0;
  const T t2i = akc2 - ak3;
  const T t3r = ak0 - akc1;
  const T t3i = akc3 + ak2;
  const T t4r = ak1 - akc0;
  const T t4i = akc2 + ak3;
  const T x1p = t3r + t4i;
  const T y1p = t3i - t4r;
  const T x2p = t1r - t2r;
  const T y2p = t1i - t2i;
  const T x3p = t3r - t4i;
  const T y3p = t3i + t4r;
  bk0 = t1r + t2r;
  bc0 = t1i + t2i;
  bk1 = w.c1 * x1p - w.s1 * y1p;
  bc1 = w.c1 * y1p + w.s1 * x1p;
  bk2 = w.c2 * x2p - w.s2 * y2p;
  bc2 = w.c2 * y2p + w.s2 * x2p;
  bk3 = w.c3 * x3p - w.s3 * y3p;
  bc3 = w.c3 * y3p + w.s3 * x3p;
}
template <class T>
__device__ __forceinline__ void r4_zero(T a0, T a1, T a2, T a3, T &b0, T &b1, T &b2, T &b3) {
  const T t1r = a0 + a2;
  const T t2r = a1;
  const T t3r = a0 - a2;
  const T t4r = a3;
  b0 = t1r + t2r;
  b1 = t3r + t4r;
  b2 = t1r - t2r;
  b3 = t3r - t4r;
}
template <class T>
__device__ __forceinline__ void r4_mid(T a0, T a1, T a2, T a3, T &b0, T &b1, T &b2, T &b3) {
  const T rtf12 = (T)0.7071067811865475244008443621048490392848359376884740365883398689953662;
  b0 = a0 + a1;
  b2 = a3 - a2;
  const T t3r = a0 - a1;
  const T t4r = a3 + a2;
  b1 = rtf12 * (t3r + t4r);
  b3 = rtf12 * (t4r - t3r);
}

// ---- passes -----------------------------------------------------------------
// Pass kinds, by the stages they hold (named in forward order; backward runs
// them mirrored): P24 the 2 and the first 4; P44A the first two 4s (lv = 1);
// P44 two 4s of lv = l and 4 l; P4 a single, last 4 of lv = l.
enum PassKind { P24, P44A, P44, P4 };
template <int N, int PASS, bool NARROW>  // PASS in forward order
struct Pass {
  static constexpr int L2N = __builtin_ctz(N);
  static constexpr bool has2 = L2N & 1;
  static constexpr int n4 = L2N >> 1;
  static constexpr int rest = n4 - (has2 ? 1 : 2);  // 4s after the first pass
  static constexpr int npass = 1 + (NARROW ? rest : (rest + 1) / 2);
  static constexpr int l = PASS == 0 ? 1 : (has2 ? 8 : 16) << ((NARROW ? 2 : 4) * (PASS - 1));
  static constexpr PassKind kind = PASS == 0 ? (has2 ? P24 : P44A)
                                   : NARROW || (PASS == npass - 1 && rest % 2) ? P4 : P44;
  // values per unit, and the stride of the units' values on the side with
  // neighbouring rows (the input forward, the output backward)
  static constexpr int per = kind == P44 ? 32 : kind == P44A ? 16 : 8;
  static constexpr int R = kind == P4 ? N / (4 * l) : kind == P24 ? N / 8 : N / (16 * l);
  static constexpr int units = N / per;
};

// Whether the passes after the first hold one stage instead of two: half the
// values to a thread, so twice the wavefronts, for one more exchange through
// LDS.  Up to 512^2 a launch has less than a wavefront per SIMD and the
// wavefronts pay; us per launch, wide -> narrow (best batch), FP64:
//   256: one field 4.3 -> 3.6, four 4.5 -> 3.9
//   512: one field 5.1 -> 4.4, four 7.1 -> 6.7, with a derivative 8.9 -> 8.0
//  1024: one field 8.5 -> 7.7, four 18.5 -> 19.0, with a derivative 20.1 -> 21.7
// and FP32 512: one field 4.5 -> 3.9, four with a derivative 5.9 -> 5.6.
constexpr bool fft_narrow(int N) { return N >= 64 && N <= 512; }
// Threads per vector: 32 values to a thread, 16 with narrow passes, fewer
// for the shortest lengths.
constexpr int fft_threads_per_vector(int N) {
  return N <= 16 ? 1 : N <= 64 ? 4 : N / (fft_narrow(N) ? 16 : 32);
}

// Positions of unit u's values: one or two rows of H values, value j of a
// row at base + step j.  WIDE: the side where a row's values lie R apart,
// else R l apart.
template <class P>
struct Rows {
  static constexpr int n = P::kind == P24 || P::kind == P44A ? 1 : 2;
  static constexpr int H = P::per / n;
  template <bool WIDE>
  static constexpr int step() {
    return n == 1 || WIDE ? P::R : P::R * P::l;
  }
  template <bool WIDE>
  static __device__ __forceinline__ int base(int u, int row) {
    if constexpr (n == 1) return u;
    const int i = u % P::R, q = u / P::R;
    // row q and its partner l - q; q = 0: rows 0 and l / 2
    const int k = row == 0 ? q : (q == 0 ? P::l / 2 : P::l - q);
    return i + P::R * (WIDE ? H * k : k);
  }
};

// unit u's stages in place
template <int N, class P, bool FWD, class T>
__device__ __forceinline__ void unit_stages(T (&x)[P::per], int u, const T *__restrict__ trig) {
  constexpr int l = P::l;
  if constexpr (P::kind == P24) {
    T y[8];
    if (FWD) {
      T z0[4], z1[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        z0[j] = x[j] + x[j + 4];
        z1[j] = x[j] - x[j + 4];
      }
      f4_zero(z0[0], z0[1], z0[2], z0[3], y[0], y[2], y[4], y[6]);
      f4_mid(z1[0], z1[1], z1[2], z1[3], y[1], y[3], y[5], y[7]);
    } else {
      T w0[4], w1[4];
      r4_zero(x[0], x[2], x[4], x[6], w0[0], w0[1], w0[2], w0[3]);
      r4_mid(x[1], x[3], x[5], x[7], w1[0], w1[1], w1[2], w1[3]);
#pragma unroll
      for (int j = 0; j < 4; j++) {
        y[j] = w0[j] + w1[j];
        y[j + 4] = w0[j] - w1[j];
      }
    }
#pragma unroll
    for (int j = 0; j < 8; j++) x[j] = y[j];
  } else if constexpr (P::kind == P4) {
    const int k = u / P::R;
    if (k == 0) {
      if (FWD) {
        f4_zero(x[0], x[1], x[2], x[3], x[0], x[1], x[2], x[3]);
        f4_mid(x[4], x[5], x[6], x[7], x[4], x[5], x[6], x[7]);
      } else {
        r4_zero(x[0], x[1], x[2], x[3], x[0], x[1], x[2], x[3]);
        r4_mid(x[4], x[5], x[6], x[7], x[4], x[5], x[6], x[7]);
      }
    } else {
      const Tw<T> w = twiddle<N>(trig, l, k);
      if (FWD)
        f4_pair(x[0], x[1], x[2], x[3], x[4], x[5], x[6], x[7], w, x[0], x[1], x[2], x[3], x[4],
                x[5], x[6], x[7]);
      else
        r4_pair(x[0], x[1], x[2], x[3], x[4], x[5], x[6], x[7], w, x[0], x[1], x[2], x[3], x[4],
                x[5], x[6], x[7]);
    }
  } else {
    // the rows of k = 0 (and of k = l/2 when the pass has l > 1)
    auto row0 = [&](T *v) {
      if (FWD) {
        // stage lv = l: row 0 of each offset; then rows 0, (l, 3l), 2l of 4l
#pragma unroll
        for (int j = 0; j < 4; j++)
          f4_zero(v[j], v[j + 4], v[j + 8], v[j + 12], v[j], v[j + 4], v[j + 8], v[j + 12]);
        const Tw<T> w = twiddle<N>(trig, 4 * l, l);
        T y[16];
        f4_zero(v[0], v[1], v[2], v[3], y[0], y[4], y[8], y[12]);
        f4_pair(v[4], v[5], v[6], v[7], v[12], v[13], v[14], v[15], w, y[1], y[5], y[9], y[13],
                y[3], y[7], y[11], y[15]);
        f4_mid(v[8], v[9], v[10], v[11], y[2], y[6], y[10], y[14]);
#pragma unroll
        for (int j = 0; j < 16; j++) v[j] = y[j];
      } else {
        const Tw<T> w = twiddle<N>(trig, 4 * l, l);
        T y[16];  // y[4 J + j]: row l J of stage 4 l, offset j
        r4_zero(v[0], v[4], v[8], v[12], y[0], y[1], y[2], y[3]);
        r4_pair(v[1], v[5], v[9], v[13], v[3], v[7], v[11], v[15], w, y[4], y[5], y[6], y[7],
                y[12], y[13], y[14], y[15]);
        r4_mid(v[2], v[6], v[10], v[14], y[8], y[9], y[10], y[11]);
#pragma unroll
        for (int j = 0; j < 4; j++)
          r4_zero(y[j], y[4 + j], y[8 + j], y[12 + j], v[j], v[j + 4], v[j + 8], v[j + 12]);
      }
    };
    if constexpr (P::kind == P44A) {
      row0(x);
    } else {
      const int k = u / P::R;
      T *a = x, *b = x + 16;
      if (k == 0) {
        row0(a);
        const Tw<T> w0 = twiddle<N>(trig, 4 * l, l / 2), w1 = twiddle<N>(trig, 4 * l, l / 2 + l);
        T y[16];
        if (FWD) {
#pragma unroll
          for (int j = 0; j < 4; j++)
            f4_mid(b[j], b[j + 4], b[j + 8], b[j + 12], b[j], b[j + 4], b[j + 8], b[j + 12]);
          f4_pair(b[0], b[1], b[2], b[3], b[12], b[13], b[14], b[15], w0, y[0], y[4], y[8], y[12],
                  y[3], y[7], y[11], y[15]);
          f4_pair(b[4], b[5], b[6], b[7], b[8], b[9], b[10], b[11], w1, y[1], y[5], y[9], y[13],
                  y[2], y[6], y[10], y[14]);
#pragma unroll
          for (int j = 0; j < 16; j++) b[j] = y[j];
        } else {
          r4_pair(b[0], b[4], b[8], b[12], b[3], b[7], b[11], b[15], w0, y[0], y[1], y[2], y[3],
                  y[12], y[13], y[14], y[15]);
          r4_pair(b[1], b[5], b[9], b[13], b[2], b[6], b[10], b[14], w1, y[4], y[5], y[6], y[7],
                  y[8], y[9], y[10], y[11]);
#pragma unroll
          for (int j = 0; j < 4; j++)
            r4_mid(y[j], y[4 + j], y[8 + j], y[12 + j], b[j], b[j + 4], b[j + 8], b[j + 12]);
        }
      } else if (FWD) {
        {
          const Tw<T> w = twiddle<N>(trig, l, k);
#pragma unroll
          for (int j = 0; j < 4; j++)
            f4_pair(a[j], a[j + 4], a[j + 8], a[j + 12], b[j], b[j + 4], b[j + 8], b[j + 12], w,
                    a[j], a[j + 4], a[j + 8], a[j + 12], b[j], b[j + 4], b[j + 8], b[j + 12]);
        }
        // a[4 j + j'], b[4 j + j']: rows k + l j and l - k + l j of stage 4 l;
        // the pairs (k + l j, l - k + l (3 - j)), each with its lower row first
        T ya[16], yb[16];
        f4_pair(a[0], a[1], a[2], a[3], b[12], b[13], b[14], b[15], twiddle<N>(trig, 4 * l, k),
                ya[0], ya[4], ya[8], ya[12], yb[3], yb[7], yb[11], yb[15]);
        f4_pair(a[4], a[5], a[6], a[7], b[8], b[9], b[10], b[11], twiddle<N>(trig, 4 * l, k + l),
                ya[1], ya[5], ya[9], ya[13], yb[2], yb[6], yb[10], yb[14]);
        f4_pair(b[0], b[1], b[2], b[3], a[12], a[13], a[14], a[15], twiddle<N>(trig, 4 * l, l - k),
                yb[0], yb[4], yb[8], yb[12], ya[3], ya[7], ya[11], ya[15]);
        f4_pair(b[4], b[5], b[6], b[7], a[8], a[9], a[10], a[11],
                twiddle<N>(trig, 4 * l, 2 * l - k), yb[1], yb[5], yb[9], yb[13], ya[2], ya[6],
                ya[10], ya[14]);
#pragma unroll
        for (int j = 0; j < 16; j++) {
          a[j] = ya[j];
          b[j] = yb[j];
        }
      } else {
        T ya[16], yb[16];  // [4 J + j]
        r4_pair(a[0], a[4], a[8], a[12], b[3], b[7], b[11], b[15], twiddle<N>(trig, 4 * l, k),
                ya[0], ya[1], ya[2], ya[3], yb[12], yb[13], yb[14], yb[15]);
        r4_pair(a[1], a[5], a[9], a[13], b[2], b[6], b[10], b[14], twiddle<N>(trig, 4 * l, k + l),
                ya[4], ya[5], ya[6], ya[7], yb[8], yb[9], yb[10], yb[11]);
        r4_pair(b[0], b[4], b[8], b[12], a[3], a[7], a[11], a[15], twiddle<N>(trig, 4 * l, l - k),
                yb[0], yb[1], yb[2], yb[3], ya[12], ya[13], ya[14], ya[15]);
        r4_pair(b[1], b[5], b[9], b[13], a[2], a[6], a[10], a[14],
                twiddle<N>(trig, 4 * l, 2 * l - k), yb[4], yb[5], yb[6], yb[7], ya[8], ya[9],
                ya[10], ya[11]);
        const Tw<T> w = twiddle<N>(trig, l, k);
#pragma unroll
        for (int j = 0; j < 4; j++)
          r4_pair(ya[j], ya[4 + j], ya[8 + j], ya[12 + j], yb[j], yb[4 + j], yb[8 + j], yb[12 + j],
                  w, a[j], a[j + 4], a[j + 8], a[j + 12], b[j], b[j + 4], b[j + 8], b[j + 12]);
      }
    }
  }
}

// ---- the kernel -------------------------------------------------------------
// Layouts: "strided" means element e of vector v is x[v + m e] (the
// reference's x(m,n) with the vector index fastest); "rows" means
// x[e + N v].  ROWS: a forward pass writes rows, a backward one reads them;
// the other side is strided.  Lanes run over the vectors first on a strided
// side and over the elements first on a rows side.  LDS holds a vector's
// values side by side, the vectors 64/V values further apart than N, so that
// the lanes of either order fall into different banks.  Blocks are mapped so
// that the blocks one XCD runs hold neighbouring vectors (shared L2 lines on
// the strided side).
template <int N, int V>
constexpr int fft_row_stride() {
  return N + (V < 64 ? 64 / V : 1);
}

// A thread's units of pass P to and from LDS.
template <class P, bool WIDE, class T, int U>
__device__ __forceinline__ void lds_put(const T (&x)[U][P::per], T *row, int u, int tv) {
#pragma unroll
  for (int i = 0; i < U; i++)
#pragma unroll
    for (int r = 0; r < Rows<P>::n; r++) {
      T *q = row + Rows<P>::template base<WIDE>(u + tv * i, r);
#pragma unroll
      for (int j = 0; j < Rows<P>::H; j++)
        q[Rows<P>::template step<WIDE>() * j] = x[i][Rows<P>::H * r + j];
    }
}
template <class P, bool WIDE, class T, int U>
__device__ __forceinline__ void lds_get(T (&x)[U][P::per], const T *row, int u, int tv) {
#pragma unroll
  for (int i = 0; i < U; i++)
#pragma unroll
    for (int r = 0; r < Rows<P>::n; r++) {
      const T *q = row + Rows<P>::template base<WIDE>(u + tv * i, r);
#pragma unroll
      for (int j = 0; j < Rows<P>::H; j++)
        x[i][Rows<P>::H * r + j] = q[Rows<P>::template step<WIDE>() * j];
    }
}

// Pass I and the ones after it: x holds what the pass before left in the
// lanes' order of (va, ua), xl receives the last pass's values in that of
// (vl, ul); between, lanes run over the vectors first (vs, us).
template <int N, bool FWD, bool NW, int I, int NP, class T, int U, int PER, int UL, int PERL>
__device__ __forceinline__ void fft_passes(const T (&x)[U][PER], T (&xl)[UL][PERL], T *lds, int va,
                                           int ua, int vs, int us, int vl, int ul, int tv,
                                           const T *__restrict__ trig) {
  constexpr int npass = Pass<N, 0, NW>::npass;
  using PP = Pass<N, FWD ? I - 1 : npass - I, NW>;
  using PC = Pass<N, FWD ? I : npass - 1 - I, NW>;
  if constexpr (I > 1) __syncthreads();  // every value has been read
  lds_put<PP, !FWD>(x, lds + va * NP, ua, tv);
  __syncthreads();
  if constexpr (I == npass - 1) {
    lds_get<PC, FWD>(xl, lds + vl * NP, ul, tv);
#pragma unroll
    for (int i = 0; i < UL; i++) unit_stages<N, PC, FWD>(xl[i], ul + tv * i, trig);
  } else {
    constexpr int UC = U * PER / PC::per;
    T y[UC][PC::per];
    lds_get<PC, FWD>(y, lds + vs * NP, us, tv);
#pragma unroll
    for (int i = 0; i < UC; i++) unit_stages<N, PC, FWD>(y[i], us + tv * i, trig);
    fft_passes<N, FWD, NW, I + 1, NP>(y, xl, lds, vs, us, vs, us, vl, ul, tv, trig);
  }
}

template <int N, bool FWD, class TI, class T, class TO, int V, bool ROWS>
__global__ void __launch_bounds__(V *fft_threads_per_vector(N)) fft_kernel(FftArgs g) {
  constexpr bool NW = fft_narrow(N);
  constexpr int TV = fft_threads_per_vector(N);
  constexpr int NP = fft_row_stride<N, V>();
  constexpr int npass = Pass<N, 0, NW>::npass;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  T *lds = (T *)lds_raw;
  const int f = blockIdx.y, tid = threadIdx.x, m = g.m;
  const T *__restrict__ trig = (const T *)g.trig;
  const int nb = gridDim.x;
  const int bid = (nb % 8 == 0) ? (blockIdx.x % 8) * (nb / 8) + blockIdx.x / 8 : blockIdx.x;
  const int v0 = bid * V;
  constexpr int nhalf = N / 2;
  // (vector, first unit) of this thread for lanes over vectors or elements
  const int vs = tid % V, us = tid / V, vr = tid / TV, ur = tid % TV;

  // first pass: global memory -> registers.  Lanes beyond the last vector
  // load it again and store nothing.
  using P0 = Pass<N, FWD ? 0 : npass - 1, NW>;
  using R0 = Rows<P0>;
  constexpr bool rows_in = !FWD && ROWS;
  constexpr int PER0 = P0::per, U0 = P0::units / TV, H0 = R0::H;
  constexpr int S0 = R0::template step<FWD>();
  const int va = rows_in ? vr : vs, ua = rows_in ? ur : us;
  const int vga = min(v0 + va, m - 1);
  T x0[U0][PER0];
  const TI *__restrict__ gin = (const TI *)g.in[f];
  const int pre = FWD ? 0 : g.pre[f];
  // the source element: mirrored for a derivative (sta2dfft.f90:169-245)
  const int vsrc = pre == 1 ? (vga == 0 ? 0 : m - vga) : vga;
  const int64_t se = rows_in ? 1 : m;  // between elements
  const TI *gv = gin + (rows_in ? (int64_t)vsrc * N : (int64_t)vsrc);
  TI raw[U0][PER0];
#pragma unroll
  for (int i = 0; i < U0; i++)
#pragma unroll
    for (int r = 0; r < R0::n; r++) {
      const int b = R0::template base<FWD>(ua + TV * i, r);
      if (pre == 2) {  // element n - e (0 for 0, which is not used)
        const TI *q = gv + se * (N - b);
        raw[i][H0 * r] = b == 0 ? gv[0] : q[0];
#pragma unroll
        for (int j = 1; j < H0; j++) raw[i][H0 * r + j] = q[-se * (S0 * j)];
      } else {
        const TI *q = gv + se * b;
#pragma unroll
        for (int j = 0; j < H0; j++) raw[i][H0 * r + j] = q[se * (S0 * j)];
      }
    }
  if constexpr (FWD) {
    if (g.sub) {
      // con2grid's mean removal (contours.f90:338-345) fused into the load
      const double subv = *g.sub / g.subdiv;
#pragma unroll
      for (int i = 0; i < U0; i++)
#pragma unroll
        for (int j = 0; j < PER0; j++) x0[i][j] = (T)(raw[i][j] - subv);
    } else {
#pragma unroll
      for (int i = 0; i < U0; i++)
#pragma unroll
        for (int j = 0; j < PER0; j++) x0[i][j] = (T)raw[i][j];
    }
  } else {
    // the derivative's wavenumber, filtered
    const double *__restrict__ dk = g.dk[f];
    if (pre == 2) {
      // along elements: der(e) from var(n-e), 0 for e = 0 and n/2
#pragma unroll
      for (int i = 0; i < U0; i++)
#pragma unroll
        for (int r = 0; r < R0::n; r++) {
          const int b = R0::template base<FWD>(ua + TV * i, r);
#pragma unroll
          for (int j = 0; j < H0; j++) {
            const int e = b + S0 * j;
            const bool z = e == 0 || e == nhalf;
            const T dkv = (T)dk[z ? 0 : 2 * (e < nhalf ? e : N - e) - 1];
            const T x = (T)raw[i][H0 * r + j];
            x0[i][H0 * r + j] = z ? (T)0.0 : (e < nhalf ? -dkv * x : dkv * x);
          }
        }
    } else if (pre == 1) {
      // across vectors (the vector index is the wavenumber, m its length)
      const int mh = m / 2;
      const bool z = vga == 0 || vga == mh;
      const T dv = (T)dk[z ? 0 : 2 * (vga < mh ? vga : m - vga) - 1];
      const T sv = vga < mh ? -dv : dv;
#pragma unroll
      for (int i = 0; i < U0; i++)
#pragma unroll
        for (int j = 0; j < PER0; j++) x0[i][j] = z ? (T)0.0 : sv * (T)raw[i][j];
    } else {
#pragma unroll
      for (int i = 0; i < U0; i++)
#pragma unroll
        for (int j = 0; j < PER0; j++) x0[i][j] = (T)raw[i][j];
    }
    // revfft pre-processing, stafft.f90:311-325
#pragma unroll
    for (int i = 0; i < U0; i++)
#pragma unroll
      for (int r = 0; r < R0::n; r++) {
        const int b = R0::template base<FWD>(ua + TV * i, r);
#pragma unroll
        for (int j = 0; j < H0; j++) {
          const int e = b + S0 * j;
          T x = x0[i][H0 * r + j];
          if (e >= nhalf + 1) x = -x;
          if (e == 0 || e == nhalf) x = (T)0.5 * x;
          x0[i][H0 * r + j] = x;
        }
      }
  }
#pragma unroll
  for (int i = 0; i < U0; i++) unit_stages<N, P0, FWD>(x0[i], ua + TV * i, trig);

  // last pass: registers -> global memory
  using PL = Pass<N, FWD ? npass - 1 : 0, NW>;
  using RL = Rows<PL>;
  constexpr bool rows_out = FWD && ROWS;
  constexpr int PERL = PL::per, UL = PL::units / TV, HL = RL::H;
  const int vl = npass == 1 ? va : (rows_out ? vr : vs);
  const int ul = npass == 1 ? ua : (rows_out ? ur : us);
  T xl[UL][PERL];
  if constexpr (npass == 1) {
#pragma unroll
    for (int i = 0; i < UL; i++)
#pragma unroll
      for (int j = 0; j < PERL; j++) xl[i][j] = x0[i][j];
  } else {
    fft_passes<N, FWD, NW, 1, NP>(x0, xl, lds, va, ua, vs, us, vl, ul, TV, trig);
  }
  const int vgl = v0 + vl;
  if (vgl >= m) return;
  // normalisation folded in, stafft.f90:275-284 / 394-403
  const T post = (T)g.post[f];
  constexpr int SL = RL::template step<!FWD>();
  const int64_t so = rows_out ? 1 : m;
  TO *go = (TO *)g.out[f] + (rows_out ? (int64_t)vgl * N : (int64_t)vgl);
#pragma unroll
  for (int i = 0; i < UL; i++)
#pragma unroll
    for (int r = 0; r < RL::n; r++) {
      TO *q = go + so * RL::template base<!FWD>(ul + TV * i, r);
#pragma unroll
      for (int j = 0; j < HL; j++) q[so * (SL * j)] = (TO)(xl[i][HL * r + j] * post);
    }
}

// A launch of one kernel; with timing events (ea, eb) they are recorded at
// the dispatch's own start and end, without, an ordinary launch (the one
// stream capture records).
template <int N, bool FWD, class TI, class T, class TO, int V, bool ROWS>
static int fft_launch_one(const FftArgs &g, int F, hipStream_t s, hipEvent_t ea, hipEvent_t eb) {
  constexpr int threads = V * fft_threads_per_vector(N);
  constexpr size_t shm = Pass<N, 0, fft_narrow(N)>::npass == 1 ? 0 : sizeof(T) * V * fft_row_stride<N, V>();
  auto kern = fft_kernel<N, FWD, TI, T, TO, V, ROWS>;
  if constexpr (shm > 65536) {
    // more than 64 KiB of LDS per workgroup must be requested (gfx950: 160 KiB)
    static std::atomic<bool> raised{false};
    if (!raised.load(std::memory_order_acquire)) {
      HYD_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  160 * 1024));
      raised.store(true, std::memory_order_release);
    }
  }
  const dim3 grid((g.m + V - 1) / V, F);
  if (ea && eb)
    hipExtLaunchKernelGGL(kern, grid, dim3(threads), (uint32_t)shm, s, ea, eb, 0u, g);
  else
    hipLaunchKernelGGL(kern, grid, dim3(threads), shm, s, g);
  HYD_HIP(hipGetLastError());
  return HYD_OK;
}

// Vectors per block that a length and type can run with: 32 to 512 threads
// (16 vectors of the shortest lengths) and at most 160 KiB of LDS.
constexpr bool fft_v_fits(int N, int V, int tsize) {
  const int tv = fft_threads_per_vector(N), t = V * tv;
  return t <= 512 && (t >= 32 || V == kMaxV) && (V > 1 || tv >= 64) &&
         tsize * V * (N + 64 / V) <= 160 * 1024;
}

template <int N, bool FWD, class TI, class T, class TO, bool ROWS>
static int fft_launch_v(int V, const FftArgs &g, int F, hipStream_t s, hipEvent_t ea,
                        hipEvent_t eb) {
#define HYD_FFT_V(VV)                                                                          \
  if constexpr (fft_v_fits(N, VV, (int)sizeof(T)))                                             \
    if (V == VV) {                                                                             \
      return fft_launch_one<N, FWD, TI, T, TO, VV, ROWS>(g, F, s, ea, eb);                     \
    }
  HYD_FFT_V(1)
  HYD_FFT_V(2)
  HYD_FFT_V(4)
  HYD_FFT_V(8)
  HYD_FFT_V(16)
#undef HYD_FFT_V
  set_error("fft: unsupported batch");
  return HYD_EARG;
}

// The lengths up to 512 (lo) and from 1024 (hi): one translation unit per
// range and precision instantiates these, so that they compile in parallel.
template <bool FWD, class TI, class T, class TO, bool ROWS>
int fft_run_lo(int n, int V, const FftArgs &g, int F, hipStream_t s, hipEvent_t ea,
               hipEvent_t eb) {
  switch (n) {
    case 8: return fft_launch_v<8, FWD, TI, T, TO, ROWS>(V, g, F, s, ea, eb);
    case 16: return fft_launch_v<16, FWD, TI, T, TO, ROWS>(V, g, F, s, ea, eb);
    case 32: return fft_launch_v<32, FWD, TI, T, TO, ROWS>(V, g, F, s, ea, eb);
    case 64: return fft_launch_v<64, FWD, TI, T, TO, ROWS>(V, g, F, s, ea, eb);
    case 128: return fft_launch_v<128, FWD, TI, T, TO, ROWS>(V, g, F, s, ea, eb);
    case 256: return fft_launch_v<256, FWD, TI, T, TO, ROWS>(V, g, F, s, ea, eb);
    default: return fft_launch_v<512, FWD, TI, T, TO, ROWS>(V, g, F, s, ea, eb);
  }
}
template <bool FWD, class TI, class T, class TO, bool ROWS>
int fft_run_hi(int n, int V, const FftArgs &g, int F, hipStream_t s, hipEvent_t ea,
               hipEvent_t eb) {
  switch (n) {
    case 1024: return fft_launch_v<1024, FWD, TI, T, TO, ROWS>(V, g, F, s, ea, eb);
    case 2048: return fft_launch_v<2048, FWD, TI, T, TO, ROWS>(V, g, F, s, ea, eb);
    default: return fft_launch_v<4096, FWD, TI, T, TO, ROWS>(V, g, F, s, ea, eb);
  }
}
#define HYD_FFT_INSTANTIATE(RUN, FWD, TI, T, TO, ROWS)                                      \
  template int RUN<FWD, TI, T, TO, ROWS>(int, int, const FftArgs &, int, hipStream_t,       \
                                         hipEvent_t, hipEvent_t);

}  // namespace hyd
