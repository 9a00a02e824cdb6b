// fft.hip -- the 2D and 1D transforms of stafft/sta2dfft built from batched
// passes of the kernel of fft_kernel.h (compiled in fft64_*.hip and
// fft32_*.hip).
//
// ptospc = x-transform reading strided (ny vectors) and writing rows (this
// is the transpose of sta2dfft.f90:122-126), then an in-place strided
// y-transform.  spctop = strided y-inverse into a work array, then an
// x-inverse reading rows and writing strided (sta2dfft.f90:152-162).
// Derivatives and the mean removal are fused into the passes.
#include "fft_kernel.h"

namespace hyd {

#define HYD_FFT_EXTERN(FWD, TI, T, TO, ROWS)                                              \
  extern template int fft_run_lo<FWD, TI, T, TO, ROWS>(int, int, const FftArgs &, int,    \
                                                       hipStream_t, hipEvent_t, hipEvent_t); \
  extern template int fft_run_hi<FWD, TI, T, TO, ROWS>(int, int, const FftArgs &, int,    \
                                                       hipStream_t, hipEvent_t, hipEvent_t);
HYD_FFT_EXTERN(true, double, double, double, true)
HYD_FFT_EXTERN(true, double, double, double, false)
HYD_FFT_EXTERN(false, double, double, double, false)
HYD_FFT_EXTERN(false, double, double, double, true)
HYD_FFT_EXTERN(true, float, float, float, true)
HYD_FFT_EXTERN(true, float, float, double, false)
HYD_FFT_EXTERN(false, double, float, float, false)
HYD_FFT_EXTERN(false, float, float, float, true)

// Batch without a tuned value: up to 256 threads and 80 KiB (two blocks a
// CU), no more vectors than the next power of two of m.
static int fft_default_v(int n, int m, int tsize) {
  int best = 0;
  for (int V = kMaxV; V >= 1; V /= 2)
    if (fft_v_fits(n, V, tsize)) {
      if (best == 0) best = V;
      const bool roomy = V * fft_threads_per_vector(n) <= 256 && tsize * V * (n + 64 / V) <= 81920;
      if (!roomy || V >= 2 * m) continue;
      return V;
    }
  return best;
}

template <bool FWD, class TI, class T, class TO, bool ROWS>
static int fft_launch_t(Ctx &c, int F, const TI *const *in, TO *const *out, int n, int m,
                        const int *pre, const double *const *dk, const double *post,
                        const T *trig, const double *sub = nullptr, double subdiv = 1.0) {
  if (F < 1 || F > kMaxF) {
    set_error("fft: batch of 1..4 fields");
    return HYD_EARG;
  }
  if (n < 8 || n > 4096 || (n & (n - 1))) {
    set_error("fft: transform length must be a power of two in [8, 4096]");
    return HYD_EFACTOR;
  }
  FftArgs g;
  for (int f = 0; f < kMaxF; f++) {
    const int q = f < F ? f : 0;
    g.in[f] = in[q];
    g.out[f] = out[q];
    g.dk[f] = dk ? dk[q] : nullptr;
    g.pre[f] = pre ? pre[q] : 0;
    g.post[f] = post[q];
  }
  g.trig = trig;
  g.sub = sub;
  g.subdiv = subdiv;
  g.m = m;
  // batch per workgroup: the autotuned value of this layout class and field
  // count at the context's length, else a default
  const int cls = FWD ? (ROWS ? 0 : 1) : (ROWS ? 3 : 2);
  int V = 0;
  if (n == c.c.nx && m == n) {
    if (sizeof(T) == 4) V = c.fft_v32[cls];
    else if (F == 1) V = c.fft_v1[cls];
    else if (F >= 3) V = c.fft_v4[cls];
    else V = c.fft_v[cls];
  }
  if (V < 1 || !fft_v_fits(n, V, (int)sizeof(T))) V = fft_default_v(n, m, (int)sizeof(T));
  // one launch reads and writes F x m vectors of n values
  KTimer tk(c, sizeof(T) == 8 ? (FWD ? "k:fft_fwd" : "k:fft_rev") : (FWD ? "k:fft32_fwd" : "k:fft32_rev"),
            (int64_t)(sizeof(TI) + sizeof(TO)) * n * m * F, true);
  if (n <= 512) return fft_run_lo<FWD, TI, T, TO, ROWS>(n, V, g, F, c.s, tk.start(), tk.stop());
  return fft_run_hi<FWD, TI, T, TO, ROWS>(n, V, g, F, c.s, tk.start(), tk.stop());
}

// Holds the stream for some 40 us, so that the launches timed after it are
// queued ahead of the GPU: at 3-10 us a pass, launches issued to an idle
// stream would time the host instead.
__global__ void fft_tune_hold() {
  for (int i = 0; i < 12; i++) __builtin_amdgcn_s_sleep(127);
}

// A pair of events for each batch that a class can try.
static constexpr int kTuneV = 5;  // 1, 2, 4, 8, 16
static_assert(1 << (kTuneV - 1) == kMaxV, "batches");
struct TuneEvents {
  hipEvent_t a[kTuneV] = {}, b[kTuneV] = {};
};

// The best batch of one layout class: each candidate timed over three
// rounds that visit the candidates in turn (so that a slow spell of the
// device does not favour one), keeping its best round.  A round is queued
// whole behind one hold and waited for once (a hold and a wait for each
// candidate: hyd_init took 12.0 ms instead of 8.3 at ng=128, 21.7 instead of
// 16.1 at ng=256).  Every V gives
// bit-identical results (each vector's arithmetic is the same).
template <class RUN>
static int fft_tune_class(Ctx &c, int n, int tsize, int &tab, const TuneEvents &ev, RUN run) {
  float best[kTuneV];
  for (float &b : best) b = 1e30f;
  for (int round = 0; round < 3; round++) {
    hipLaunchKernelGGL(fft_tune_hold, dim3(1), dim3(64), 0, c.s);
    for (int k = 0; k < kTuneV; k++) {
      if (!fft_v_fits(n, 1 << k, tsize)) continue;
      tab = 1 << k;
      HYD_CHECK(run());
      HYD_HIP(hipEventRecord(ev.a[k], c.s));
      for (int r = 0; r < 8; r++) HYD_CHECK(run());
      HYD_HIP(hipEventRecord(ev.b[k], c.s));
    }
    HYD_HIP(hipStreamSynchronize(c.s));
    for (int k = 0; k < kTuneV; k++) {
      if (!fft_v_fits(n, 1 << k, tsize)) continue;
      float ms = 0.0f;
      HYD_HIP(hipEventElapsedTime(&ms, ev.a[k], ev.b[k]));
      best[k] = std::min(best[k], ms);
    }
  }
  int bk = 0;
  for (int k = 1; k < kTuneV; k++)
    if (best[k] < best[bk]) bk = k;
  tab = 1 << bk;
  return HYD_OK;
}

// Autotuner: the batch V of each layout class (forward strided->rows,
// forward strided->strided, reverse strided->strided, reverse rows->strided)
// on scratch fields, for two-field launches (fft_v), one-field ones (fft_v1:
// half the grid, so a smaller batch may fill the device better) and
// four-field ones (fft_v4; outputs in the fine-grid scratch), and for the
// mixed step's FP32 passes (fft_v32).
static int fft_tune_all(Ctx &c, const TuneEvents &ev) {
  const int n = c.c.nx;
  const double post[4] = {1.0, 1.0, 1.0, 1.0};
  for (int F : {2, 1, 4}) {
    int *tab = F == 2 ? c.fft_v : (F == 1 ? c.fft_v1 : c.fft_v4);
    const double *in[4] = {c.wa, c.wc, c.wb, c.wd};
    double *out[4] = {F == 4 ? c.fq : c.wb, F == 4 ? c.fq + c.N : c.wd, c.fq + 2 * c.N,
                      c.fq + 3 * c.N};
    HYD_CHECK(fft_tune_class(c, n, 8, tab[0], ev, [&]() {
      return fft_launch_t<true, double, double, double, true>(c, F, in, out, n, n, nullptr, nullptr,
                                                              post, c.xtrig);
    }));
    HYD_CHECK(fft_tune_class(c, n, 8, tab[1], ev, [&]() {
      return fft_launch_t<true, double, double, double, false>(c, F, in, out, n, n, nullptr,
                                                               nullptr, post, c.xtrig);
    }));
    HYD_CHECK(fft_tune_class(c, n, 8, tab[2], ev, [&]() {
      return fft_launch_t<false, double, double, double, false>(c, F, in, out, n, n, nullptr,
                                                                nullptr, post, c.ytrig);
    }));
    HYD_CHECK(fft_tune_class(c, n, 8, tab[3], ev, [&]() {
      return fft_launch_t<false, double, double, double, true>(c, F, in, out, n, n, nullptr,
                                                               nullptr, post, c.ytrig);
    }));
  }
  if (c.p.precision == 1) {
    const float *in[2] = {c.fa32, c.fc32};
    float *out[2] = {c.fb32, c.fd32};
    const double *ind[2] = {c.wa, c.wc};
    double *outd[2] = {c.wb, c.wd};
    int *tab = c.fft_v32;
    HYD_CHECK(fft_tune_class(c, n, 4, tab[0], ev, [&]() {
      return fft_launch_t<true, float, float, float, true>(c, 2, in, out, n, n, nullptr, nullptr,
                                                           post, c.xtrig32);
    }));
    HYD_CHECK(fft_tune_class(c, n, 4, tab[1], ev, [&]() {
      return fft_launch_t<true, float, float, double, false>(c, 2, in, outd, n, n, nullptr, nullptr,
                                                             post, c.xtrig32);
    }));
    HYD_CHECK(fft_tune_class(c, n, 4, tab[2], ev, [&]() {
      return fft_launch_t<false, double, float, float, false>(c, 2, ind, out, n, n, nullptr,
                                                              nullptr, post, c.ytrig32);
    }));
    HYD_CHECK(fft_tune_class(c, n, 4, tab[3], ev, [&]() {
      return fft_launch_t<false, float, float, float, true>(c, 2, in, out, n, n, nullptr, nullptr,
                                                            post, c.ytrig32);
    }));
  }
  return HYD_OK;
}

int fft_autotune(Ctx &c) {
  TuneEvents ev;
  int rc = HYD_OK;
  for (int k = 0; k < kTuneV; k++)
    if (hipEventCreate(&ev.a[k]) != hipSuccess || hipEventCreate(&ev.b[k]) != hipSuccess)
      rc = HYD_EHIP;
  if (rc == HYD_OK) rc = fft_tune_all(c, ev);
  for (int k = 0; k < kTuneV; k++) {
    if (ev.a[k]) hipEventDestroy(ev.a[k]);
    if (ev.b[k]) hipEventDestroy(ev.b[k]);
  }
  if (rc != HYD_OK) set_error("fft autotuning failed");
  return rc;
}

// ---- FP64 transforms --------------------------------------------------------
// ptospc, sta2dfft.f90:103-132, of F fields; sub/subdiv a mean to remove.
static int fft_forward_2d(Ctx &c, int F, const double *const *rvar, double *const *svar,
                          const double *sub = nullptr, double subdiv = 1.0) {
  const int n = c.c.nx;
  KTimer t(c, "fft_ptospc", 4 * 8 * c.N * F);
  const double p[kMaxF] = {c.plan.fnorm, c.plan.fnorm, c.plan.fnorm, c.plan.fnorm};
  HYD_CHECK((fft_launch_t<true, double, double, double, true>(c, F, rvar, svar, n, n, nullptr,
                                                              nullptr, p, c.xtrig, sub,
                                                              subdiv)));
  HYD_CHECK((fft_launch_t<true, double, double, double, false>(
      c, F, (const double *const *)svar, svar, n, n, nullptr, nullptr, p, c.ytrig)));
  return HYD_OK;
}

// ptospc of rvar - *sum / ndiv (the subtraction done while loading).
int fft_ptospc_mean(Ctx &c, const double *rvar, const double *sum, double ndiv, double *svar) {
  return fft_forward_2d(c, 1, &rvar, &svar, sum, ndiv);
}

int fft_ptospc(Ctx &c, const double *rvar, double *svar) {
  return fft_forward_2d(c, 1, &rvar, &svar);
}

int fft_ptospc_n(Ctx &c, int F, const double *const *rvar, double *const *svar) {
  return fft_forward_2d(c, F, rvar, svar);
}

// spctop, sta2dfft.f90:136-165, of F fields (two launches whatever F is),
// each with an optional fused xderiv / yderiv of the input
// (spectral.f90:328-332, 359-363) and a sign folded into the last store
// (spectral.f90:335-339).  tmp: (nx,ny) work arrays.
int fft_spctop_n(Ctx &c, int F, const double *const *svar, double *const *rvar, const int *pre,
                 const double *post_sign, double *const *tmp) {
  const int n = c.c.nx;
  KTimer t(c, "fft_spctop", 4 * 8 * c.N * F);
  const double *dk[kMaxF];
  double p1[kMaxF], p2[kMaxF];
  for (int f = 0; f < F; f++) {
    dk[f] = pre[f] == PRE_XDERIV ? c.hrkx : (pre[f] == PRE_YDERIV ? c.hrky : nullptr);
    p1[f] = c.plan.rnorm;
    p2[f] = c.plan.rnorm * post_sign[f];
  }
  // y-inverse: vectors kx (strided), elements ky.  xderiv acts across the
  // vectors (pre=1), yderiv along the elements (pre=2).
  HYD_CHECK((fft_launch_t<false, double, double, double, false>(c, F, svar, tmp, n, n, pre, dk, p1,
                                                                c.ytrig)));
  HYD_CHECK((fft_launch_t<false, double, double, double, true>(
      c, F, (const double *const *)tmp, rvar, n, n, nullptr, nullptr, p2, c.xtrig)));
  return HYD_OK;
}

int fft_spctop(Ctx &c, const double *svar, double *rvar, int pre, double post_sign, double *tmp) {
  return fft_spctop_n(c, 1, &svar, &rvar, &pre, &post_sign, &tmp);
}

// forfft(m, n, x) / revfft(m, n, x) on a strided (m, n) array in place
// (stafft.f90:187-406): scaled by 1/sqrt(n) forward, 2/sqrt(n) backward,
// revfft's halving of the real-only entries inside the pass.
int fft_1d(Ctx &c, bool fwd, int m, int n, double *x, const double *trig) {
  const double scale = fwd ? 1.0 / sqrt((double)n) : 2.0 / sqrt((double)n);
  const double *in = x;
  if (fwd)
    return fft_launch_t<true, double, double, double, false>(c, 1, &in, &x, n, m, nullptr, nullptr,
                                                             &scale, trig);
  return fft_launch_t<false, double, double, double, false>(c, 1, &in, &x, n, m, nullptr, nullptr,
                                                            &scale, trig);
}

// ---- mixed precision --------------------------------------------------------
// FP32 arithmetic, FP64 spectral state: ptospc from FP32 physical fields to
// FP64 coefficients, spctop from FP64 coefficients (optionally
// differentiated) to FP32 fields.
int fft_ptospc32_n(Ctx &c, int F, const float *const *rvar, double *const *svar,
                   float *const *tmp, const double *mean) {
  const int n = c.c.nx;
  const double p[kMaxF] = {c.plan.fnorm, c.plan.fnorm, c.plan.fnorm, c.plan.fnorm};
  HYD_CHECK((fft_launch_t<true, float, float, float, true>(c, F, rvar, tmp, n, n, nullptr, nullptr,
                                                           p, c.xtrig32, mean, 1.0)));
  HYD_CHECK((fft_launch_t<true, float, float, double, false>(
      c, F, (const float *const *)tmp, svar, n, n, nullptr, nullptr, p, c.ytrig32)));
  return HYD_OK;
}

// ptospc32 of rvar - *mean (the subtraction done in double while loading,
// as con2grid_mixed's mean removal).
int fft_ptospc32_mean(Ctx &c, const float *rvar, const double *mean, double *svar) {
  return fft_ptospc32_n(c, 1, &rvar, &svar, &c.tmp32, mean);
}

int fft_spctop32_n(Ctx &c, int F, const double *const *svar, float *const *rvar, const int *pre,
                   const double *post_sign, float *const *tmp) {
  const int n = c.c.nx;
  const double *dk[kMaxF];
  double p1[kMaxF], p2[kMaxF];
  for (int f = 0; f < F; f++) {
    dk[f] = pre[f] == PRE_XDERIV ? c.hrkx : (pre[f] == PRE_YDERIV ? c.hrky : nullptr);
    p1[f] = c.plan.rnorm;
    p2[f] = c.plan.rnorm * post_sign[f];
  }
  HYD_CHECK((fft_launch_t<false, double, float, float, false>(c, F, svar, tmp, n, n, pre, dk, p1,
                                                              c.ytrig32)));
  HYD_CHECK((fft_launch_t<false, float, float, float, true>(
      c, F, (const float *const *)tmp, rvar, n, n, nullptr, nullptr, p2, c.xtrig32)));
  return HYD_OK;
}

int fft_spctop32(Ctx &c, const double *svar, float *rvar, int pre, double post_sign) {
  return fft_spctop32_n(c, 1, &svar, &rvar, &pre, &post_sign, &c.tmp32);
}

}  // namespace hyd
