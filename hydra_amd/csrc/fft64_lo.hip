// The FP64 FFT passes, lengths up to 512.
#include "fft_kernel.h"

namespace hyd {

HYD_FFT_INSTANTIATE(fft_run_lo, true, double, double, double, true)
HYD_FFT_INSTANTIATE(fft_run_lo, true, double, double, double, false)
HYD_FFT_INSTANTIATE(fft_run_lo, false, double, double, double, false)
HYD_FFT_INSTANTIATE(fft_run_lo, false, double, double, double, true)

}  // namespace hyd
