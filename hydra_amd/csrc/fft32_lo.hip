// The FP32 FFT passes, lengths up to 512.
#include "fft_kernel.h"

namespace hyd {

HYD_FFT_INSTANTIATE(fft_run_lo, true, float, float, float, true)
HYD_FFT_INSTANTIATE(fft_run_lo, true, float, float, double, false)
HYD_FFT_INSTANTIATE(fft_run_lo, false, double, float, float, false)
HYD_FFT_INSTANTIATE(fft_run_lo, false, float, float, float, true)

}  // namespace hyd
