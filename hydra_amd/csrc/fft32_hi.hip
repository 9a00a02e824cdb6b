// The FP32 FFT passes, lengths from 1024.
#include "fft_kernel.h"

namespace hyd {

HYD_FFT_INSTANTIATE(fft_run_hi, true, float, float, float, true)
HYD_FFT_INSTANTIATE(fft_run_hi, true, float, float, double, false)
HYD_FFT_INSTANTIATE(fft_run_hi, false, double, float, float, false)
HYD_FFT_INSTANTIATE(fft_run_hi, false, float, float, float, true)

}  // namespace hyd
