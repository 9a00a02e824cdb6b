// The FP64 FFT passes, lengths from 1024.
#include "fft_kernel.h"

namespace hyd {

HYD_FFT_INSTANTIATE(fft_run_hi, true, double, double, double, true)
HYD_FFT_INSTANTIATE(fft_run_hi, true, double, double, double, false)
HYD_FFT_INSTANTIATE(fft_run_hi, false, double, double, double, false)
HYD_FFT_INSTANTIATE(fft_run_hi, false, double, double, double, true)

}  // namespace hyd
