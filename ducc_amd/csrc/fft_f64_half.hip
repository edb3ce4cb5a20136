// fft_f64_half.hip -- k_fft in double precision, workgroups of up to 32 KiB of lines
// (see fft_impl.h).
#include "fft_impl.h"

DMX_INSTANTIATE_FFT(double, FFT_MAXEL64 / 2)
