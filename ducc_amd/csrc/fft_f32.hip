// fft_f32.hip -- k_fft in single precision, workgroups of up to 64 KiB of lines
// (see fft_impl.h).
#include "fft_impl.h"

DMX_INSTANTIATE_FFT(float, FFT_MAXEL32)
