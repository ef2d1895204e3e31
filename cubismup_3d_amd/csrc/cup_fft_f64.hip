// cup_fft_f64.hip -- the FP64 forms of cup_fft.hip, compiled beside the rest of it.
#define CUP_FFT_F64
#include "cup_fft.hip"
