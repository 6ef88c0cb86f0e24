// Two-DFT FFT passes (pp_fft2.h) of the lengths PP_FFT2_D.
#include "pp_fft2.h"

PP_FFT2_TABLE(fft2_table_d, PP_FFT2_D)
