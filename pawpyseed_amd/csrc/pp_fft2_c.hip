// Two-DFT FFT passes (pp_fft2.h) of the lengths PP_FFT2_C.
#include "pp_fft2.h"

PP_FFT2_TABLE(fft2_table_c, PP_FFT2_C)
