// Two-DFT FFT passes (pp_fft2.h) of the lengths PP_FFT2_E.
#include "pp_fft2.h"

PP_FFT2_TABLE(fft2_table_e, PP_FFT2_E)
