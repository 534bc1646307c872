// Specialised FFT kernels of the lengths in SFNO_FFT_LENGTHS_C.
#include "fft_kernels.h"

#include "fft_fast.h"
#include "fft_lengths.h"

SFNO_FFT_PART(C, SFNO_FFT_LENGTHS_C)
