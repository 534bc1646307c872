// Specialised FFT kernels of the lengths in SFNO_FFT_LENGTHS_D.
#include "fft_kernels.h"

#include "fft_fast.h"
#include "fft_lengths.h"

SFNO_FFT_PART(D, SFNO_FFT_LENGTHS_D)
