// Internal entry points of the source files that instantiate the specialised FFTs (fft_kernels.h), each for its share of the
// lengths (fft_lengths.h).
#pragma once
#include "sfno_internal.h"

namespace sfno {

// all answer SFNO_EUNSUPPORTED for a length the part does not hold
#define SFNO_FFT_PART_DECL(P)                                                                                                 \
    int fft_part_lon_##P(bool inverse, const FftPlan& p, const void* in, const void* in2, void* out, int64_t rows, int nlat, int mmax, int ld, \
                         int grid_dtype, hipStream_t s, float2* lat_stats, const int* kept, int width);                                                                   \
    int fft_part_lat_##P(bool inverse, const FftPlan& p, const float* in, float* out, int mmax, int lmax, int ld, const float* mscale, hipStream_t s);   \
    int fft_part_rows_##P(bool inverse, const FftPlan& p, const float* in, float* out, int64_t rows, int nlat, int mmax, int cs, hipStream_t s); \
    int fft_part_cols_##P(bool inverse, const FftPlan& p, const float2* in, float2* out, int64_t rows, int mmax, int lmax, \
                          const float* mscale, hipStream_t s)
SFNO_FFT_PART_DECL(A);
SFNO_FFT_PART_DECL(B);
SFNO_FFT_PART_DECL(C);
SFNO_FFT_PART_DECL(D);
SFNO_FFT_PART_DECL(E);
SFNO_FFT_PART_DECL(F);

}  // namespace sfno

#define SFNO_FFT_LON_CASE(N_, A_, B_, C_)                                                                                    \
    case N_:                                                                                                                  \
        return grid_dtype == SFNO_DTYPE_BF16 ? go_fast<N_, A_, B_, C_, true>(inverse, p, in, in2, out, rows, nlat, mmax, ld, lat_stats, kept, width, s) \
                                             : go_fast<N_, A_, B_, C_, false>(inverse, p, in, in2, out, rows, nlat, mmax, ld, lat_stats, kept, width, s);
#define SFNO_FFT_LAT_CASE(N_, A_, B_, C_)                                                                                     \
    case N_:                                                                                                                  \
        if constexpr (N_ <= kLatMax) return go_lat<N_, A_, B_, C_>(inverse, p, in, out, mmax, lmax, ld, mscale, s);           \
        break;
#define SFNO_FFT_ROWS_CASE(N_, A_, B_, C_) \
    case N_: return go_rows<N_, A_, B_, C_>(inverse, p, in, out, rows, nlat, mmax, cs, s);
#define SFNO_FFT_COLS_CASE(N_, A_, B_, C_)                                                                                    \
    case N_:                                                                                                                  \
        if constexpr (N_ <= kLatMax) return go_cols<N_, A_, B_, C_>(inverse, p, in, out, rows, mmax, lmax, mscale, s); \
        break;
// the definition of one part: instantiates every kernel of its lengths
#define SFNO_FFT_PART(P, LENGTHS)                                                                                             \
    namespace sfno {                                                                                                          \
    int fft_part_lon_##P(bool inverse, const FftPlan& p, const void* in, const void* in2, void* out, int64_t rows, int nlat, int mmax, int ld, \
                        int grid_dtype, hipStream_t s, float2* lat_stats, const int* kept, int width) {                                                                   \
        switch (p.n) { LENGTHS(SFNO_FFT_LON_CASE) }                                                                           \
        return SFNO_EUNSUPPORTED;                                                                                             \
    }                                                                                                                         \
    int fft_part_lat_##P(bool inverse, const FftPlan& p, const float* in, float* out, int mmax, int lmax, int ld, const float* mscale, hipStream_t s) { \
        switch (p.n) { LENGTHS(SFNO_FFT_LAT_CASE) }                                                                           \
        return SFNO_EUNSUPPORTED;                                                                                             \
    }                                                                                                                         \
    int fft_part_rows_##P(bool inverse, const FftPlan& p, const float* in, float* out, int64_t rows, int nlat, int mmax, int cs, hipStream_t s) { \
        switch (p.n) { LENGTHS(SFNO_FFT_ROWS_CASE) }                                                                          \
        return SFNO_EUNSUPPORTED;                                                                                             \
    }                                                                                                                         \
    int fft_part_cols_##P(bool inverse, const FftPlan& p, const float2* in, float2* out, int64_t rows, int mmax, int lmax, \
                          const float* mscale, hipStream_t s) {                                                               \
        switch (p.n) { LENGTHS(SFNO_FFT_COLS_CASE) }                                                                          \
        return SFNO_EUNSUPPORTED;                                                                                             \
    }                                                                                                                         \
    }
