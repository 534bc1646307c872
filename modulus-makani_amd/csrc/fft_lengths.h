// Transform lengths with specialised kernels (fft_kernels.h): X(length, R0, R1, R2), grouped by the source file that
// instantiates them (fft_fast_*.hip).  The grids they serve: 5 to 0.25 degrees (72 ... 1440), powers of two, the reduced Gaussian
// grids (160, 320, 640, 1280) and what scale factors make of those.
//
// Choice of the radices: few passes of radix <= 16 (two below 200 points), an odd last radix where there is one -- the last pass
// walks groups of that many complex numbers, and an even stride puts a wavefront's groups on half of the LDS banks or fewer --
// and among those the order with the fewest LDS cycles over the passes and the Hermitian step (counted with the bank of
// every address of every wavefront: 180 as 12 * 15 takes 60 cycles per sequence where 4 * 5 * 9 took 90, 240 as 16 * 15
// 82 against 111 for 16 * 5 * 3).
#pragma once
#define SFNO_FFT_LENGTHS_A(X) X(1536, 16, 12, 8) X(1440, 16, 10, 9) X(1280, 16, 8, 10) X(1200, 16, 5, 15)
#define SFNO_FFT_LENGTHS_B(X) X(1152, 16, 8, 9) X(1024, 16, 8, 8) X(960, 8, 8, 15) X(800, 16, 10, 5) X(768, 16, 8, 6)
#define SFNO_FFT_LENGTHS_C(X) X(720, 16, 5, 9) X(640, 16, 8, 5) X(600, 5, 8, 15) X(576, 8, 8, 9) X(512, 8, 8, 8)
#define SFNO_FFT_LENGTHS_D(X) X(480, 4, 8, 15) X(400, 10, 8, 5) X(384, 16, 8, 3) X(360, 8, 5, 9) X(320, 8, 8, 5) X(288, 4, 8, 9)
#define SFNO_FFT_LENGTHS_E(X) \
    X(256, 16, 16, 1) X(240, 16, 15, 1) X(200, 5, 8, 5) X(192, 16, 12, 1) X(180, 12, 15, 1) X(160, 4, 8, 5) X(144, 16, 9, 1) X(128, 8, 16, 1)
#define SFNO_FFT_LENGTHS_F(X) \
    X(120, 8, 15, 1) X(100, 10, 10, 1) X(96, 8, 12, 1) X(80, 16, 5, 1) X(72, 8, 9, 1) X(64, 8, 8, 1) X(60, 4, 15, 1) X(48, 16, 3, 1) X(40, 8, 5, 1) \
        X(36, 4, 9, 1) X(32, 4, 8, 1) X(24, 8, 3, 1) X(20, 4, 5, 1) X(16, 4, 4, 1) X(12, 4, 3, 1) X(8, 4, 2, 1)
#define SFNO_FFT_LENGTHS(X) \
    SFNO_FFT_LENGTHS_A(X) SFNO_FFT_LENGTHS_B(X) SFNO_FFT_LENGTHS_C(X) SFNO_FFT_LENGTHS_D(X) SFNO_FFT_LENGTHS_E(X) SFNO_FFT_LENGTHS_F(X)
