// Plans and dispatch of the specialised FFTs (fft_kernels.h); the kernels of each length live in fft_fast_*.hip.
#include "fft_fast.h"

#include <algorithm>
#include <cmath>
#include <vector>

#include "fft_kernels.h"
#include "fft_lengths.h"

namespace sfno {

namespace {

struct FastEntry {
    int n, r0, r1, r2;
};
#define SFNO_FFT_ENTRY(N_, A_, B_, C_) {N_, A_, B_, C_},
const FastEntry kFast[] = {SFNO_FFT_LENGTHS(SFNO_FFT_ENTRY)};
#undef SFNO_FFT_ENTRY

const FastEntry* find_fast(int n) {
    for (const auto& e : kFast)
        if (e.n == n) return &e;
    return nullptr;
}

// inter-pass twiddles of the specialised passes of length f.n
int upload_pass_twiddles(const FastEntry& f, FftPlan& p) {
    const int N = f.n, nb = N / f.r0;
    // (one slab per factor index, see fft_kernels.h)
    std::vector<float2> tw0((size_t)std::max(1, (f.r0 - 1) * nb), make_float2(1.f, 0.f)), tw1((size_t)std::max(1, (f.r1 - 1) * f.r2), make_float2(1.f, 0.f));
    for (int k0 = 1; k0 < f.r0; ++k0)
        for (int j = 0; j < nb; ++j) {
            double a = -kTwoPi * (double)(((int64_t)k0 * j) % N) / (double)N;
            tw0[(size_t)(k0 - 1) * nb + j] = make_float2((float)std::cos(a), (float)std::sin(a));
        }
    for (int k1 = 1; k1 < f.r1; ++k1)
        for (int n2 = 0; n2 < f.r2; ++n2) {
            double a = -kTwoPi * (double)(((int64_t)f.r0 * k1 * n2) % N) / (double)N;
            tw1[(size_t)(k1 - 1) * f.r2 + n2] = make_float2((float)std::cos(a), (float)std::sin(a));
        }
    // slots of bin m and of bin N - m after the decimation-in-frequency passes (= before the decimation-in-time passes)
    std::vector<unsigned> post((size_t)N / 2 + 1);
    auto slot = [&](int m) {
        const int k0 = m % f.r0, t = m / f.r0, k1 = t % f.r1, k2 = t / f.r1;
        return (unsigned)(k0 * (f.r1 * f.r2) + k1 * f.r2 + k2);
    };
    for (int m = 0; m <= N / 2; ++m) post[m] = slot(m) | (slot((N - m) % N) << 16);
    if (hipMalloc(&p.d_post, sizeof(unsigned) * post.size()) != hipSuccess) return SFNO_ENOMEM;
    if (hipMemcpy(p.d_post, post.data(), sizeof(unsigned) * post.size(), hipMemcpyHostToDevice) != hipSuccess) return SFNO_EHIP;
    if (hipMalloc(&p.d_tw0, sizeof(float2) * tw0.size()) != hipSuccess) return SFNO_ENOMEM;
    if (hipMalloc(&p.d_tw1, sizeof(float2) * tw1.size()) != hipSuccess) return SFNO_ENOMEM;
    if (hipMemcpy(p.d_tw0, tw0.data(), sizeof(float2) * tw0.size(), hipMemcpyHostToDevice) != hipSuccess) return SFNO_EHIP;
    if (hipMemcpy(p.d_tw1, tw1.data(), sizeof(float2) * tw1.size(), hipMemcpyHostToDevice) != hipSuccess) return SFNO_EHIP;
    return SFNO_OK;
}

int largest_prime_factor(int n) {
    int best = 1;
    for (int q = 2; (int64_t)q * q <= n; ++q)
        while (n % q == 0) { best = q; n /= q; }
    return n > 1 ? n : best;
}

}  // namespace

bool fft_fast_supported(int n) { return find_fast(n) != nullptr; }

int fft_chirp_plan_init(FftPlan& p) {
    const int n = p.n;
    if (find_fast(n) || largest_prime_factor(n) <= 7) return SFNO_OK;      // the plain passes serve these lengths well
    const int M = 2 * n - 1 <= 512 ? 512 : 2 * n - 1 <= 1536 ? 1536 : 0;
    if (!M) return SFNO_OK;
    const FastEntry* f = find_fast(M);
    // chirp c[k] = exp(-i pi k^2 / n), the angle reduced exactly in integers
    std::vector<double> cr(n), ci(n);
    std::vector<float2> chirp(M, make_float2(0.f, 0.f));
    for (int k = 0; k < n; ++k) {
        const double a = -(kTwoPi / 2) * (double)(((int64_t)k * k) % (2 * (int64_t)n)) / (double)n;
        cr[k] = std::cos(a);
        ci[k] = std::sin(a);
        chirp[k] = make_float2((float)cr[k], (float)ci[k]);
    }
    // v = conj(c) wrapped around M (v[M - k] = v[k]); its transform, real-symmetric input pairs folded:
    // V[q] = v[0] + sum_{k=1}^{n-1} v[k] 2 cos(2 pi q k / M)
    std::vector<float2> vhat(M);
    std::vector<double> cosM(M);
    for (int j = 0; j < M; ++j) cosM[j] = std::cos(kTwoPi * (double)j / (double)M);
    const int r0 = f->r0, r1 = f->r1, r2 = f->r2;
    for (int q = 0; q < M; ++q) {
        double sr = cr[0], si = -ci[0];
        for (int k = 1; k < n; ++k) {
            const double w = 2.0 * cosM[(int)(((int64_t)q * k) % M)];
            sr += cr[k] * w;
            si -= ci[k] * w;
        }
        const int k0 = q % r0, t = q / r0, k1 = t % r1, k2 = t / r1;        // slot of bin q after the decimation-in-frequency passes
        vhat[k0 * (r1 * r2) + k1 * r2 + k2] = make_float2((float)(sr / M), (float)(si / M));
    }
    int rc = upload_pass_twiddles(*f, p);
    if (rc != SFNO_OK) return rc;
    if (hipMalloc(&p.d_chirp, sizeof(float2) * M) != hipSuccess || hipMalloc(&p.d_vhat, sizeof(float2) * M) != hipSuccess) return SFNO_ENOMEM;
    if (hipMemcpy(p.d_chirp, chirp.data(), sizeof(float2) * M, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(p.d_vhat, vhat.data(), sizeof(float2) * M, hipMemcpyHostToDevice) != hipSuccess)
        return SFNO_EHIP;
    p.chirp_m = M;
    return SFNO_OK;
}

int latfft_fast_launch(bool inverse, const FftPlan& p, const float* in, float* out, int mmax, int lmax, int ld, const float* mscale, hipStream_t s) {
    if (p.chirp_m == 1536) return go_chirp<1536, 16, 12, 8>(inverse, p, in, out, mmax, lmax, ld, mscale, s);
    if (p.chirp_m == 512) return go_chirp<512, 8, 8, 8>(inverse, p, in, out, mmax, lmax, ld, mscale, s);
    for (auto part : {fft_part_lat_A, fft_part_lat_B, fft_part_lat_C, fft_part_lat_D, fft_part_lat_E, fft_part_lat_F}) {
        const int rc = part(inverse, p, in, out, mmax, lmax, ld, mscale, s);
        if (rc != SFNO_EUNSUPPORTED) return rc;
    }
    return SFNO_EUNSUPPORTED;
}

int fft_col_shift(int n) { return n <= kLatMax && find_fast(n) ? col_shift(n) : 0; }

int fft_rows_launch(bool inverse, const FftPlan& p, const float* in, float* out, int64_t rows, int nlat, int mmax, int cs, hipStream_t s) {
    for (auto part : {fft_part_rows_A, fft_part_rows_B, fft_part_rows_C, fft_part_rows_D, fft_part_rows_E, fft_part_rows_F}) {
        const int rc = part(inverse, p, in, out, rows, nlat, mmax, cs, s);
        if (rc != SFNO_EUNSUPPORTED) return rc;
    }
    return SFNO_EUNSUPPORTED;
}

int fft_cols_launch(bool inverse, const FftPlan& p, const float2* in, float2* out, int64_t rows, int mmax, int lmax, const float* mscale,
                    hipStream_t s) {
    if (lmax < 1 || lmax > p.n || mmax < 1 || !mscale) return SFNO_EINVAL;
    for (auto part : {fft_part_cols_A, fft_part_cols_B, fft_part_cols_C, fft_part_cols_D, fft_part_cols_E, fft_part_cols_F}) {
        const int rc = part(inverse, p, in, out, rows, mmax, lmax, mscale, s);
        if (rc != SFNO_EUNSUPPORTED) return rc;
    }
    return SFNO_EUNSUPPORTED;
}

int fft_fast_plan_init(FftPlan& p) {
    const FastEntry* f = find_fast(p.n);
    return f ? upload_pass_twiddles(*f, p) : SFNO_OK;
}

int fft_fast_launch(bool inverse, const FftPlan& p, const void* in, void* out, int64_t rows, int nlat, int mmax, int ld, int grid_dtype,
                    hipStream_t s, float2* lat_stats, const void* in2, const int* kept, int width) {
    if (grid_dtype != SFNO_DTYPE_BF16 && grid_dtype != SFNO_DTYPE_F32) return SFNO_EUNSUPPORTED;
    if ((lat_stats && !inverse) || (in2 && inverse) || (width && !in2)) return SFNO_EINVAL;
    for (auto part : {fft_part_lon_A, fft_part_lon_B, fft_part_lon_C, fft_part_lon_D, fft_part_lon_E, fft_part_lon_F}) {
        const int rc = part(inverse, p, in, in2, out, rows, nlat, mmax, ld, grid_dtype, s, lat_stats, kept, width);
        if (rc != SFNO_EUNSUPPORTED) return rc;
    }
    return SFNO_EUNSUPPORTED;
}

}  // namespace sfno
