// Per-degree power of spherical harmonic coefficients held in the spectral layout float [mmax][lmax][ld]
// ((re, im) of channel row r at 2r, 2r+1; only entries with l >= m exist):
//     power[r][l] = |c[r,l,0]|^2 + 2 sum_{0 < m <= min(l, mmax-1)} |c[r,l,m]|^2
// This is what GeometricH1Loss reduces its transform output to before weighting the degrees with l(l+1)
// (makani/utils/losses.py:301-305 and 320-331), computed here straight from the output of the Legendre analysis,
// without the pass to the reference coefficient layout.  The gradient kernel writes the spectral-layout cotangent
// the adjoint analysis consumes.  Both are bound by the one pass over the coefficients.
#include "sfno_internal.h"

#include <algorithm>

namespace sfno {
namespace {

// A workgroup owns one degree (the longest first) and up to 128 channel rows: nx threads side by side along the row of coefficients,
// two rows (16 bytes) each, and as many of those as fit along the orders, each with several loads in flight.  One 8-byte load at a time by
// four order groups of 64 rows left the 73-row transform at 721 x 1440 waiting on latency, a second workgroup with 9 of 64 lanes busy:
// 78 us per power and 117 us per gradient for 152 MB of coefficients; now 35 (4.4 TB/s) and 69 (read and written, 4.4 TB/s).
constexpr int DP_THREADS = 512;
constexpr int DP_NX = 64;     // pairs of rows per workgroup
constexpr int DP_NY = 32;     // orders in parallel

struct DpThread {
    int l, mtop, ny, tx, ty;
    int64_t pair;
    bool on;
};
// pairs = number of 16-byte pieces of a row of coefficients that are to be covered
__device__ __forceinline__ DpThread dp_thread(int64_t pairs, int lmax, int mmax) {
    DpThread t;
    t.l = lmax - 1 - (int)blockIdx.x;
    t.mtop = min(t.l, mmax - 1);
    const int nx = (int)min((int64_t)DP_NX, pairs);
    t.ny = min(DP_NY, DP_THREADS / nx);
    t.ty = (int)threadIdx.x / nx;
    t.tx = (int)threadIdx.x - t.ty * nx;
    t.pair = (int64_t)blockIdx.y * DP_NX + t.tx;
    t.on = t.ty < t.ny && t.pair < pairs;
    return t;
}

// grid (lmax, ceil(rows / 2 / DP_NX), sets of rows), block DP_THREADS; the second set's powers follow the first's
__global__ __launch_bounds__(DP_THREADS) void degree_power_kernel(const float* __restrict__ spec, const float* __restrict__ spec2, float* __restrict__ power,
                                                                  int64_t rows, int lmax, int mmax, int ld) {
    __shared__ float2 part[DP_NY][DP_NX];
    const DpThread t = dp_thread((rows + 1) / 2, lmax, mmax);
    float2 acc = make_float2(0.f, 0.f);
    if (blockIdx.z) power += rows * lmax;
    if (t.on) {
        const float* c0 = (blockIdx.z ? spec2 : spec) + (int64_t)t.l * ld + 4 * t.pair;
#pragma unroll 4
        for (int m = t.ty; m <= t.mtop; m += t.ny) {
            const float4 c = *reinterpret_cast<const float4*>(c0 + (int64_t)m * lmax * ld);
            const float w = m == 0 ? 1.f : 2.f;
            acc.x = fmaf(w, fmaf(c.x, c.x, c.y * c.y), acc.x);
            acc.y = fmaf(w, fmaf(c.z, c.z, c.w * c.w), acc.y);
        }
        part[t.ty][t.tx] = acc;
    }
    __syncthreads();
    if (t.ty == 0 && t.on) {
        for (int j = 1; j < t.ny; ++j) {
            acc.x += part[j][t.tx].x;
            acc.y += part[j][t.tx].y;
        }
        power[2 * t.pair * lmax + t.l] = acc.x;
        if (2 * t.pair + 1 < rows) power[(2 * t.pair + 1) * lmax + t.l] = acc.y;
    }
}

// cotangent of the power of row r at degree l: given as a tensor ...
struct PowerGrad {
    const float* gpower;
    int lmax;
    __device__ __forceinline__ float operator()(int64_t r, int l) const { return gpower[r * lmax + l]; }
};
// ... or that of the norms of degree_norm_kernel
struct NormGrad {
    const float *weights, *gnorms;
    const float2* sums;
    int64_t channels;
    float alpha;
    int squared;
    __device__ __forceinline__ float operator()(int64_t r, int l) const {
        const int b = (int)(r / channels);
        const float g = gnorms[b], a = alpha * g, h = (1.f - alpha) * g;
        const float2 s = sums[b];
        return squared ? fmaf(h, weights[l], a) : fmaf(h / (2.f * sqrtf(s.y)), weights[l], a / (2.f * sqrtf(s.x)));
    }
};

// gspec[m][l][2r..2r+1] = w_m * 2 * g(r, l) * c[r,l,m]  (w_0 = 1, w_m = 2 otherwise); padding columns zero
// grid (lmax, ceil(ld / 4 / DP_NX)), block DP_THREADS
template <class Grad>
__global__ __launch_bounds__(DP_THREADS) void degree_power_grad_kernel(const float* __restrict__ spec, Grad gpower, float* __restrict__ gspec, int64_t rows,
                                                                       int lmax, int mmax, int ld) {
    const DpThread t = dp_thread(ld / 4, lmax, mmax);
    if (!t.on) return;
    const int64_t r = 2 * t.pair;
    const bool has0 = r < rows, has1 = r + 1 < rows;
    const float g0 = has0 ? 2.f * gpower(r, t.l) : 0.f, g1 = has1 ? 2.f * gpower(r + 1, t.l) : 0.f;
    const int64_t at = (int64_t)t.l * ld + 4 * t.pair;
#pragma unroll 4
    for (int m = t.ty; m <= t.mtop; m += t.ny) {
        const int64_t i = at + (int64_t)m * lmax * ld;
        float4 c = *reinterpret_cast<const float4*>(spec + i);
        const float w = m == 0 ? 1.f : 2.f;
        c.x = has0 ? w * g0 * c.x : 0.f;           // (a padding column may hold anything)
        c.y = has0 ? w * g0 * c.y : 0.f;
        c.z = has1 ? w * g1 * c.z : 0.f;
        c.w = has1 ? w * g1 * c.w : 0.f;
        *reinterpret_cast<float4*>(gspec + i) = c;
    }
}

// Sums of an example's powers, plain and weighted by degree, in double precision: one workgroup per segment of the example's channels * lmax
// values (grid (batch, segments): only a grid's first side may pass 65535); a single one also forms the norm.  With a second kernel where there
// are several, this takes the place of nine elementwise and reduction kernels of 4 to 10 us (73 x 721 values).
constexpr int DN_THREADS = 512;
__device__ __forceinline__ void norm_of(double a, double h, float alpha, int squared, float2* sums, float* norm) {
    const float2 s = make_float2((float)a, (float)h);
    *sums = s;
    *norm = squared ? alpha * s.x + (1.f - alpha) * s.y : alpha * sqrtf(s.x) + (1.f - alpha) * sqrtf(s.y);
}

// norms of one batch, or of two
struct NormOut {
    float *first, *second;
    int batch;
    __device__ __forceinline__ float* at(int b) const { return b < batch ? first + b : second + (b - batch); }
};

__global__ __launch_bounds__(DN_THREADS) void degree_norm_kernel(const float* __restrict__ power, const float* __restrict__ weights,
                                                                 double2* __restrict__ partial, float2* __restrict__ sums, NormOut norms, int64_t n,
                                                                 int lmax, float alpha, int squared) {
    const int b = blockIdx.x, nseg = gridDim.y;
    const int64_t from = n * blockIdx.y / nseg, to = n * (blockIdx.y + 1) / nseg;
    const float* __restrict__ p = power + (int64_t)b * n;
    double a = 0.0, h = 0.0;
    int l = (int)((from + threadIdx.x) % lmax);
    const int step = DN_THREADS % lmax;
#pragma unroll 4
    for (int64_t i = from + threadIdx.x; i < to; i += DN_THREADS) {
        const double v = p[i];
        a += v;
        h += v * (double)weights[l];
        l += step;
        if (l >= lmax) l -= lmax;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_down(a, off, 64);
        h += __shfl_down(h, off, 64);
    }
    __shared__ double2 red[DN_THREADS / 64];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = make_double2(a, h);
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < DN_THREADS / 64; ++w) {
            a += red[w].x;
            h += red[w].y;
        }
        if (nseg == 1)
            norm_of(a, h, alpha, squared, sums + b, norms.at(b));
        else
            partial[(int64_t)b * nseg + blockIdx.y] = make_double2(a, h);
    }
}

// one wavefront per example; nseg <= 64
__global__ __launch_bounds__(64) void degree_norm_finish_kernel(const double2* __restrict__ partial, float2* __restrict__ sums, NormOut norms, int nseg,
                                                                float alpha, int squared) {
    const int b = blockIdx.x;
    double2 t = make_double2(0.0, 0.0);
    if ((int)threadIdx.x < nseg) t = partial[(int64_t)b * nseg + threadIdx.x];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        t.x += __shfl_down(t.x, off, 64);
        t.y += __shfl_down(t.y, off, 64);
    }
    if (threadIdx.x == 0) norm_of(t.x, t.y, alpha, squared, sums + b, norms.at(b));
}

}  // namespace

// (sfno_spectral_ld makes ld a multiple of 4: whole 16-byte pieces)
int degree_power_launch(const float* spec, const float* spec2, float* power, int64_t rows, int lmax, int mmax, int ld, hipStream_t s) {
    const int64_t blocks = ((rows + 1) / 2 + DP_NX - 1) / DP_NX;
    if (rows < 1 || lmax < 1 || mmax < 1 || ld < 2 * rows || ld % 4 != 0 || blocks > 65535) return SFNO_EINVAL;
    hipLaunchKernelGGL(degree_power_kernel, dim3(lmax, (unsigned)blocks, spec2 ? 2 : 1), dim3(DP_THREADS), 0, s, spec, spec2, power, rows, lmax, mmax, ld);
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

int degree_power_grad_launch(const float* spec, const float* gpower, float* gspec, int64_t rows, int lmax, int mmax, int ld, hipStream_t s) {
    const int64_t blocks = (ld / 4 + DP_NX - 1) / DP_NX;
    if (rows < 1 || lmax < 1 || mmax < 1 || ld < 2 * rows || ld % 4 != 0 || blocks > 65535) return SFNO_EINVAL;
    hipLaunchKernelGGL(degree_power_grad_kernel<PowerGrad>, dim3(lmax, (unsigned)blocks), dim3(DP_THREADS), 0, s, spec, PowerGrad{gpower, lmax}, gspec, rows, lmax,
                       mmax, ld);
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

// some 8 thousand values per workgroup; by an example's size alone, so that it gives the same norm alone and in a batch
int degree_norm_segments(int64_t channels, int lmax) { return (int)std::max<int64_t>(1, std::min<int64_t>(channels * lmax / 8192, 64)); }

int degree_norm_launch(const float* power, const float* weights, double2* partial, float2* sums, float* norms, float* norms2, int batch, int64_t channels,
                       int lmax, float alpha, int squared, hipStream_t s) {
    if (batch < 1 || channels < 1 || lmax < 1) return SFNO_EINVAL;
    const int nseg = degree_norm_segments(channels, lmax);
    const NormOut out{norms, norms2, batch};
    const unsigned n = norms2 ? 2u * batch : batch;
    hipLaunchKernelGGL(degree_norm_kernel, dim3(n, nseg), dim3(DN_THREADS), 0, s, power, weights, partial, sums, out, channels * lmax, lmax, alpha, squared);
    if (nseg > 1) hipLaunchKernelGGL(degree_norm_finish_kernel, dim3(n), dim3(64), 0, s, partial, sums, out, nseg, alpha, squared);
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

int degree_norm_grad_launch(const float* spec, const float* weights, const float2* sums, const float* gnorms, float* gspec, int batch, int64_t channels, int lmax,
                            int mmax, int ld, float alpha, int squared, hipStream_t s) {
    const int64_t rows = batch * channels, blocks = (ld / 4 + DP_NX - 1) / DP_NX;
    if (batch < 1 || channels < 1 || lmax < 1 || mmax < 1 || ld < 2 * rows || ld % 4 != 0 || blocks > 65535) return SFNO_EINVAL;
    hipLaunchKernelGGL(degree_power_grad_kernel<NormGrad>, dim3(lmax, (unsigned)blocks), dim3(DP_THREADS), 0, s, spec,
                       NormGrad{weights, gnorms, sums, channels, alpha, squared}, gspec, rows, lmax, mmax, ld);
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

}  // namespace sfno
