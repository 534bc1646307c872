// Per-degree power of spherical harmonic coefficients held in the spectral layout float [mmax][lmax][ld]
// ((re, im) of channel row r at 2r, 2r+1; only entries with l >= m exist):
//     power[r][l] = |c[r,l,0]|^2 + 2 sum_{0 < m <= min(l, mmax-1)} |c[r,l,m]|^2
// This is what GeometricH1Loss reduces its transform output to before weighting the degrees with l(l+1)
// (makani/utils/losses.py:301-305 and 320-331), computed here straight from the output of the Legendre analysis,
// without the pass to the reference coefficient layout.  The gradient kernel writes the spectral-layout cotangent
// the adjoint analysis consumes.  Both are bound by the one pass over the coefficients.
#include "sfno_internal.h"

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

// grid (lmax, ceil(rows / 2 / DP_NX)), block DP_THREADS
__global__ __launch_bounds__(DP_THREADS) void degree_power_kernel(const float* __restrict__ spec, float* __restrict__ power, int64_t rows, int lmax,
                                                                  int mmax, int ld) {
    __shared__ float2 part[DP_NY][DP_NX];
    const DpThread t = dp_thread((rows + 1) / 2, lmax, mmax);
    float2 acc = make_float2(0.f, 0.f);
    if (t.on) {
        const float* c0 = spec + (int64_t)t.l * ld + 4 * t.pair;
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

// gspec[m][l][2r..2r+1] = w_m * 2 * gpower[r][l] * c[r,l,m]  (w_0 = 1, w_m = 2 otherwise); padding columns zero
// grid (lmax, ceil(ld / 4 / DP_NX)), block DP_THREADS
__global__ __launch_bounds__(DP_THREADS) void degree_power_grad_kernel(const float* __restrict__ spec, const float* __restrict__ gpower,
                                                                       float* __restrict__ gspec, int64_t rows, int lmax, int mmax, int ld) {
    const DpThread t = dp_thread(ld / 4, lmax, mmax);
    if (!t.on) return;
    const int64_t r = 2 * t.pair;
    const bool has0 = r < rows, has1 = r + 1 < rows;
    const float g0 = has0 ? 2.f * gpower[r * lmax + t.l] : 0.f, g1 = has1 ? 2.f * gpower[(r + 1) * lmax + t.l] : 0.f;
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

}  // namespace

// (sfno_spectral_ld makes ld a multiple of 4: whole 16-byte pieces)
int degree_power_launch(const float* spec, float* power, int64_t rows, int lmax, int mmax, int ld, hipStream_t s) {
    const int64_t blocks = ((rows + 1) / 2 + DP_NX - 1) / DP_NX;
    if (rows < 1 || lmax < 1 || mmax < 1 || ld < 2 * rows || ld % 4 != 0 || blocks > 65535) return SFNO_EINVAL;
    hipLaunchKernelGGL(degree_power_kernel, dim3(lmax, (unsigned)blocks), dim3(DP_THREADS), 0, s, spec, power, rows, lmax, mmax, ld);
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

int degree_power_grad_launch(const float* spec, const float* gpower, float* gspec, int64_t rows, int lmax, int mmax, int ld, hipStream_t s) {
    const int64_t blocks = (ld / 4 + DP_NX - 1) / DP_NX;
    if (rows < 1 || lmax < 1 || mmax < 1 || ld < 2 * rows || ld % 4 != 0 || blocks > 65535) return SFNO_EINVAL;
    hipLaunchKernelGGL(degree_power_grad_kernel, dim3(lmax, (unsigned)blocks), dim3(DP_THREADS), 0, s, spec, gpower, gspec, rows, lmax, mmax, ld);
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

}  // namespace sfno
