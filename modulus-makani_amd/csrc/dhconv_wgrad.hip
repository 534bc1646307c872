// Gradient of the dhconv contraction with respect to its weight:
//     gw[i][o][l] = sum over rows (m, b) of conj(x[m,b][i]) * g[m,b][o]
// (the backward of einsum("bixy,iox->boxy") at makani/models/common/contractions.py:130-136 with
// respect to `bc`).  Per degree l this is four real GEMMs whose K dimension is the rows of the spectral layout,
//     Re gw = Xr^T Gr + Xi^T Gi,      Im gw = Xr^T Gi - Xi^T Gr,
// with fp32 accuracy from the bf16 matrix pipe: every value is cut exactly into three bf16 numbers, each the rounded remainder
// of those before it (8 + 8 + 8 significant bits), and x g is the six partial products x0 g0 + x0 g1 + x1 g0 + x0 g2 + x1 g1 +
// x2 g0, each exact, into the fp32 accumulator.  What is left out is below 2^-23 |x g| for every single product: the cut has
// no scale, so rows whose magnitudes differ by any power of two keep their bits.  (Two fp16 numbers per value under a scale
// per channel and 16 rows need half the matrix instructions, but keep a product only as far as its operands lie
// near the largest of their rows: with x rising and g falling by 2^22 within 16 rows, so that all products count alike, the error
// against float64 is 1e-5.)  The parts of an infinite value are no sum of it: a row that holds one gives NaN.
//
// Operands.  v_mfma_f32_32x32x16_bf16 wants, per lane, 8 consecutive k of one channel.  Rows are K here, so a lane that loads the
// (re, im) pair of its channel from 8 rows holds its fragment without any transpose: lanes 0-31 take rows 0-7 of a chunk
// of 16, lanes 32-63 rows 8-15, each load is 256 contiguous bytes per half.
//
// A workgroup is 8 wavefronts = the 8 degrees that share 64-byte lines of gw ([i][o][l], l fastest),
// all on the same tile of (i, o).  The results meet in LDS and leave as whole lines.
//
// What bounds it: per chunk and 64 x 64 tile a wavefront issues 96 matrix instructions (3072 cycles) and about 400 vector
// instructions, most of them cutting the 64 values it loaded, on a SIMD shared by two wavefronts; the store of gw (283 MB for
// 384 x 384 x 240) follows the sums.  384 x 384 channels, 240 degrees: 231 / 430 / 765 us for 1 / 2 / 4 samples (on
// v_mfma_f32_32x32x2_f32, 512 matrix cycles per 16 rows and product instead of 192: 387 / 689 / 1322; two fp16 numbers, 96 cycles:
// 191 / 338 / 578), 241 degrees, whose lines of gw are partial, 390 for one sample (416; 354).  Error against float64 of operands of
// one magnitude, 1080 rows: 7.2e-7 (fp32 instruction 8.3e-7), and the same where they differ.
#include <algorithm>

#include "sfno_internal.h"

namespace sfno {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u4 __attribute__((ext_vector_type(4)));

constexpr int WG_DEG = 8;            // degrees (wavefronts) per workgroup
constexpr int WG_KC = 16;            // rows per chunk: one matrix K step
constexpr int WG_PITCH = WG_DEG + 1; // float2 per staged line of gw; odd so that the 32 lanes of a store hit 32 banks pairs

// rounds a pair of numbers to bf16 (packed) and leaves what that lost
__device__ __forceinline__ unsigned take_bf16(float& a, float& b) {
    const unsigned h = __builtin_bit_cast(unsigned, __builtin_convertvector(f2{a, b}, bf16x2));
    a -= __uint_as_float(h << 16);
    b -= __uint_as_float(h & 0xffff0000u);
    return h;
}

// gw is written once and read by another kernel: past the caches, which the rows of X and G need
__device__ __forceinline__ void store_line(float2* p, float2 z) {
    __builtin_nontemporal_store(__builtin_bit_cast(double, z), reinterpret_cast<double*>(p));
}

struct Planes {                      // a channel's 8 rows: real and imaginary part, in three bf16 numbers each
    u4 r[3], i[3];
};

// IB, OB: 32-channel blocks of i and o per workgroup: 2 x 2, or 1 x 1 (half of the registers and LDS) where those leave CUs idle
// OFF: type of a lane's byte offset within a row chunk (64 bits only where 16 row strides do not fit 32)
template <int IB, int OB, typename OFF>
__global__ __launch_bounds__(64 * WG_DEG, OB == 1 && sizeof(OFF) == 4 ? 4 : 2) void dhconv_wgrad_kernel(DhconvWgradArgs p, int ni, int no, int split) {
    constexpr int WG_TI = 32 * IB, WG_TO = 32 * OB;      // channels per workgroup
    __shared__ float2 stage[32 * WG_TO * WG_PITCH];

    // Workgroups are dealt to the 8 XCDs round-robin by linear id.  A unit is the tiles of one group of 8 degrees, or (split = 2) of its upper or
    // lower half of the input channels; its tiles run as neighbours in one XCD's queue, where they share the rows of X and G in
    // that XCD's L2.  The units go to the XCDs highest degrees (most rows) first, in alternating direction round by round: the
    // work of a group grows linearly with its degree, and dealing every round in the same direction would give the first XCD a
    // quarter more rows than the average.
    const int xcd = blockIdx.x & 7, tiles = ni * no;
    int k = (int)(blockIdx.x >> 3) / tiles, t = (int)(blockIdx.x >> 3) - k * tiles;      // turn of dealing, tile in the unit
    int half = 0;
    if (split == 2) {
        // (two turns in a row are one lower and one upper half)
        const int low = ni / 2 * no, first = xcd & 1 ? tiles - low : low;
        half = xcd & 1;
        k *= 2;
        if (t >= first) {
            t -= first;
            half ^= 1;
            ++k;
        }
        if (half) t += low;
    }
    const int u = 8 * k + ((k & 1) ? 7 - xcd : xcd);
    const int lg = (p.L + WG_DEG - 1) / WG_DEG - 1 - (split == 2 ? u >> 1 : u);
    if (lg < 0) return;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int l = lg * WG_DEG + wave;
    const int i0 = (t / no) * WG_TI, o0 = (t % no) * WG_TO;
    const int kg = lane >> 5, jj = lane & 31;

    // a wavefront whose degree does not exist (last group when L is not a multiple of 8) has no rows
    const int nm = l < p.L ? (p.tri ? min(l + 1, p.M) : p.M) : 0;      // orders of this degree: rows (m, b), sample by sample
    const int nch = (nm + WG_KC - 1) / WG_KC;
    const int64_t ms_x = (int64_t)p.L * p.ld_in * 4, ms_g = (int64_t)p.L * p.ld_out * 4;     // bytes from order to order
    const char* __restrict__ X = reinterpret_cast<const char*>(p.X + (int64_t)min(l, p.L - 1) * p.ld_in);
    const char* __restrict__ G = reinterpret_cast<const char*>(p.G + (int64_t)min(l, p.L - 1) * p.ld_out);

    // Rows of a chunk: lanes of half 0 take rows first .. first + 7, half 1 the 8 rows `hr` further on.  A chunk near the end of
    // the buffer starts earlier than its turn so that no load leaves the buffer; rows of the chunk before it, and orders the
    // degree does not have (their memory is unwritten), are zeroed in both operands.
    // A degree of at most 8 orders takes two samples per chunk, the second half the rows of the second one (the last chunk of an odd
    // number starts a sample early): half the additions, whose rounding is what such short sums lose.
    const bool two = nm > 0 && nm <= 8 && p.B > 1;
    const int hr = two ? 0 : p.M >= WG_KC ? 8 : max(p.M - 8, 0);
    OFF offx[IB], offg[OB];          // byte offset of my channel (clamped to the last one) in my half of a chunk
#pragma unroll
    for (int ib = 0; ib < IB; ++ib) offx[ib] = (OFF)(hr * kg) * (OFF)ms_x + (two ? (OFF)(8 * kg) * (OFF)p.I : 0) + 8u * min(i0 + 32 * ib + jj, p.I - 1);
#pragma unroll
    for (int ob = 0; ob < OB; ++ob) offg[ob] = (OFF)(hr * kg) * (OFF)ms_g + (two ? (OFF)(8 * kg) * (OFF)p.O : 0) + 8u * min(o0 + 32 * ob + jj, p.O - 1);

    f32x16 re[IB][OB], im[IB][OB];
#pragma unroll
    for (int ib = 0; ib < IB; ++ib)
#pragma unroll
        for (int ob = 0; ob < OB; ++ob)
#pragma unroll
            for (int v = 0; v < 16; ++v) re[ib][ob][v] = im[ib][ob][v] = 0.f;
    // 8 rows of one channel, each from a wavefront-uniform row address plus a lane offset
    auto load = [&](const char* base, int64_t ms, OFF off, int m0, float2 (&r)[8]) {
        const char* row = base + max(min(m0, p.M - WG_KC), 0) * ms;
        asm("" : "+v"(off));             // (32 bits until it is added: see below)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            uint64_t rj = (uint64_t)(row + min(j, p.M - 1) * ms);
            asm("" : "+s"(rj));      // (keeps the row address scalar: base + lane offset, no vector additions)
            const f2 z = *reinterpret_cast<const __attribute__((address_space(1))) f2*>(reinterpret_cast<const __attribute__((address_space(1))) char*>(rj) + off);
            r[j] = make_float2(z[0], z[1]);
        }
    };
    // zeroes the rows of chunk m0 that do not count (see above); counted: the first half's sample has had its turn
    auto mask = [&](int m0, bool counted, float2 (&r)[8]) {
        const int first = max(min(m0, p.M - WG_KC), 0) + hr * kg;
        const int lo = two ? (!kg && counted ? 8 : 0) : kg && p.M < WG_KC ? 8 : m0;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (first + j < lo || first + j >= nm) r[j] = make_float2(0.f, 0.f);
    };
    auto cut = [&](float2 (&r)[8], Planes& f) {
#pragma unroll
        for (int w = 0; w < 4; ++w)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                f.r[k][w] = take_bf16(r[2 * w].x, r[2 * w + 1].x);
                f.i[k][w] = take_bf16(r[2 * w].y, r[2 * w + 1].y);
            }
    };
    const int64_t nchunks = two ? (p.B + 1) / 2 : (int64_t)nch * p.B;
    if (nchunks > 0) {
        float2 rx[IB][8], rg[OB][8];
        const char *Xb = X, *Gb = G;             // rows of the sample the next loads belong to
        int m0 = 0;
#pragma unroll
        for (int ib = 0; ib < IB; ++ib) {
            load(Xb, ms_x, offx[ib], 0, rx[ib]);
            __builtin_amdgcn_sched_barrier(0);   // (in the order the loop waits for them)
        }
#pragma unroll
        for (int ob = 0; ob < OB; ++ob) {
            load(Gb, ms_g, offg[ob], 0, rg[ob]);
            __builtin_amdgcn_sched_barrier(0);
        }
        for (int64_t c = 0; c < nchunks; ++c) {
            const int mc = m0;
            if (mc + WG_KC > nm || mc > p.M - WG_KC) {
                const bool counted = 2 * c > p.B - 2;
#pragma unroll
                for (int ib = 0; ib < IB; ++ib) mask(mc, counted, rx[ib]);
#pragma unroll
                for (int ob = 0; ob < OB; ++ob) mask(mc, counted, rg[ob]);
            }
            // the next chunk (the last one again after it) is requested into the registers of this one as they come free
            if (c + 1 < nchunks) {
                m0 += WG_KC;
                if (m0 >= nm) {
                    m0 = 0;
                    const int samples = two && 2 * (int)c + 4 <= p.B ? 2 : 1;
                    Xb += 8 * (int64_t)p.I * samples;
                    Gb += 8 * (int64_t)p.O * samples;
                }
            }
            Planes fx[IB];
#pragma unroll
            for (int ib = 0; ib < IB; ++ib) {
                cut(rx[ib], fx[ib]);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int ob = 0; ob < OB; ++ob) {
                Planes fg;
                cut(rg[ob], fg);
                __builtin_amdgcn_sched_barrier(0);
                // part A of x times part B of g; consecutive instructions go to different accumulators
                auto step = [&](int A, int B) {
                    const bf16x8 gr = __builtin_bit_cast(bf16x8, fg.r[B]), gi = __builtin_bit_cast(bf16x8, fg.i[B]);
                    const bf16x8 ng = __builtin_bit_cast(bf16x8, fg.r[B] ^ 0x80008000u);     // -Gr
#pragma unroll
                    for (int ib = 0; ib < IB; ++ib) {
                        const bf16x8 xr = __builtin_bit_cast(bf16x8, fx[ib].r[A]);
                        re[ib][ob] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xr, gr, re[ib][ob], 0, 0, 0);
                        im[ib][ob] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xr, gi, im[ib][ob], 0, 0, 0);
                    }
#pragma unroll
                    for (int ib = 0; ib < IB; ++ib) {
                        const bf16x8 xi = __builtin_bit_cast(bf16x8, fx[ib].i[A]);
                        re[ib][ob] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xi, gi, re[ib][ob], 0, 0, 0);
                        im[ib][ob] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xi, ng, im[ib][ob], 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                };
                // smallest terms first
                step(2, 0);
                step(1, 1);
                step(0, 2);
                step(1, 0);
                // (only now, with parts 1 and 2 of x spent, are there registers for its next rows)
                if (ob == OB - 1) {
#pragma unroll
                    for (int ib = 0; ib < IB; ++ib) load(Xb, ms_x, offx[ib], m0, rx[ib]);
                }
                load(Gb, ms_g, offg[ob], m0, rg[ob]);
                __builtin_amdgcn_sched_barrier(0);
                step(0, 1);
                step(0, 0);
            }
        }
    }

    // The 8 wavefronts hold the same (i, o) tile for 8 consecutive degrees: one block of 32 i at a time they
    // write it to LDS as [i][o][degree], and the workgroup stores it as the 64-byte lines of gw.
    float2* __restrict__ gw = reinterpret_cast<float2*>(p.GW);
#pragma unroll
    for (int ib = 0; ib < IB; ++ib) {
        if (ib) __syncthreads();
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int il = 8 * (v >> 2) + 4 * kg + (v & 3);
#pragma unroll
            for (int ob = 0; ob < OB; ++ob)
                stage[(il * WG_TO + 32 * ob + jj) * WG_PITCH + wave] = make_float2(re[ib][ob][v], im[ib][ob][v]);
        }
        __syncthreads();
        // eight lanes per line, 64 lines per pass
        constexpr int IP = 64 / WG_TO;
        const int d = threadIdx.x & 7, ln = threadIdx.x >> 3, is = ln / WG_TO;
        const int i = i0 + 32 * ib + is, o = o0 + ln % WG_TO, ll = lg * WG_DEG + d;
        const float2* src = stage + ln * WG_PITCH + d;
        float2* dst = gw + ((int64_t)i * p.O + o) * p.L + ll;
        const int64_t istep = (int64_t)IP * p.O * p.L;
        if (o < p.O && ll < p.L) {
            if (i0 + 32 * ib + 32 <= p.I) {
#pragma unroll 8
                for (int k = 0; k < 32 / IP; ++k) store_line(dst + k * istep, src[k * 64 * WG_PITCH]);
            } else {
                for (int k = 0; i + k * IP < p.I && k < 32 / IP; ++k) store_line(dst + k * istep, src[k * 64 * WG_PITCH]);
            }
        }
    }
}

// the fullest XCD's queue, in chunks of rows, of the units of dhconv_wgrad_kernel; a tile's way to its first chunk and its stores take about 2.5
int64_t fullest_queue(const DhconvWgradArgs& a, int ni, int no, int split) {
    const int groups = (a.L + WG_DEG - 1) / WG_DEG;
    int64_t q[8] = {};
    for (int u = 0; u < groups * split; ++u) {
        const int g = u / split, s = u - g * split, top = std::min(WG_DEG * (groups - g), a.tri ? a.M : a.L), rows = a.tri ? top : a.M;
        const int64_t tiles = (int64_t)(ni * (s + 1) / split - ni * s / split) * no;
        q[(u >> 3) & 1 ? 7 - (u & 7) : u & 7] += tiles * (2 * (int64_t)((rows + WG_KC - 1) / WG_KC) * a.B + 5);
    }
    return *std::max_element(q, q + 8);
}

}  // namespace

int dhconv_wgrad_launch(const DhconvWgradArgs& a, hipStream_t s) {
    // a lane's offset in a row chunk: 16 row strides and the channel, in 32 bits
    const int64_t ld = a.ld_in > a.ld_out ? a.ld_in : a.ld_out;
    const bool wide = 64 * (int64_t)a.L * ld + 4 * ld > 0xffffffffLL;
    const int64_t groups = 8 * (((a.L + WG_DEG - 1) / WG_DEG + 7) / 8);
    // 64 x 64 tiles cut and load half as much per product, 32 x 32 tiles need half the registers and LDS (two workgroups per CU, four
    // times as many): 31 against 15 us for 128 x 128 channels and 90 degrees (64 tiles of 64 x 64), 84 against 72 for 384 x 384 and
    // 120 (576 tiles), but 214 against 240 for 384 x 384 and 240 (1152 tiles).  The line: three tiles per CU.
    const int64_t n2 = (int64_t)((a.I + 63) / 64) * ((a.O + 63) / 64);
    const bool narrow = !wide && ((a.I <= 32 && a.O <= 32) || groups * n2 < 768);
    const int tile = narrow ? 32 : 64;
    const int ni = (a.I + tile - 1) / tile, no = (a.O + tile - 1) / tile;
    // Two units per group: as many queues as XCDs where there are few groups (384 x 384 channels, 45 degrees, eight samples 158 -> 107 us; 190 x 190 and 60
    // degrees, two samples, 28 -> 22.5), more shares than an XCD's 32 CUs can take at a time where there are many (36 tiles of 64 x 64 of a group: 240 degrees
    // with 2 samples 425 -> 411, 241 with one 387 -> 353).  One unit, whose tiles share all rows, where they find a place at once: large tiles of 250 shapes, time of
    // two units against one 0.95 for 30 and more of them (the worst 1.03), 0.97 for 5 x 5 with several samples and 1.02 with one, 1.02 for 16 to 28 of them (up to
    // 1.12: 367 -> 248 channels, 204 degrees) unless one XCD's queue is the longer by more than a fifteenth (0.79 to 1).  Small tiles, 770 shapes: 1.01 with less than twelve
    // of them, where the queues are even 1.02 (120 degrees 75.5 against 77), else 0.91 on average, 0.54 at best; 68 lose more than 3 %, one sample of 40 to 64
    // degrees up to 15, which no line drawn by queues, tiles and samples tells from those that gain 25.
    int split = 1;
    if (ni >= 2) {
        const int64_t n = (int64_t)ni * no, one = fullest_queue(a, ni, no, 1), two = fullest_queue(a, ni, no, 2);
        if (narrow ? n >= 12 && 10 * one > 11 * two : n >= 30 || (n >= 25 && ni >= 5 && no >= 5 && a.B > 1) || 14 * one > 15 * two) split = 2;
    }
    const int64_t blocks = groups * ni * no;
    if (blocks > 0x7fffffffLL) return SFNO_EUNSUPPORTED;
    const dim3 grid((unsigned)blocks), block(64 * WG_DEG);
    if (wide)
        hipLaunchKernelGGL((dhconv_wgrad_kernel<2, 2, uint64_t>), grid, block, 0, s, a, ni, no, split);
    else if (narrow)
        hipLaunchKernelGGL((dhconv_wgrad_kernel<1, 1, unsigned>), grid, block, 0, s, a, ni, no, split);
    else
        hipLaunchKernelGGL((dhconv_wgrad_kernel<2, 2, unsigned>), grid, block, 0, s, a, ni, no, split);
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

}  // namespace sfno
