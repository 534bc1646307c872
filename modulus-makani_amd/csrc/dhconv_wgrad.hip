// Gradient of the dhconv contraction with respect to its weight:
//     gw[i][o][l] = sum over rows (m, b) of conj(x[m,b][i]) * g[m,b][o]
// (the backward of einsum("bixy,iox->boxy") at makani/models/common/contractions.py:130-136 with
// respect to `bc`).  Per degree l this is four real GEMMs whose K dimension is the rows of the spectral layout,
//     Re gw = Xr^T Gr + Xi^T Gi,      Im gw = Xr^T Gi - Xi^T Gr,
// with fp32 accuracy from the fp16 matrix pipe: every value, scaled by a power of two below 2^15, is the sum of two fp16
// numbers (both rounded to nearest: the value to 2^-24 on average), and x g = x0 g0 + x0 g1 + x1 g0, each product exact,
// into the fp32 accumulator (see dhconv_f16.hip, which computes the forward and the input gradient this way).
//
// Operands.  v_mfma_f32_32x32x16_f16 wants, per lane, 8 consecutive k of one channel.  Rows are K here, so a lane that loads the
// (re, im) pair of its channel from 8 rows holds its fragment without any transpose: lanes 0-31 take rows 0-7 of a chunk
// of 16, lanes 32-63 rows 8-15, each load is 256 contiguous bytes per half.  Scales are per channel and chunk, a bound on the exponent
// that follows the rows as they stream by and rescales the partial sums when it moves (the first chunks only, in practice): a
// value keeps 22 bits or more down to 2^-14 of the largest of its channel within the 16 rows, and down to 2^-38 of the
// largest of all its rows.
//
// A workgroup is 8 wavefronts = the 8 degrees that share 64-byte lines of gw ([i][o][l], l fastest),
// all on the same tile of (i, o).  The results meet in LDS and leave as whole lines.
//
// What bounds it: per chunk and 64 x 64 tile a wavefront issues 48 matrix instructions (1536 cycles) and about 330 vector
// instructions, most of them cutting the 64 values it loaded, on a SIMD shared by two wavefronts; they overlap little (leaving out
// the cut or every load takes a tenth off each), and the store of gw (283 MB for 384 x 384 x 240) follows the sums.  384 x 384 channels,
// 240 degrees: 182 / 334 / 566 us for 1 / 2 / 4 samples (on v_mfma_f32_32x32x2_f32, 512 matrix cycles per 16 rows instead of 96: 433 /
// 710 / 1324), error against float64 2.1e-7 (3.2e-7 there: the sums are shorter).
#include "sfno_internal.h"

namespace sfno {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u4 __attribute__((ext_vector_type(4)));

constexpr int WG_TI = 64;            // i per workgroup
constexpr int WG_DEG = 8;            // degrees (wavefronts) per workgroup
constexpr int WG_KC = 16;            // rows per chunk: one matrix K step
constexpr int WG_PITCH = WG_DEG + 1; // float2 per staged line of gw; odd so that the 32 lanes of a store hit 32 banks pairs
constexpr int WG_SH = 14 + 127;      // scaled = x * 2^(SH - E), E = biased exponent bound of the channel: magnitudes below 2^15
constexpr int WG_HEAD = 3;           // bits of headroom left when a bound is set
constexpr int WG_SLACK = 7;          // a bound this far above a chunk's magnitudes (and the headroom) comes down
constexpr int WG_DOWN = 24;

// (value, remainder) of two numbers as packed fp16, both rounded to nearest
__device__ __forceinline__ void cut_pair(float a, float b, unsigned& hi, unsigned& lo) {
    const f16x2 h = __builtin_convertvector(f2{a, b}, f16x2);
    hi = __builtin_bit_cast(unsigned, h);
    lo = __builtin_bit_cast(unsigned, __builtin_convertvector(f2{__builtin_fmaf((float)h[0], -1.0f, a), __builtin_fmaf((float)h[1], -1.0f, b)}, f16x2));
}

// gw is written once and read by another kernel: past the caches, which the rows of X and G need
__device__ __forceinline__ void store_line(float2* p, float2 z) {
    __builtin_nontemporal_store(__builtin_bit_cast(double, z), reinterpret_cast<double*>(p));
}

struct Planes {                      // a channel's 8 rows: real and imaginary part, value and remainder
    u4 r0, r1, i0, i1;
};

// IB, OB: 32-channel blocks of i and o per workgroup (1 for up to 32 channels, and OB = 1 where larger tiles would leave CUs idle)
// OFF: type of a lane's byte offset within a row chunk (64 bits only where 16 row strides do not fit 32)
template <int IB, int OB, typename OFF>
__global__ __launch_bounds__(64 * WG_DEG, OB == 1 && sizeof(OFF) == 4 ? 4 : 2) void dhconv_wgrad_kernel(DhconvWgradArgs p, int ni, int no) {
    constexpr int WG_TO = 32 * OB;   // o per workgroup
    __shared__ float2 stage[32 * WG_TO * WG_PITCH];

    // Workgroups are dealt to the 8 XCDs round-robin by linear id.  All tiles of one group of 8 degrees run
    // as neighbours in one XCD's queue, where they share the rows of X and G in that XCD's L2.  The groups go
    // to the XCDs highest degrees (most rows) first, in alternating direction round by round: the work of a
    // group grows linearly with its degree, and dealing every round in the same direction would give the
    // first XCD a quarter more rows than the average.
    const int xcd = blockIdx.x & 7, q = blockIdx.x >> 3;
    const int tiles = ni * no;
    const int t = q % tiles, gl = q / tiles;
    const int lg = (p.L + WG_DEG - 1) / WG_DEG - 1 - (gl * 8 + ((gl & 1) ? 7 - xcd : xcd));
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
    const int hr = p.M >= WG_KC ? 8 : max(p.M - 8, 0);
    OFF offx[IB], offg[OB];          // byte offset of my channel (clamped to the last one) in my half of a chunk
#pragma unroll
    for (int ib = 0; ib < IB; ++ib) offx[ib] = (OFF)(hr * kg) * (OFF)ms_x + 8u * min(i0 + 32 * ib + jj, p.I - 1);
#pragma unroll
    for (int ob = 0; ob < OB; ++ob) offg[ob] = (OFF)(hr * kg) * (OFF)ms_g + 8u * min(o0 + 32 * ob + jj, p.O - 1);

    f32x16 re[IB][OB], im[IB][OB];
#pragma unroll
    for (int ib = 0; ib < IB; ++ib)
#pragma unroll
        for (int ob = 0; ob < OB; ++ob)
#pragma unroll
            for (int v = 0; v < 16; ++v) re[ib][ob][v] = im[ib][ob][v] = 0.f;
    int ex[IB], eg[OB], tx[IB], tg[OB];   // biased exponent bounds of my channels (lanes jj and jj + 32 agree), and their highest values
#pragma unroll
    for (int ib = 0; ib < IB; ++ib) ex[ib] = tx[ib] = 0;
#pragma unroll
    for (int ob = 0; ob < OB; ++ob) eg[ob] = tg[ob] = 0;

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
    // zeroes the rows of chunk m0 that do not count (see above)
    auto mask = [&](int m0, float2 (&r)[8]) {
        const int first = max(min(m0, p.M - WG_KC), 0) + hr * kg;
        const int lo = kg && p.M < WG_KC ? 8 : m0;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (first + j < lo || first + j >= nm) r[j] = make_float2(0.f, 0.f);
    };
    // moves the channel's bound to the chunk's largest magnitude where that exceeds it, or lies far below it; returns the change
    // the partial sums have to follow.  The bound comes down by at most WG_DOWN from its highest value top (the sums would
    // overflow; what a chunk so far below loses is 2^-60 of the largest product).
    auto bound = [&](const float2 (&r)[8], int& e, int& top) {
        float mx = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(mx) : "v"(r[j].x), "v"(r[j].y));
        const unsigned mb = __builtin_bit_cast(unsigned, mx);
        const auto sw = __builtin_amdgcn_permlane32_swap(mb, mb, false, false);      // the other 8 rows sit 32 lanes away
        const int eb = (int)(max(sw[0], sw[1]) >> 23);
        int en = e;
        if (eb > e || eb < e - WG_HEAD - WG_SLACK) en = max(eb + WG_HEAD, top - WG_DOWN);
        top = max(top, en);
        const int d = e - en;
        e = en;
        return d;
    };
    auto cut = [&](const float2 (&r)[8], int e, Planes& f) {
        const int sh = WG_SH - e;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            unsigned h, s;
            cut_pair(__builtin_ldexpf(r[2 * w].x, sh), __builtin_ldexpf(r[2 * w + 1].x, sh), h, s);
            f.r0[w] = h;
            f.r1[w] = s;
            cut_pair(__builtin_ldexpf(r[2 * w].y, sh), __builtin_ldexpf(r[2 * w + 1].y, sh), h, s);
            f.i0[w] = h;
            f.i1[w] = s;
        }
    };
    // D row of accumulator element v, as the lane that holds that i: 4 x (4 kg) (made opaque where it is used, so that the
    // sixteen addresses are not kept in registers) plus a constant
    auto row_lane = [](int base, int v) { return base + 4 * (8 * (v >> 2) + (v & 3)); };

    const int64_t nchunks = (int64_t)nch * p.B;
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
#pragma unroll
                for (int ib = 0; ib < IB; ++ib) mask(mc, rx[ib]);
#pragma unroll
                for (int ob = 0; ob < OB; ++ob) mask(mc, rg[ob]);
            }
            // the next chunk (the last one again after it) is requested into the registers of this one once they are cut and a
            // batch of matrix instructions is issued
            if (c + 1 < nchunks) {
                m0 += WG_KC;
                if (m0 >= nm) {
                    m0 = 0;
                    Xb += 8 * (int64_t)p.I;
                    Gb += 8 * (int64_t)p.O;
                }
            }
            Planes fx[IB];
#pragma unroll
            for (int ib = 0; ib < IB; ++ib) {
                const int d = bound(rx[ib], ex[ib], tx[ib]);
                cut(rx[ib], ex[ib], fx[ib]);
                __builtin_amdgcn_sched_barrier(0);
                if (__builtin_amdgcn_ballot_w64(d != 0) != 0) {
                    int rl = 16 * kg;
                    asm volatile("" : "+v"(rl));
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const int dv = __builtin_amdgcn_ds_bpermute(row_lane(rl, v), d);
#pragma unroll
                        for (int ob = 0; ob < OB; ++ob) {
                            re[ib][ob][v] = __builtin_ldexpf(re[ib][ob][v], dv);
                            im[ib][ob][v] = __builtin_ldexpf(im[ib][ob][v], dv);
                        }
                    }
                }
            }
#pragma unroll
            for (int ob = 0; ob < OB; ++ob) {
                Planes fg;
                const int d = bound(rg[ob], eg[ob], tg[ob]);
                cut(rg[ob], eg[ob], fg);
                if (__builtin_amdgcn_ballot_w64(d != 0) != 0) {
#pragma unroll
                    for (int ib = 0; ib < IB; ++ib)
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            re[ib][ob][v] = __builtin_ldexpf(re[ib][ob][v], d);
                            im[ib][ob][v] = __builtin_ldexpf(im[ib][ob][v], d);
                        }
                }
                __builtin_amdgcn_sched_barrier(0);
                const f16x8 gr0 = __builtin_bit_cast(f16x8, fg.r0), gr1 = __builtin_bit_cast(f16x8, fg.r1);
                const f16x8 gi0 = __builtin_bit_cast(f16x8, fg.i0), gi1 = __builtin_bit_cast(f16x8, fg.i1);
                const f16x8 ng0 = __builtin_bit_cast(f16x8, fg.r0 ^ 0x80008000u), ng1 = __builtin_bit_cast(f16x8, fg.r1 ^ 0x80008000u);     // -Gr
                // smallest terms first; consecutive instructions go to different accumulators
#define WG_STEP(A, B, C, D)                                                                                                     \
    _Pragma("unroll") for (int ib = 0; ib < IB; ++ib) {                                                                        \
        re[ib][ob] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, fx[ib].A), B, re[ib][ob], 0, 0, 0);       \
        im[ib][ob] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, fx[ib].C), D, im[ib][ob], 0, 0, 0);       \
    }
                WG_STEP(r1, gr0, r1, gi0)
                WG_STEP(i1, gi0, i1, ng0)
                WG_STEP(r0, gr1, r0, gi1)
                WG_STEP(i0, gi1, i0, ng1)
                WG_STEP(r0, gr0, r0, gi0)
                WG_STEP(i0, gi0, i0, ng0)
#undef WG_STEP
                __builtin_amdgcn_sched_barrier(0);
                if (ob == 0) {
#pragma unroll
                    for (int ib = 0; ib < IB; ++ib) load(Xb, ms_x, offx[ib], m0, rx[ib]);
                }
                load(Gb, ms_g, offg[ob], m0, rg[ob]);
                __builtin_amdgcn_sched_barrier(0);
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
            const int er = __builtin_amdgcn_ds_bpermute(row_lane(16 * kg, v), ex[ib]) - 2 * WG_SH;
            const int il = 8 * (v >> 2) + 4 * kg + (v & 3);
#pragma unroll
            for (int ob = 0; ob < OB; ++ob)
                stage[(il * WG_TO + 32 * ob + jj) * WG_PITCH + wave] =
                    make_float2(__builtin_ldexpf(re[ib][ob][v], er + eg[ob]), __builtin_ldexpf(im[ib][ob][v], er + eg[ob]));
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

}  // namespace

int dhconv_wgrad_launch(const DhconvWgradArgs& a, hipStream_t s) {
    // a lane's offset in a row chunk: 16 row strides and the channel, in 32 bits
    const int64_t ld = a.ld_in > a.ld_out ? a.ld_in : a.ld_out;
    const bool wide = 64 * (int64_t)a.L * ld + 4 * ld > 0xffffffffLL;
    const int64_t groups = 8 * (((a.L + WG_DEG - 1) / WG_DEG + 7) / 8);
    const int ni = (a.I + WG_TI - 1) / WG_TI;
    // 64 x 64 tiles cut and load a third less per product, 64 x 32 tiles need half the registers and LDS (two workgroups per CU,
    // twice as many): 182 against 273 us for 384 x 384 channels and 240 degrees (1080 tiles of 64 x 64), 43 against 32 us for
    // 128 x 128 and 90 (48 tiles).  The line: two tiles per CU.
    const int no2 = (a.O + 63) / 64;
    const bool narrow = a.O <= 32 || (!wide && groups * ni * no2 < 512);
    const int no = narrow ? (a.O + 31) / 32 : no2;
    const int64_t blocks = groups * ni * no;
    if (blocks > 0x7fffffffLL) return SFNO_EUNSUPPORTED;
    const dim3 grid((unsigned)blocks), block(64 * WG_DEG);
    if (wide)
        hipLaunchKernelGGL((dhconv_wgrad_kernel<2, 2, uint64_t>), grid, block, 0, s, a, ni, no);
    else if (!narrow)
        hipLaunchKernelGGL((dhconv_wgrad_kernel<2, 2, unsigned>), grid, block, 0, s, a, ni, no);
    else if (a.I > 32)
        hipLaunchKernelGGL((dhconv_wgrad_kernel<2, 1, unsigned>), grid, block, 0, s, a, ni, no);
    else
        hipLaunchKernelGGL((dhconv_wgrad_kernel<1, 1, unsigned>), grid, block, 0, s, a, ni, no);
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

}  // namespace sfno
