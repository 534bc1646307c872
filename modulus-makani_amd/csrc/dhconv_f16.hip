// dhconv with fp32 accuracy on the fp16 matrix pipe of gfx950 (the default fp32 path for even channel counts):
//
//   y[b,o,l,m] = sum_i x[b,i,l,m] w[i,o,l]        (makani/models/common/contractions.py:130-136)
//
// An fp32 number scaled by a power of two into the range of fp16 is, to 22 of its 24 significant bits, the sum of
// two fp16 numbers (11 significant bits each): x 2^s = h0 + h1.  With both operands cut that way
//   x w = (a0 b0 + a0 b1 + a1 b0) 2^-(s+t)  up to  a1 b1  (below 2^-21 of the product) and the two cut-off tails,
// three v_mfma_f32_32x32x16_f16 per K = 16 step into the fp32 accumulator, each product exact.
//
// Per degree l the contraction is four real GEMMs on the real and imaginary parts,
//   Yr = Xr Wr + (-Xi) Wi,   Yi = Xr Wi + Xi Wr,
// with rows (m, b) of the spectral layout as A operands (read straight from HBM/L2, de-interleaved and cut in
// registers; -Xi costs one sign flip per packed pair) and the weights as B operands: the packed stream holds, per
// (degree, block of 32 NTC output channels, chunk of 16 input channels), the image of one LDS stage -- (Wr, Wi) x two
// fp16 planes x output channel x 16 input channels -- which the wavefronts move with global_load_lds_dwordx4 into a
// ring of three stages, two chunks ahead of the matrix instructions.  8 bytes per complex weight, read once.
//
// Scales.  fp16 keeps 11 significant bits only above 2^-14, so every operand row is brought close to the top of the
// range (magnitudes below 2^15) by a power of two, which costs no accuracy and is undone when the result is stored:
//   weights: one scale per (degree, output channel), from the largest |Re|, |Im| over the input channels, chosen when
//            the weights are packed;
//   activations: one scale per row (m, l, b), found while the row streams by.  A wavefront owns 32 rows and reads
//            each in chunks of 16 complex values; it keeps a bound on the row's exponent that is raised (with a few
//            bits of headroom) when a chunk exceeds it, and then rescales the row's partial sums by the same power of two.
// Entries much smaller than the largest entry of their row (by more than 2^17) keep fewer bits: the error of a
// product is bounded by 2^-21 |x w| + 2^-38 max|x| max|w|, where fp32 arithmetic has 2^-24 |x w|.
#include "dhconv_map.h"
#include <algorithm>

#include "sfno_internal.h"

namespace sfno {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __fp16 fp16x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u4 __attribute__((ext_vector_type(4)));

constexpr int DHF_KC = 16;             // complex input channels per chunk: one matrix K step per part
constexpr int DHF_TOP = 14;            // scaled magnitudes stay below 2^(TOP + 1)
constexpr int DHF_HEAD = 3;            // bits of headroom left when a row's exponent bound is raised
constexpr int DHF_SH = DHF_TOP + 127;  // scaled = x * 2^(SH - E), E = biased exponent bound of the row
constexpr int DHF_STAGES = 3;

__device__ __forceinline__ unsigned int pk_rtz(float a, float b) {
    return __builtin_bit_cast(unsigned int, __builtin_amdgcn_cvt_pkrtz(a, b));
}
// 16 bytes per lane from global memory to LDS base + 16 lane (M0 carries the base; the compiler reserves M0 and does not
// accept it on a clobber list: nothing else in this file may depend on M0 -- no indexed register arrays, no LDS-DMA builtins)
__device__ __forceinline__ void dhf_dma16(const void* g, unsigned lds_byte_addr) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(lds_byte_addr) : "memory");
}
// byte offset, within one (part, plane) of a stage, of the 16-byte piece (output channel o, half kg of the chunk):
// the halves swap places every 8 channels so that the 16-byte reads of 16 consecutive lanes cover all banks
__host__ __device__ constexpr int dhf_piece(int o, int kg) { return o * 32 + ((kg ^ ((o >> 3) & 1)) * 16); }

// grid = dh_blocks workgroups (see dh_map), row groups of 128; a.nob = ceil(O / (32 NTC)); requires 2*I % 4 == 0
template <int NTC>
__global__ __launch_bounds__(256, 2) void dhconv_f16_kernel(DhconvArgs a) {
    constexpr int CO = 32 * NTC;                     // complex output channels per workgroup
    constexpr int STAGE = 4 * CO * 32;               // bytes: (Wr, Wi) x 2 planes x CO x 16 fp16
    constexpr int ND = STAGE / 4096;                 // direct-to-LDS loads per wavefront and chunk
    constexpr int NX = 4;                            // activation loads per lane and chunk
    __shared__ __align__(16) unsigned char lds[DHF_STAGES * STAGE];

    int l, ob, r0, ncols, rot;
    if (!dh_map(a, 128, l, ob, r0, ncols, rot)) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wslot = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave = (wslot + rot) & 3;
    const bool active = r0 + 32 * wave < ncols;
    const int nc = a.nc;                                           // chunks of 16 complex input channels
    const int kg = lane >> 5, cl = lane & 31;
    const unsigned lds0 = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)lds);

    const int n = min(r0 + 32 * wave + cl, ncols - 1);
    const int mm = n / a.B, bb = n - mm * a.B;
    const float* xrow = a.X + ((int64_t)mm * a.L + l) * a.ld_in + (int64_t)bb * a.I2;
    // packed weights of (l, ob): nc stage images; this wavefront moves bytes [ND wslot KiB, ND (wslot + 1) KiB) of each
    const unsigned char* wsrc = reinterpret_cast<const unsigned char*>(a.W) + ((int64_t)l * a.nob + ob) * nc * STAGE + wslot * (ND * 1024) + lane * 16;
    const unsigned wdst = lds0 + wslot * (ND * 1024);

    floatx16 yr[NTC], yi[NTC];
#pragma unroll
    for (int t = 0; t < NTC; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            yr[t][v] = 0.0f;
            yi[t][v] = 0.0f;
        }
    int E = 0;                 // biased exponent bound of my row (lanes cl and cl + 32 hold the same row and agree)
    int pend = 0;              // change of E by the last chunk that was cut, not yet applied to the partial sums

    // my 8 complex activations of chunk c: i = 16c + 8kg .. +7, (re, im) interleaved (clamped in groups of two complex
    // values; the weights are zero past I)
    auto x_load = [&](int c, f4 (&xr)[NX]) {
        const int k = 2 * DHF_KC * c + 16 * kg;
#pragma unroll
        for (int j = 0; j < NX; ++j) xr[j] = *reinterpret_cast<const f4*>(xrow + min(k + 4 * j, a.I2 - 4));
    };
    auto w_dma = [&](int c, int stage) {
#pragma unroll
        for (int j = 0; j < ND; ++j) dhf_dma16(wsrc + (int64_t)c * STAGE + j * 1024, wdst + stage * STAGE + j * 1024);
    };
    // exponent bound of the row after this chunk
    auto bound = [&](const f4 (&xr)[NX]) {
        float mx = 0.f;
#pragma unroll
        for (int j = 0; j < NX; ++j)
            mx = __builtin_fmaxf(__builtin_fmaxf(mx, __builtin_fmaxf(__builtin_fabsf(xr[j][0]), __builtin_fabsf(xr[j][1]))),
                                 __builtin_fmaxf(__builtin_fabsf(xr[j][2]), __builtin_fabsf(xr[j][3])));
        const unsigned int mb = __builtin_bit_cast(unsigned int, mx);
        // the other half of the row's chunk sits 32 lanes away
        const auto sw = __builtin_amdgcn_permlane32_swap(mb, mb, false, false);
        const int eb = (int)(max(sw[0], sw[1]) >> 23);
        const int en = eb > E ? eb + DHF_HEAD : E;
        pend = E - en;
        E = en;
    };
    // planes of the chunk: pl[0], pl[1] = Xr (upper, lower part), pl[2], pl[3] = Xi; word e of a plane holds the channels
    // 2e, 2e + 1 of the lane's eight
    auto cut_quad = [&](const f4 (&xr)[NX], int e, u4 (&pl)[4]) {
        const f4 s = xr[e];
        const int sh = DHF_SH - E;
        const float ra = __builtin_ldexpf(s[0], sh), ia = __builtin_ldexpf(s[1], sh), rb = __builtin_ldexpf(s[2], sh), ib = __builtin_ldexpf(s[3], sh);
        const fp16x2 hr = __builtin_amdgcn_cvt_pkrtz(ra, rb), hi = __builtin_amdgcn_cvt_pkrtz(ia, ib);
        pl[0][e] = __builtin_bit_cast(unsigned int, hr);
        pl[1][e] = pk_rtz(__builtin_fmaf((float)hr[0], -1.0f, ra), __builtin_fmaf((float)hr[1], -1.0f, rb));
        pl[2][e] = __builtin_bit_cast(unsigned int, hi);
        pl[3][e] = pk_rtz(__builtin_fmaf((float)hi[0], -1.0f, ia), __builtin_fmaf((float)hi[1], -1.0f, ib));
    };
    // partial sums follow their row's scale: D row 8 (v / 4) + 4 kg + v % 4 belongs to the lanes of that number
    auto rescale = [&]() {
        if (__builtin_amdgcn_ballot_w64(pend != 0) == 0) return;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int d = __builtin_amdgcn_ds_bpermute(4 * (8 * (v >> 2) + 4 * kg + (v & 3)), pend);
#pragma unroll
            for (int t = 0; t < NTC; ++t) {
                yr[t][v] = __builtin_ldexpf(yr[t][v], d);
                yi[t][v] = __builtin_ldexpf(yi[t][v], d);
            }
        }
    };
    // one chunk of matrix instructions on stage `stage` with the planes pc
    const int frag = dhf_piece(cl, kg);
    auto contract = [&](int stage, const u4 (&pc)[4]) {
        const unsigned char* sb = lds + stage * STAGE + frag;
        const f16x8 xr0 = __builtin_bit_cast(f16x8, pc[0]), xr1 = __builtin_bit_cast(f16x8, pc[1]);
        const f16x8 xi0 = __builtin_bit_cast(f16x8, pc[2]), xi1 = __builtin_bit_cast(f16x8, pc[3]);
        // -Xi: one sign flip per packed pair
        const f16x8 ni0 = __builtin_bit_cast(f16x8, pc[2] ^ 0x80008000u), ni1 = __builtin_bit_cast(f16x8, pc[3] ^ 0x80008000u);
#pragma unroll
        for (int t = 0; t < NTC; ++t) {
            const f16x8 wr0 = *reinterpret_cast<const f16x8*>(sb + (0 * CO + 32 * t) * 32), wr1 = *reinterpret_cast<const f16x8*>(sb + (1 * CO + 32 * t) * 32);
            const f16x8 wi0 = *reinterpret_cast<const f16x8*>(sb + (2 * CO + 32 * t) * 32), wi1 = *reinterpret_cast<const f16x8*>(sb + (3 * CO + 32 * t) * 32);
            // smallest terms first; the two sums alternate so that no instruction waits for the one before it
            yr[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xr1, wr0, yr[t], 0, 0, 0);
            yi[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xr1, wi0, yi[t], 0, 0, 0);
            yr[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ni1, wi0, yr[t], 0, 0, 0);
            yi[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xi1, wr0, yi[t], 0, 0, 0);
            yr[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xr0, wr1, yr[t], 0, 0, 0);
            yi[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xr0, wi1, yi[t], 0, 0, 0);
            yr[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ni0, wi1, yr[t], 0, 0, 0);
            yi[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xi0, wr1, yi[t], 0, 0, 0);
            yr[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xr0, wr0, yr[t], 0, 0, 0);
            yi[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xr0, wi0, yi[t], 0, 0, 0);
            yr[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ni0, wi0, yr[t], 0, 0, 0);
            yi[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xi0, wr0, yi[t], 0, 0, 0);
        }
    };

    // Pipeline, three weight stages.  Iteration c: cut the activations of chunk c + 1 (requested during iteration c - 1;
    // the compiler's wait for them also covers this wavefront's pieces of the weights of chunk c + 1, which were requested
    // before them), barrier (every wavefront's pieces of chunk c + 1 have landed and every wavefront is done reading
    // chunk c - 1), request chunk c + 2 into the stage of chunk c - 1, contract chunk c, and let the partial sums follow
    // the scale chunk c + 1 was cut with.  The requests thus have one contraction (48 or 24 matrix instructions) to land.
    // Only the weight requests are written in assembly (the compiler would make every LDS read wait for them); their
    // wait is the explicit one before the barrier.
    f4 X0[NX], X1[NX];
    u4 P0[4], P1[4];
    if (active) x_load(0, X0);
    w_dma(0, 0);
    if (nc > 1) {
        if (active) x_load(1, X1);
        w_dma(1, 1);
    }
    if (active) {
        bound(X0);
#pragma unroll
        for (int e = 0; e < NX; ++e) cut_quad(X0, e, P0);
    }
    pend = 0;                                                       // nothing has been summed yet

    auto iter = [&](int c, int stage, const u4 (&pc)[4], u4 (&pn)[4], f4 (&xc)[NX], const f4 (&xn)[NX]) {
        const bool more1 = c + 1 < nc, more2 = c + 2 < nc;         // uniform over the workgroup
        if (active && more1) {
            bound(xn);
#pragma unroll
            for (int e = 0; e < NX; ++e) cut_quad(xn, e, pn);
        }
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (more2) {
            // xc held chunk c, cut during the previous iteration
            if (active) x_load(c + 2, xc);
            w_dma(c + 2, stage == 0 ? 2 : stage - 1);
        }
        if (active) {
            contract(stage, pc);
            rescale();
            pend = 0;
        }
    };
    int c = 0, stage = 0;
    for (; c + 1 < nc; c += 2) {
        iter(c, stage, P0, P1, X0, X1);
        stage = stage == 2 ? 0 : stage + 1;
        iter(c + 1, stage, P1, P0, X1, X0);
        stage = stage == 2 ? 0 : stage + 1;
    }
    if (c < nc) iter(c, stage, P0, P1, X0, X1);

    if (!active) return;
    // Undo the scales: row by 2^(E - SH) (the partial sums carry the scale of the last cut), column by the factor stored
    // with the weights.
    float cinv[NTC];
#pragma unroll
    for (int t = 0; t < NTC; ++t) cinv[t] = a.cinv[(int64_t)l * (a.nob * CO) + CO * ob + 32 * t + cl];
    const int Efinal = E;
    const int nn0 = r0 + 32 * wave + 4 * kg;                       // my first row; the others are 8 (v / 4) + v % 4 further on
    if (a.B == 1 && r0 + 32 * wave + 32 <= ncols && 2 * (CO * ob + CO) <= a.O2) {
        // one sample and no row or channel of my tile outside the tensor: row = order, one address, constant steps
        float* o = a.Y + ((int64_t)nn0 * a.L + l) * a.ld_out + 2 * (CO * ob + cl);
        const int64_t rstep = (int64_t)a.L * a.ld_out;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int er = __builtin_amdgcn_ds_bpermute(4 * (8 * (v >> 2) + 4 * kg + (v & 3)), Efinal);
            float* orow = o + (8 * (v >> 2) + (v & 3)) * rstep;
#pragma unroll
            for (int t = 0; t < NTC; ++t)
                *reinterpret_cast<f2*>(orow + 64 * t) = f2{__builtin_ldexpf(yr[t][v], er - DHF_SH) * cinv[t], __builtin_ldexpf(yi[t][v], er - DHF_SH) * cinv[t]};
        }
        return;
    }
    if ((a.B & (a.B - 1)) == 0 && r0 + 32 * wave + 32 <= ncols && 2 * (CO * ob + CO) <= a.O2) {
        // a power-of-two number of samples, whole tile inside: (order, sample) of a row by shift and mask, no checks
        const int lb = 31 - __builtin_clz(a.B);
        float* o = a.Y + (int64_t)l * a.ld_out + 2 * (CO * ob + cl);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int er = __builtin_amdgcn_ds_bpermute(4 * (8 * (v >> 2) + 4 * kg + (v & 3)), Efinal);
            const int nn = nn0 + 8 * (v >> 2) + (v & 3);
            float* orow = o + (int64_t)(nn >> lb) * a.L * a.ld_out + (int64_t)(nn & (a.B - 1)) * a.O2;
#pragma unroll
            for (int t = 0; t < NTC; ++t)
                *reinterpret_cast<f2*>(orow + 64 * t) = f2{__builtin_ldexpf(yr[t][v], er - DHF_SH) * cinv[t], __builtin_ldexpf(yi[t][v], er - DHF_SH) * cinv[t]};
        }
        return;
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int er = __builtin_amdgcn_ds_bpermute(4 * (8 * (v >> 2) + 4 * kg + (v & 3)), Efinal);
        const int nn = nn0 + 8 * (v >> 2) + (v & 3);
        if (nn >= ncols) continue;
        const int m2 = nn / a.B, b2 = nn - m2 * a.B;
        float* orow = a.Y + ((int64_t)m2 * a.L + l) * a.ld_out + (int64_t)b2 * a.O2;
#pragma unroll
        for (int t = 0; t < NTC; ++t) {
            const int oc = 2 * (CO * ob + 32 * t + cl);
            if (oc < a.O2)
                *reinterpret_cast<f2*>(orow + oc) = f2{__builtin_ldexpf(yr[t][v], er - DHF_SH) * cinv[t], __builtin_ldexpf(yi[t][v], er - DHF_SH) * cinv[t]};
        }
    }
}

// cmax[o][l] = largest |Re|, |Im| of w[.][o][l] over the input channels (adjoint: of w[o][.][l], w being [O][I][L]).  A thread
// takes DHF_CMAX_I input channels of one (o, l) and joins the others with an integer atomic maximum on the bit pattern (the
// values are magnitudes: their order as unsigned integers is their order as floats, a NaN ranks above all and stays); cmax is
// cleared by the kernel in front.  Degrees [lb, lb + ln).  grid (ceil(O ln / 256), ceil(I / DHF_CMAX_I))
constexpr int DHF_CMAX_I = 16;
__global__ __launch_bounds__(256) void dhconv_colmax_clear_kernel(float* __restrict__ cmax, int64_t n) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx < n) cmax[idx] = 0.f;
}
__global__ __launch_bounds__(256) void dhconv_colmax_kernel(const float2* __restrict__ w, float* __restrict__ cmax, int I, int O, int L, int adjoint,
                                                            int lb, int ln) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;     // o * ln + l - lb
    if (idx >= (int64_t)O * ln) return;
    const int o = (int)(idx / ln), l = lb + (int)(idx - (int64_t)o * ln);
    const int i0 = blockIdx.y * DHF_CMAX_I, i1 = min(i0 + DHF_CMAX_I, I);
    float mx = 0.f;
#pragma unroll 8
    for (int i = i0; i < i1; ++i) {
        const float2 z = adjoint ? w[((int64_t)o * I + i) * L + l] : w[((int64_t)i * O + o) * L + l];
        mx = fmaxf(mx, fmaxf(fabsf(z.x), fabsf(z.y)));
    }
    atomicMax(reinterpret_cast<unsigned int*>(cmax) + (int64_t)o * L + l, __float_as_uint(mx));
}

// Writes the stage images.  packed[l][ob][c] = [part (Re, Im)][plane][o (CO)][two 16-byte halves, see dhf_piece]: the half kg
// of channel o holds plane `plane` of part `part` of w[16c + 8kg + e][CO ob + o][l] * 2^s[l][o], e = 0..7, as fp16; plane 0 is
// the value rounded to fp16, plane 1 the rounded remainder; zero outside the weight (adjoint: the weight is conj(w[o][i][l]),
// w being [O][I][L]).  cinv[l][CO ob + o] = 2^-s.  The parameter has l fastest, the stream has it slowest: a workgroup moves
// the 16 x 32 channel pairs of one (c, ob, quarter of the channel block) for 16 degrees through LDS, reading 128 contiguous
// bytes per pair, whole lines where L is a multiple of 16 (8 degrees and half lines: column
// maxima and packing of 384 x 384 x 240 264 us, then 236; 128 x 128 x 90 21.6 -> 16.0).  A thread cuts its values into all four of their pieces
// (one piece per thread read every value four times and waited for its column maximum in each of eight rounds: 176 -> 147 us for this kernel).  grid (nc * nob * (CO / 32), ceil(L / 16)), block 512
constexpr int DHF_PL = 16;
// Weight bytes of a slab of degrees whose maxima are taken and which is packed before the next one: the packing reads it from the memory-side
// cache of 256 MB, which holds the slab and what is written meanwhile.  384 x 384 x 240 (283 MB) in three slabs: maxima 72 -> 81 us,
// packing 147 -> 113; smaller weights are one slab.
constexpr int64_t DHF_SLAB_BYTES = 96 << 20;
template <int NTC>
__global__ __launch_bounds__(512) void dhconv_pack_f16_kernel(const float2* __restrict__ w, const float* __restrict__ cmax, unsigned char* __restrict__ packed,
                                                              float* __restrict__ cinv, int I, int O, int L, int nob, int nc, int adjoint, int lb) {
    constexpr int CO = 32 * NTC, STAGE = 4 * CO * 32;
    __shared__ float2 tile[512][DHF_PL + 1];         // [pair = ii * 32 + o][degree], padded
    const int q = blockIdx.x % NTC, c = (blockIdx.x / NTC) % nc, ob = blockIdx.x / (NTC * nc);
    const int l0 = lb + blockIdx.y * DHF_PL;
    const int tid = threadIdx.x, dl = tid & (DHF_PL - 1);
#pragma unroll
    for (int pass = 0; pass < DHF_PL; ++pass) {
        const int pr = pass * (512 / DHF_PL) + tid / DHF_PL;     // sixteen lanes per pair: one 128-byte segment
        const int ii = pr >> 5, o = pr & 31;
        const int i = DHF_KC * c + ii, oo = CO * ob + 32 * q + o, l = l0 + dl;
        float2 z = make_float2(0.f, 0.f);
        if (i < I && oo < O && l < L) {
            if (adjoint) {
                z = w[((int64_t)oo * I + i) * L + l];
                z.y = -z.y;
            } else {
                z = w[((int64_t)i * O + oo) * L + l];
            }
        }
        tile[pr][dl] = z;
    }
    // wavefront -> degrees wave and wave + 8, lane -> (half kg, channel o): all four 16-byte pieces of a lane's eight values; the column
    // maxima are requested before the barrier
    const int o = tid & 31, kg = (tid >> 5) & 1, wave = tid >> 6;
    const int oo = CO * ob + 32 * q + o;
    int sh[DHF_PL / 8];
#pragma unroll
    for (int k = 0; k < DHF_PL / 8; ++k) {
        const int l = l0 + 8 * k + wave;
        // scale: the column's largest magnitude lands in [2^TOP, 2^(TOP+1))
        const unsigned int mb = oo < O && l < L ? __builtin_bit_cast(unsigned int, cmax[(int64_t)oo * L + l]) : 0u;
        sh[k] = mb != 0 ? DHF_SH - (int)(mb >> 23) : 0;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < DHF_PL / 8; ++k) {
        const int d = 8 * k + wave, l = l0 + d;
        if (l >= L) break;
        if (c == 0 && kg == 0) cinv[(int64_t)l * (nob * CO) + CO * ob + 32 * q + o] = __builtin_ldexpf(1.0f, -sh[k]);
        unsigned short h[2][2][8];      // [part][plane][value]
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float2 z = tile[(8 * kg + e) * 32 + o][d];
#pragma unroll
            for (int part = 0; part < 2; ++part) {
                const float v = __builtin_ldexpf(part ? z.y : z.x, sh[k]);
                const _Float16 v0 = (_Float16)v;
                h[part][0][e] = __builtin_bit_cast(unsigned short, v0);
                h[part][1][e] = __builtin_bit_cast(unsigned short, (_Float16)(v - (float)v0));
            }
        }
        unsigned char* dst = packed + (((int64_t)l * nob + ob) * nc + c) * STAGE + 32 * q * 32 + dhf_piece(o, kg);
#pragma unroll
        for (int pp = 0; pp < 4; ++pp) {
            u4 piece;
#pragma unroll
            for (int e2 = 0; e2 < 4; ++e2)
                piece[e2] = (unsigned int)h[pp >> 1][pp & 1][2 * e2] | ((unsigned int)h[pp >> 1][pp & 1][2 * e2 + 1] << 16);
            *reinterpret_cast<u4*>(dst + pp * CO * 32) = piece;
        }
    }
}

int dhconv_f16_ntc(int O) { return O > 64 ? 4 : 2; }

int dhconv_pack_f16_launch(const float2* w, void* packed, float* cinv, float* cmax, int I, int O, int L, int adjoint, hipStream_t s) {
    const int ntc = dhconv_f16_ntc(O);
    const int nob = (O + 32 * ntc - 1) / (32 * ntc), nc = (I + DHF_KC - 1) / DHF_KC;
    if ((int64_t)nob * nc * ntc > 0x7fffffffLL || (L + DHF_PL - 1) / DHF_PL > 65535) return SFNO_EUNSUPPORTED;
    const int64_t cols = (int64_t)O * L;
    if ((cols + 255) / 256 > 0x7fffffffLL) return SFNO_EUNSUPPORTED;
    if ((I + DHF_CMAX_I - 1) / DHF_CMAX_I > 65535) return SFNO_EUNSUPPORTED;
    hipLaunchKernelGGL(dhconv_colmax_clear_kernel, dim3((unsigned)((cols + 255) / 256)), dim3(256), 0, s, cmax, cols);
    // maxima and packing a slab of degrees at a time, so that the packing finds the slab in the memory-side cache (256 MB)
    const int64_t per16 = (int64_t)sizeof(float2) * I * O * DHF_PL;
    const int slab = DHF_PL * (int)std::max<int64_t>(1, std::min<int64_t>((L + DHF_PL - 1) / DHF_PL, DHF_SLAB_BYTES / per16));
    for (int lb = 0; lb < L; lb += slab) {
        const int ln = std::min(slab, L - lb);
        hipLaunchKernelGGL(dhconv_colmax_kernel, dim3((unsigned)(((int64_t)O * ln + 255) / 256), (unsigned)((I + DHF_CMAX_I - 1) / DHF_CMAX_I)), dim3(256), 0, s,
                           w, cmax, I, O, L, adjoint, lb, ln);
        const dim3 grid((unsigned)(nob * nc * ntc), (unsigned)((ln + DHF_PL - 1) / DHF_PL));
        if (ntc == 4)
            hipLaunchKernelGGL((dhconv_pack_f16_kernel<4>), grid, dim3(512), 0, s, w, cmax, reinterpret_cast<unsigned char*>(packed), cinv, I, O, L, nob, nc,
                               adjoint, lb);
        else
            hipLaunchKernelGGL((dhconv_pack_f16_kernel<2>), grid, dim3(512), 0, s, w, cmax, reinterpret_cast<unsigned char*>(packed), cinv, I, O, L, nob, nc,
                               adjoint, lb);
    }
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

// A weight w[i][o][l] and its conjugate transpose packed together (training: the backward wants the second one).  HBM bounds this: one
// reading for both maxima and one for both packings instead of two each, and the writes.  384 x 384 x 240 (283 MB) 370 -> 272 us for the pair
// (maxima 94, packing 174), 128 x 128 x 90 30 -> 17.4, 32 x 32 x 4 18.7 -> 11.5 (launches).
//
// cmax[o][l] over the input channels and amax[i][l] over the output channels: a workgroup takes 16 x 16 channel pairs of 64 degrees, a
// wavefront two input channels and a lane one degree (runs of 512 bytes: 384 x 384 x 240 in 94 us; 32 x 32 pairs of 16 degrees, runs of 128 bytes: 213).  The
// maxima leave as above.  Degrees [lb, lb + ln).  grid (ceil(O / 16), ceil(I / 16), ceil(ln / 64)), block 512
__global__ __launch_bounds__(256) void dhconv_bothmax_clear_kernel(float* __restrict__ cmax, int64_t n, float* __restrict__ amax, int64_t na) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx < n) cmax[idx] = 0.f;
    if (idx < na) amax[idx] = 0.f;
}
__global__ __launch_bounds__(512) void dhconv_bothmax_kernel(const float2* __restrict__ w, float* __restrict__ cmax, float* __restrict__ amax, int I, int O,
                                                             int L, int lb, int ln) {
    __shared__ float part[8][16][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int o0 = 16 * blockIdx.x, i0 = 16 * blockIdx.y + 2 * wave;
    const int l = lb + 64 * blockIdx.z + lane;
    const bool in = l < lb + ln;
    // (no load under a branch: channels past the end repeat the last one's values)
    const int lc = in ? l : lb;
    float2 z[2][16];
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int k = 0; k < 16; ++k) z[e][k] = w[((int64_t)min(i0 + e, I - 1) * O + min(o0 + k, O - 1)) * L + lc];
    float cm[16], rm[2] = {0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        cm[k] = 0.f;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float v = fmaxf(fabsf(z[e][k].x), fabsf(z[e][k].y));
            cm[k] = fmaxf(cm[k], v);
            rm[e] = fmaxf(rm[e], v);
        }
    }
#pragma unroll
    for (int e = 0; e < 2; ++e)
        if (in && i0 + e < I) atomicMax(reinterpret_cast<unsigned int*>(amax) + (int64_t)(i0 + e) * L + l, __float_as_uint(rm[e]));
#pragma unroll
    for (int k = 0; k < 16; ++k) part[wave][k][lane] = cm[k];
    __syncthreads();
#pragma unroll
    for (int k = wave; k < 16; k += 8) {
        float v = part[0][k][lane];
#pragma unroll
        for (int p = 1; p < 8; ++p) v = fmaxf(v, part[p][k][lane]);
        if (in && o0 + k < O) atomicMax(reinterpret_cast<unsigned int*>(cmax) + (int64_t)(o0 + k) * L + l, __float_as_uint(v));
    }
}

// One operand stream of dhconv_pack_both_kernel (layout as dhconv_pack_f16_kernel writes it).
struct DhfStream {
    unsigned char* packed;
    float* cinv;
    const float* cmax;
    int nob, nc, co;                // column blocks, chunks of 16 input channels, channels per column block
};
__device__ __forceinline__ int dhf_shift(const float* __restrict__ cmax, int64_t idx) {
    const unsigned int mb = __builtin_bit_cast(unsigned int, cmax[idx]);
    return mb != 0 ? DHF_SH - (int)(mb >> 23) : 0;
}
// eight values of a column, scaled by 2^sh, as the four pieces of their half chunk
template <class Get>
__device__ __forceinline__ void dhf_store_pieces(unsigned char* dst, int co, int sh, float sign, Get get) {
    unsigned short h[2][2][8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float2 z = get(e);
#pragma unroll
        for (int part = 0; part < 2; ++part) {
            const float v = __builtin_ldexpf(part ? sign * z.y : z.x, sh);
            const _Float16 v0 = (_Float16)v;
            h[part][0][e] = __builtin_bit_cast(unsigned short, v0);
            h[part][1][e] = __builtin_bit_cast(unsigned short, (_Float16)(v - (float)v0));
        }
    }
#pragma unroll
    for (int pp = 0; pp < 4; ++pp) {
        u4 piece;
#pragma unroll
        for (int e2 = 0; e2 < 4; ++e2)
            piece[e2] = (unsigned int)h[pp >> 1][pp & 1][2 * e2] | ((unsigned int)h[pp >> 1][pp & 1][2 * e2 + 1] << 16);
        *reinterpret_cast<u4*>(dst + pp * co * 32) = piece;
    }
}
// A workgroup moves 16 input x 32 output channels of 16 degrees through LDS: as a chunk of the weight (f, lane = half chunk and output
// channel) and as 16 columns of two chunks of its conjugate transpose (t, lane = half chunk and input channel; the input channels' pitch
// spreads them over all banks).  Tiles that only one of the streams has, in its padding, are zeros.
// grid (tiles of 16 input channels, tiles of 32 output channels, ceil(ln / 16)), block 512
constexpr int DHF_PITCH = 32 * (DHF_PL + 1) + 1;
__global__ __launch_bounds__(512) void dhconv_pack_both_kernel(const float2* __restrict__ w, DhfStream f, DhfStream t, int I, int O, int L, int lb) {
    __shared__ float2 tile[DHF_KC * DHF_PITCH];
    const int ti = blockIdx.x, to = blockIdx.y;
    const int l0 = lb + blockIdx.z * DHF_PL;
    const int tid = threadIdx.x, dl = tid & (DHF_PL - 1);
#pragma unroll
    for (int pass = 0; pass < DHF_PL; ++pass) {
        const int pr = pass * (512 / DHF_PL) + tid / DHF_PL;     // sixteen lanes per pair: one 128-byte segment
        const int ii = pr >> 5, o = pr & 31;
        const int i = DHF_KC * ti + ii, oo = 32 * to + o, l = l0 + dl;
        float2 z = make_float2(0.f, 0.f);
        if (i < I && oo < O && l < L) z = w[((int64_t)i * O + oo) * L + l];
        tile[ii * DHF_PITCH + o * (DHF_PL + 1) + dl] = z;
    }
    const int lane = tid & 63, wave = tid >> 6;                  // wavefront -> degrees wave and wave + 8
    const int of = lane & 31, kf = lane >> 5, it = lane & 15, ot = lane >> 4;
    const int oo = 32 * to + of, ii = DHF_KC * ti + it, ct = 2 * to + (ot >> 1);
    const bool has_f = ti < f.nc && 32 * to < f.nob * f.co, has_t = ct < t.nc && DHF_KC * ti < t.nob * t.co;
    int sf[2], st[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int l = l0 + 8 * k + wave;
        sf[k] = oo < O && l < L ? dhf_shift(f.cmax, (int64_t)oo * L + l) : 0;
        st[k] = ii < I && l < L ? dhf_shift(t.cmax, (int64_t)ii * L + l) : 0;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int d = 8 * k + wave, l = l0 + d;
        if (l >= L) break;
        if (has_f) {
            if (ti == 0 && kf == 0) f.cinv[(int64_t)l * (f.nob * f.co) + oo] = __builtin_ldexpf(1.0f, -sf[k]);
            unsigned char* dst = f.packed + (((int64_t)l * f.nob + oo / f.co) * f.nc + ti) * (f.co * 128) + dhf_piece(oo % f.co, kf);
            dhf_store_pieces(dst, f.co, sf[k], 1.f, [&](int e) { return tile[(8 * kf + e) * DHF_PITCH + of * (DHF_PL + 1) + d]; });
        }
        if (has_t) {
            if (to == 0 && ot == 0) t.cinv[(int64_t)l * (t.nob * t.co) + ii] = __builtin_ldexpf(1.0f, -st[k]);
            unsigned char* dst = t.packed + (((int64_t)l * t.nob + ii / t.co) * t.nc + ct) * (t.co * 128) + dhf_piece(ii % t.co, ot & 1);
            dhf_store_pieces(dst, t.co, st[k], -1.f, [&](int e) { return tile[it * DHF_PITCH + (8 * ot + e) * (DHF_PL + 1) + d]; });
        }
    }
}

// weight bytes of a slab here, where twice as much is written; whole groups of 64 degrees
constexpr int64_t DHF_SLAB_BOTH_BYTES = 80 << 20;
int dhconv_pack_both_f16_launch(const float2* w, const sfno_dhconv_weights& fw, const sfno_dhconv_weights& tw, hipStream_t s) {
    const int I = fw.I, O = fw.O, L = fw.L;
    auto stream = [](const sfno_dhconv_weights& h) {
        return DhfStream{reinterpret_cast<unsigned char*>(h.d_W), h.d_cinv, h.d_cmax, h.nob, h.nc, 32 * dhconv_f16_ntc(h.O)};
    };
    const DhfStream f = stream(fw), t = stream(tw);
    const int64_t nti = std::max<int64_t>(f.nc, (int64_t)t.nob * t.co / 16), nto = std::max<int64_t>((int64_t)f.nob * f.co / 32, (t.nc + 1) / 2);
    const int64_t cols = (int64_t)std::max(I, O) * L;
    if (nto > 65535 || (I + 15) / 16 > 65535 || (cols + 255) / 256 > 0x7fffffffLL) return SFNO_EUNSUPPORTED;
    const int64_t per64 = (int64_t)sizeof(float2) * I * O * 64;
    // (a grid has at most 65535 layers of 16 degrees)
    const int slab = 64 * (int)std::max<int64_t>(1, std::min({(int64_t)(L + 63) / 64, DHF_SLAB_BOTH_BYTES / per64, (int64_t)16383}));
    hipLaunchKernelGGL(dhconv_bothmax_clear_kernel, dim3((unsigned)((cols + 255) / 256)), dim3(256), 0, s, fw.d_cmax, (int64_t)O * L, tw.d_cmax, (int64_t)I * L);
    for (int lb = 0; lb < L; lb += slab) {
        const int ln = std::min(slab, L - lb), nl = (ln + DHF_PL - 1) / DHF_PL;
        hipLaunchKernelGGL(dhconv_bothmax_kernel, dim3((O + 15) / 16, (I + 15) / 16, (ln + 63) / 64), dim3(512), 0, s, w, fw.d_cmax, tw.d_cmax, I, O, L, lb, ln);
        hipLaunchKernelGGL(dhconv_pack_both_kernel, dim3((unsigned)nti, (unsigned)nto, nl), dim3(512), 0, s, w, f, t, I, O, L, lb);
    }
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

int dhconv_f16_launch(const DhconvArgs& a, hipStream_t s) {
    const int64_t rows_max = (int64_t)a.M * a.B;
    if (rows_max <= 0 || a.L <= 0) return SFNO_OK;
    if (a.I2 % 4 != 0 || a.ld_in % 4 != 0 || !a.cinv) return SFNO_EUNSUPPORTED;
    const int64_t blocks = dh_blocks(a, 128);
    if (blocks > 0x7fffffffLL) return SFNO_EUNSUPPORTED;
    if (dhconv_f16_ntc(a.O2 / 2) == 4)
        hipLaunchKernelGGL((dhconv_f16_kernel<4>), dim3((unsigned)blocks), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((dhconv_f16_kernel<2>), dim3((unsigned)blocks), dim3(256), 0, s, a);
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

}  // namespace sfno
