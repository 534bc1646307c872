// Pointwise (1x1 convolution) tail of the SFNO block on bf16 MFMA, for bf16 NCHW activations:
//   y[b][o][p] = epilogue( sum_k w[o][k] x[b][k][p] ),   p = pixel (h, w) flattened
// with bias, exact GELU and "+ scale * addend + shift" (instance norm of the addend folded into a
// per-(b, o) affine) fused into the epilogue, plus the two small passes an instance norm needs
// (row statistics -> scale/shift, and scale/shift + activation).  Replaces the nn.Conv2d(k=1) /
// nn.InstanceNorm2d / nn.GELU sequences of makani/models/networks/sfnonet.py:246-262 and
// makani/models/common/layers.py:86-133,136-216 when the activations are bf16.
//
// GEMM kernel.  v_mfma_f32_32x32x16_bf16 wants 8 consecutive k per lane for both operands, but the
// activations are pixel-contiguous.  No transposition is needed: a lane reads 2 consecutive pixels
// (4 bytes) of 8 consecutive k rows and regroups them with byte permutes into two B fragments, one
// per pixel of its pair; MFMA column q of N-tile t then stands for pixel 2q + t, so every lane ends up
// with 2 consecutive pixels of each output row and stores them as one 4-byte piece.
// Two kernels.  Convolutions with at most 96 output channels (pw_gemm_kernel): a wavefront owns 96 rows x 64
// pixels, eight (or, for few pixels, two) wavefronts side by side along the pixels; weights come from global memory (L2 resident) as A
// fragments, packed so that a fragment is 1 KiB of consecutive memory, activations through a triple-buffered LDS
// stage, both prefetched in registers.  All others (pw_gemm_dma_kernel, further down): 128, 256 or 384 rows x 256 pixels per
// workgroup with both operand streams loaded straight into LDS.
#include "sfno_internal.h"
#include <type_traits>

namespace sfno {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

constexpr int PW_MT = 3;          // 32-row tiles per wavefront
constexpr int PW_ROWS = 32 * PW_MT;
constexpr int PW_KC = 16;         // k rows per MFMA K step
constexpr int PW_KS = 2;          // MFMA K steps per chunk (one LDS stage, one barrier)
constexpr int PW_KALIGN = 64;     // K is padded to whole unrolled loop bodies (PW_KC * prefetch distance)

__device__ __forceinline__ float bf16_to_f(unsigned short h) { return __uint_as_float((unsigned int)h << 16); }
__device__ __forceinline__ unsigned short f_to_bf16(float f) { return __builtin_bit_cast(unsigned short, (__bf16)f); }
// two floats rounded to nearest-even bf16 in one word, lo in the low half (the hardware conversion takes a pair: one
// instruction where two single conversions need a shift and an or as well)
__device__ __forceinline__ unsigned int bf16_pair(float lo, float hi) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    typedef float floatx2 __attribute__((ext_vector_type(2)));
    const floatx2 f = {lo, hi};
    return __builtin_bit_cast(unsigned int, __builtin_convertvector(f, bf16x2));
}

// p[i] for a wavefront-uniform i, of an array the kernel never writes: read through the scalar unit, whose loads do not
// count against the vector memory counter
__device__ __forceinline__ float uniform_load(const float* p, int64_t i) {
    return reinterpret_cast<const __attribute__((address_space(4))) float*>(reinterpret_cast<uintptr_t>(p))[i];
}

// exact (erf) GELU for bf16 outputs.  gelu(x) = max(x, 0) - |x| erfc(|x| / sqrt 2) / 2 for both signs (no cancellation in
// the negative tail), and erfc is evaluated as 2^Q(|x|): log2 erfc(t / sqrt 2) is smooth, a degree-6 polynomial in t follows it
// to 1.1e-4 on [0, 6.5] (relative error of erfc 7e-5, a thirtieth of the half ulp of the bf16 result).  Beyond 6.5 t is
// clamped: the term is then below 3e-10 |x| / 6.5 in magnitude, where the formula x (1 + erf(x / sqrt 2)) / 2 in fp32
// arithmetic has long returned -0.  Ten full-rate instructions and one exp2, where a rational form needs a reciprocal as well.
__device__ __forceinline__ float gelu(float x) {
    // (the median of three stands for min and max: one instruction each, where fminf / fmaxf first canonicalise their operand)
    const float t = __builtin_amdgcn_fmed3f(fabsf(x), 0.f, 6.5f);
    float q = fmaf(t, 2.008575651e-05f, -5.615057212e-04f);
    q = fmaf(t, q, 6.880626770e-03f);
    q = fmaf(t, q, -5.027262948e-02f);
    q = fmaf(t, q, -4.624537704e-01f);
    q = fmaf(t, q, -1.149621597e+00f);
    // (the factor 1/2 rides in the exponent: the constant term is the fitted -1.062872110e-04 minus one)
    q = fmaf(t, q, -1.000106287211f);
    return fmaf(-fabsf(x), __builtin_amdgcn_exp2f(q), __builtin_amdgcn_fmed3f(x, 0.f, __builtin_inff()));
}

// The same in training, where the derivative passes through zero and a bf16 result no longer hides the fit above (its error of
// Phi is 4e-5): degree 11, Phi(-|x|) = 2^Q(|x|) to 7e-8 with every step in fp32, what 1 + erf in fp32 gives.
__device__ __forceinline__ float phi_neg(float x) {
    const float t = __builtin_amdgcn_fmed3f(fabsf(x), 0.f, 6.5f);
    float q = fmaf(t, 1.487025059e-09f, -6.108023598e-08f);
    q = fmaf(t, q, 1.104927378e-06f);
    q = fmaf(t, q, -1.145743681e-05f);
    q = fmaf(t, q, 7.265697059e-05f);
    q = fmaf(t, q, -2.514593652e-04f);
    q = fmaf(t, q, -8.251464169e-05f);
    q = fmaf(t, q, 7.073279005e-03f);
    q = fmaf(t, q, -5.254369602e-02f);
    q = fmaf(t, q, -4.591809213e-01f);
    q = fmaf(t, q, -1.151109934e+00f);
    q = fmaf(t, q, -9.999998808e-01f);
    return __builtin_amdgcn_exp2f(q);
}

__device__ __forceinline__ float gelu_train(float x) {
    return fmaf(-fabsf(x), phi_neg(x), __builtin_amdgcn_fmed3f(x, 0.f, __builtin_inff()));
}

// derivative of the GELU: Phi(x) + x phi(x), phi(x) = 2^(-x^2 log2(e) / 2) / sqrt(2 pi)
// (e = phi_neg(x))
__device__ __forceinline__ float gelu_grad(float x, float e) {
    const float phi = 0.39894228040143267794f * __builtin_amdgcn_exp2f(-0.72134752044448170368f * x * x);
    return fmaf(x, phi, x > 0.f ? 1.f - e : e);
}
__device__ __forceinline__ float gelu_grad(float x) { return gelu_grad(x, phi_neg(x)); }

// Training applies both to numbers that were rounded to bf16.  From 2^-11 to the clamp at 6.5 these are 1728 magnitudes, and the convolutions in
// front of and behind a GELU look phi_neg up in LDS: the same bits (but for arguments below 2^-120, whose half may round the other way) with 8 vector
// instructions a value where the GELU takes 18, and 17 where its derivative takes 27.  The vector instructions of the epilogue find no matrix instruction to
// hide behind and bounded both kernels; now memory nearly does, as it does the epilogue with an addend.  721 x 1440: derivative 384 -> 768 channels
// 1258 -> 1136 us, 384 -> 384 645 -> 588, 73 -> 384 425 -> 398; GELU 384 -> 768 1215 -> 1141, 384 -> 384 606 -> 570.  See gelu_table_pays for the others.
constexpr int GT_HI = 0x40d0, GT_N = 1728, GT_LO = GT_HI - GT_N + 1;             // 6.5 as bf16
constexpr int GT_BYTES = 4 * GT_N;
// phi_neg of a bf16 number's magnitude, of the nearest one in the table where it is smaller
__device__ __forceinline__ float gelu_look_up(const unsigned char* table, int magnitude) {
    return *reinterpret_cast<const float*>(table + 4 * (min(max(magnitude, GT_LO), GT_HI) - GT_LO));
}
// gelu_train(x) from the entry of |x|; below the table Phi(-|x|) is a straight line in fp32
__device__ __forceinline__ float gelu_from(float x, int magnitude, float entry) {
    const float e = magnitude < GT_LO ? fmaf(fabsf(x), -0.39894228040143267794f, 0.5f) : entry;
    return fmaf(-fabsf(x), e, __builtin_amdgcn_fmed3f(x, 0.f, __builtin_inff()));
}

// Epilogues: exact GELU on the output and / or "+ scale * addend + shift"; for training GELU_PRE (the output before the GELU is stored as
// well, to a.Z, and activated as stored) and GELU_BWD (the output times the GELU's derivative at `addend`)
// (GELU_PRE | FORMULA: without the table of the direct-to-LDS kernel)
enum { PW_PLAIN = 0, PW_GELU = 1, PW_ADD = 2, PW_GELU_PRE = 4, PW_GELU_BWD = 8, PW_FORMULA = 16 };

// NW = wavefronts per workgroup, side by side along the pixels, 64 pixels each: 8, or 2 where that leaves CUs idle
template <int NW, int EPI>
__global__ __launch_bounds__(64 * NW) void pw_gemm_kernel(PointwiseArgs a) {
    constexpr bool GELU = EPI & (PW_GELU | PW_GELU_PRE), AFF = EPI & PW_ADD, ADD = EPI & (PW_ADD | PW_GELU_BWD);
    constexpr int NT = 2;                         // pixels per lane = N tiles per wavefront
    constexpr int PW_THREADS = 64 * NW;
    constexpr int PW_PX = 32 * NT;                // pixels per wavefront
    constexpr int WPX = NW * PW_PX;               // pixels per workgroup
    constexpr int PITCH = WPX * 2 + 16;           // bytes per LDS row
    constexpr int CK = PW_KC * PW_KS;             // k rows per chunk = per loop step
    constexpr int STAGE = CK * PITCH;
    constexpr int D = 2;                          // prefetch distance in chunks
    constexpr int XW = CK * WPX * 2 / (16 * PW_THREADS);   // 16-byte pieces of the activation chunk per thread
    static_assert(PW_KALIGN % (CK * D) == 0, "loop body divides the padded K");
    static_assert(CK * WPX * 2 == XW * 16 * PW_THREADS, "chunk split evenly over the threads");
    __shared__ __align__(16) unsigned char lds[3 * STAGE];

    const int xcd = blockIdx.x & 7, qid = blockIdx.x >> 3;
    const int ob = qid % a.n_oblk;
    const int64_t strip_lin = (int64_t)(qid / a.n_oblk) * 8 + xcd;
    if (strip_lin >= a.n_strips * a.B) return;
    const int b = (int)(strip_lin / a.n_strips);
    const int64_t pw0 = (strip_lin - (int64_t)b * a.n_strips) * WPX;      // first pixel of the workgroup

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane & 31, ko = lane >> 5;
    const int o0 = ob * PW_ROWS;
    const int pxw = wave * PW_PX;                                         // wavefront's pixel offset inside the stage

    // input channels k < K1 come from X, the others (if any) from X2: a convolution over the concatenation of two tensors
    const int K1 = a.X2 ? a.K1 : a.K;
    const unsigned short* __restrict__ X = a.X + (int64_t)b * K1 * a.P;
    const unsigned short* __restrict__ X2 = a.X2 ? a.X2 + (int64_t)b * (a.K - K1) * a.P : X;
    // this thread's 16-byte pieces (8 pixels of one k row) of an activation chunk of CK rows x WPX pixels
    int xr[XW], loff[XW];
    int64_t xoff[XW];
#pragma unroll
    for (int u = 0; u < XW; ++u) {
        const int e = tid + PW_THREADS * u;
        xr[u] = e / (WPX / 8);
        const int c8 = e - xr[u] * (WPX / 8);
        xoff[u] = min(pw0 + 8 * c8, a.P - 8);                             // past the end: valid pixels, masked at the store
        loff[u] = xr[u] * PITCH + 16 * c8;
    }
    // weight fragments: packed blocks of 32 rows x 16 k, 16 bytes per lane (see pointwise_pack_kernel)
    const int nc16 = a.Kpad / PW_KC;
    const unsigned short* wrow[PW_MT];
#pragma unroll
    for (int mt = 0; mt < PW_MT; ++mt) wrow[mt] = a.W + ((int64_t)(o0 / 32 + mt) * nc16 * 64 + lane) * 8;

    // Kpad is a multiple of CK * D: the unrolled loop below has no conditional steps, which keeps the
    // compiler's count of loads in flight exact (a skipped step would make it wait for nearly all of them)
    const int nchunks = a.Kpad / CK;
    u32x4 araw[D][PW_KS][PW_MT];
    u32x4 xraw[D][XW];

    auto load_a = [&](int c, u32x4 (&dst)[PW_KS][PW_MT]) {
        const int cc = min(c, nchunks - 1);
#pragma unroll
        for (int ks = 0; ks < PW_KS; ++ks)
#pragma unroll
            for (int mt = 0; mt < PW_MT; ++mt) dst[ks][mt] = *reinterpret_cast<const u32x4*>(wrow[mt] + (cc * PW_KS + ks) * 512);
    };
    auto load_x = [&](int c, u32x4 (&dst)[XW]) {
        const int cc = min(c, nchunks - 1);
#pragma unroll
        for (int u = 0; u < XW; ++u) {
            const int k = min(cc * CK + xr[u], a.K - 1);                  // rows past K meet zero weights
            dst[u] = *reinterpret_cast<const u32x4*>((k < K1 ? X + (int64_t)k * a.P : X2 + (int64_t)(k - K1) * a.P) + xoff[u]);
        }
    };
    auto store_x = [&](int stage, const u32x4 (&src)[XW]) {
#pragma unroll
        for (int u = 0; u < XW; ++u) *reinterpret_cast<u32x4*>(&lds[stage * STAGE + loff[u]]) = src[u];
    };

    f32x16 acc[PW_MT][NT];
#pragma unroll
    for (int mt = 0; mt < PW_MT; ++mt)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[mt][t][v] = 0.f;

    // Bias, and the addend's scale and shift, of the wavefront's rows: row r of a 32-row tile in lanes r and r + 32, asked for here, where
    // the wait for the operands covers them.  In the epilogue a vector load between the stores would make every store wait for the one
    // before it (the counter retires in order), and scalar loads, a batch of eight rows at a time, were a chain of twelve round trips.
    // At 721 x 1440, vector loads between the stores / scalar loads / this: 457 -> 73 channels 272 / 300 / 265 us; 64 -> 64 with GELU and
    // addend 198 -> 136, 64 -> 32 83 -> 61.
    float bias[PW_MT], scale[PW_MT], shift[PW_MT];
#pragma unroll
    for (int mt = 0; mt < PW_MT; ++mt) {
        const int r = min(o0 + 32 * mt + q, a.O - 1);
        bias[mt] = a.bias ? a.bias[r] : 0.f;
        scale[mt] = AFF && a.add_scale ? a.add_scale[(int64_t)b * a.O + r] : 1.f;
        shift[mt] = AFF && a.add_shift ? a.add_shift[(int64_t)b * a.O + r] : 0.f;
    }

    // prologue: chunks 0 and 1 into LDS, chunks 2..D+1 of the activations and 0..D-1 of the weights in flight
    {
        u32x4 x0[XW], x1[XW];
        load_x(0, x0);
        load_x(1, x1);
#pragma unroll
        for (int d = 0; d < D; ++d) {
            load_x(d + 2, xraw[(d + 2) % D]);
            load_a(d, araw[d]);
        }
        store_x(0, x0);
        store_x(1, x1);
    }
    __syncthreads();

    // B fragments: lane = pixel group q (NT pixels), k rows 8 ko .. 8 ko + 7 of a 16-row sub-step.  The raw words of the next
    // sub-step are read while the MFMAs of the current one run (hence three stages: chunk c + 1 is read during chunk c).
    typedef unsigned int rw_t __attribute__((ext_vector_type(NT / 2)));
    const unsigned char* fragbase = &lds[0] + (8 * ko) * PITCH + (pxw + NT * q) * 2;
    rw_t rw[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) rw[r] = *reinterpret_cast<const rw_t*>(fragbase + r * PITCH);
    int s0 = 0;                                    // stage of chunk c
    for (int c0 = 0; c0 < nchunks; c0 += D) {
#pragma unroll
        for (int u = 0; u < D; ++u) {
            const int c = c0 + u;
            const int s1 = (s0 == 2) ? 0 : s0 + 1; // stage of chunk c + 1
            const int s2 = (s1 == 2) ? 0 : s1 + 1; // stage of chunk c + 2
#pragma unroll
            for (int ks = 0; ks < PW_KS; ++ks) {
                u32x4 bf[NT];
#pragma unroll
                for (int pp = 0; pp < NT / 2; ++pp)
#pragma unroll
                    for (int h = 0; h < 4; ++h) {
                        bf[2 * pp][h] = __builtin_amdgcn_perm(rw[2 * h + 1][pp], rw[2 * h][pp], 0x05040100u);
                        bf[2 * pp + 1][h] = __builtin_amdgcn_perm(rw[2 * h + 1][pp], rw[2 * h][pp], 0x07060302u);
                    }
                const unsigned char* fb = (ks + 1 < PW_KS) ? fragbase + s0 * STAGE + (ks + 1) * PW_KC * PITCH : fragbase + s1 * STAGE;
#pragma unroll
                for (int r = 0; r < 8; ++r) rw[r] = *reinterpret_cast<const rw_t*>(fb + r * PITCH);
#pragma unroll
                for (int mt = 0; mt < PW_MT; ++mt) {
                    const bf16x8 av = __builtin_bit_cast(bf16x8, araw[u][ks][mt]);
#pragma unroll
                    for (int t = 0; t < NT; ++t)
                        acc[mt][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, __builtin_bit_cast(bf16x8, bf[t]), acc[mt][t], 0, 0, 0);
                }
            }
            // hand chunk c + 2 to its stage, then refill the two register slots
            store_x(s2, xraw[(u + 2) % D]);
            load_x(c + 2 + D, xraw[(u + 2) % D]);
            load_a(c + D, araw[u]);
            __syncthreads();
            s0 = s1;
        }
    }

    // epilogue: lane holds rows 8 (v / 4) + 4 ko + v % 4 of each 32-row tile and pixels 2 q, 2 q + 1.  (Only whole wavefronts leave here:
    // row_value reads every lane.)
    if (pw0 + pxw >= a.P) return;
    const int64_t px = pw0 + pxw + NT * q;
    const bool inside = px < a.P;
    const int64_t pxc = inside ? px : a.P - NT;
    // (no __restrict__: the addend may be the output itself; every value is read, or its batch of rows is, before it is written)
    unsigned short* Y = a.Y + (int64_t)b * a.O * a.P;
    const unsigned short* R = ADD ? a.addend + (int64_t)b * a.O * a.P : nullptr;
    // value of row 8 g + 4 ko + j of a 32-row tile whose lane r holds that of row r
    auto row_value = [&](float v, int g, int j) {
        const int lo = __builtin_amdgcn_readlane(__float_as_int(v), 8 * g + j), hi = __builtin_amdgcn_readlane(__float_as_int(v), 8 * g + 4 + j);
        return __int_as_float(ko ? hi : lo);
    };
#pragma unroll
    for (int mt = 0; mt < PW_MT; ++mt) {
        if (o0 + 32 * mt >= a.O) break;
        rw_t rv[16];
        if constexpr (ADD) {
            // all addend loads of the tile first
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int o = min(o0 + 32 * mt + 8 * (v >> 2) + 4 * ko + (v & 3), a.O - 1);
                rv[v] = *reinterpret_cast<const rw_t*>(R + (int64_t)o * a.P + pxc);
            }
        }
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int o = o0 + 32 * mt + 8 * (v >> 2) + 4 * ko + (v & 3);
            const float bs = row_value(bias[mt], v >> 2, v & 3);
            const float sc = AFF ? row_value(scale[mt], v >> 2, v & 3) : 1.f, sh = AFF ? row_value(shift[mt], v >> 2, v & 3) : 0.f;
            if (o >= a.O || !inside) continue;
            float y0 = acc[mt][0][v] + bs, y1 = acc[mt][1][v] + bs;
            if constexpr (EPI & PW_GELU_PRE) {   // training: the pre-activation is stored as well, and activated as stored
                rw_t zz;
                zz[0] = bf16_pair(y0, y1);
                *reinterpret_cast<rw_t*>(a.Z + (int64_t)b * a.O * a.P + (int64_t)o * a.P + px) = zz;
                y0 = __uint_as_float(zz[0] << 16);
                y1 = __uint_as_float(zz[0] & 0xffff0000u);
            }
            if constexpr (EPI & PW_GELU_PRE) {
                y0 = gelu_train(y0);
                y1 = gelu_train(y1);
            } else if constexpr (GELU) {
                y0 = gelu(y0);
                y1 = gelu(y1);
            }
            if constexpr (EPI & PW_GELU_BWD) {
                y0 *= gelu_grad(__uint_as_float(rv[v][0] << 16));
                y1 *= gelu_grad(__uint_as_float(rv[v][0] & 0xffff0000u));
            }
            if constexpr (AFF) {
                y0 += fmaf(sc, __uint_as_float(rv[v][0] << 16), sh);
                y1 += fmaf(sc, __uint_as_float(rv[v][0] & 0xffff0000u), sh);
            }
            rw_t out;
            out[0] = bf16_pair(y0, y1);
            *reinterpret_cast<rw_t*>(Y + (int64_t)o * a.P + px) = out;
        }
    }
}

// ---- tall variant with direct-to-LDS loads ----------------------------------------------------------
// For O > 96 the kernel above is bound by the weight fragments every wavefront pulls through L1 for only 6 MFMAs
// each.  This variant gives a wavefront up to 96 rows x 128 pixels (3 x 4 tiles, 192 accumulator registers), eight
// wavefronts per workgroup (up to 384 rows x 256 pixels, half the weight traffic per pixel), and moves both operand
// streams with global_load_lds_dwordx4: lane i's 16 bytes land at LDS base + 16 i, no staging registers.
//
// One persistent workgroup per CU walks its tiles as one unbroken stream of 32-row K chunks, so the operands of the
// next tile are already in LDS when the stores of the current one leave.  A read only reaches the HBM rate with
// some 50 KB in flight per CU, and the memory counter of a wavefront retires in order, so a wavefront that waits for
// a weight block (an L2 hit) would also wait for every activation block it asked for earlier.  The two streams
// therefore belong to different wavefronts: wavefronts 0-3 fetch the weights into three stages of 24 KiB, wavefronts
// 4-7 the activations into five stages of 16 KiB; a stage is asked for again as soon as every wavefront has read it, so
// two to three weight chunks and four to five activation chunks (64-80 KiB) are on their way or waiting.  The loads are
// issued from inline assembly (the compiler would order every LDS read behind all outstanding direct-to-LDS loads)
// and the waits are written out by hand.  Other memory operations of a wavefront (the epilogue's stores and addend
// loads) are older than the loads a wait is meant for or younger than all of them; either way the wait covers
// at least the loads it is meant for.
//
// MT = 32-row tiles per wavefront: 128 MT rows per workgroup.  Rows past the matrix are multiplied all the same, so MT follows the
// number of output channels (pointwise_mt); with MT = 1 a workgroup needs half of the registers and, with three activation
// stages, half of the LDS, and two of them share a CU.
constexpr int DM_NT = 4;
constexpr int DM_PX = 2 * 32 * DM_NT;            // 256 pixels per workgroup
constexpr int DM_CK = 32;                        // k rows per chunk
constexpr int DM_XBLK = 1024 + 16;               // two pixel rows of the chunk (2 x 512 bytes) + padding
constexpr int DM_XBYTES = (DM_CK / 2) * DM_XBLK; // activation stage
constexpr int DM_WSTAGES = 3;                    // weight chunks in LDS or on their way
template <int MT>
struct DmGeo {
    static constexpr int ROWS = 4 * 32 * MT;         // rows per workgroup
    static constexpr int ABYTES = 2 * (ROWS / 32) * 1024;   // weight stage: 8 MT fragment blocks of 1 KiB
    static constexpr int XSTAGES = MT == 1 ? 3 : 5;  // activation chunks in LDS or on their way
    static constexpr int XBASE = DM_WSTAGES * ABYTES;
    static constexpr int LDS = XBASE + XSTAGES * DM_XBYTES;
    static constexpr int WG_PER_CU = MT == 1 ? 2 : 1;
    static_assert(WG_PER_CU * LDS <= 160 * 1024, "resident workgroups");
};
// s_waitcnt immediate: at most n vector memory operations in flight, no LDS operation
constexpr int dm_wait(int n) { return (n & 15) | ((n >> 4) << 14) | 0x70; }

// M0 carries the LDS destination.  The compiler refuses "m0" in a clobber list (a reserved register), so nothing may
// keep a value in M0 across this call: the kernels that use it index no register array dynamically and use no
// readlane/movrel/sendmsg around it.
__device__ __forceinline__ void dma16(const void* g, unsigned lds_byte_addr) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(lds_byte_addr) : "memory");
}

// Workgroup barrier of the streaming pipeline: the s_waitcnt in front of it names both counters it depends on (the
// vector-memory count that leaves later chunks in flight, and lgkmcnt(0) for this wavefront's LDS reads of the chunk
// that is about to be overwritten), so the barrier itself is the bare instruction and no fence lowering can add a
// full vmcnt(0) to it.
__device__ __forceinline__ void dm_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
}

template <int MT, int EPI>
__global__ __launch_bounds__(512, 2 * DmGeo<MT>::WG_PER_CU) void pw_gemm_dma_kernel(PointwiseArgs a) {
    using DM = DmGeo<MT>;
    constexpr bool GELU = EPI & (PW_GELU | PW_GELU_PRE), AFF = EPI & PW_ADD, ADD = EPI & (PW_ADD | PW_GELU_BWD);
    constexpr bool TAB = (EPI & (PW_GELU_PRE | PW_GELU_BWD)) && !(EPI & PW_FORMULA);
    static_assert(DM::WG_PER_CU * (DM::LDS + GT_BYTES) <= 160 * 1024, "resident workgroups");
    __shared__ __align__(16) unsigned char lds[DM::LDS + (TAB ? GT_BYTES : 0)];
    // tiles of this XCD, row block fastest: q -> (row block q % n_oblk, strip (q / n_oblk) * 8 + xcd); the workgroups of the
    // XCD deal them out round robin, so the row blocks of one strip run at the same time on one L2
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, nslot = gridDim.x >> 3;
    const int strips = (int)(a.n_strips * a.B);
    const int nq = xcd < strips ? (strips - xcd + 7) / 8 * a.n_oblk : 0;
    if (slot >= nq) return;
    const int ntl = (nq - slot + nslot - 1) / nslot;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wo = wave >> 1, wp = wave & 1;                    // 4 wavefronts along the rows x 2 along the pixels
    const int q = lane & 31, ko = lane >> 5;
    const unsigned lds0 = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)lds);
    const bool wload = wave < 4;                                // this wavefront fetches weights (else activations)
    const int lw = wave & 3;

    const int nc16 = a.Kpad / PW_KC;
    const int nchunks = a.Kpad / DM_CK;
    const int64_t wrb = (int64_t)nc16 * 512;                   // ushorts between row blocks
    // input channels k < K1 come from X, the others (if any) from X2: a convolution over the concatenation of two tensors
    const int K1 = a.X2 ? a.K1 : a.K;

    const unsigned n_oblk = (unsigned)a.n_oblk, n_strips = (unsigned)a.n_strips;
    auto tile_of = [&](int qq, int& ob, int& b, int64_t& pw0) {
        const unsigned sl = (unsigned)qq / n_oblk * 8u + (unsigned)xcd;
        ob = (int)((unsigned)qq % n_oblk);
        b = (int)(sl / n_strips);
        pw0 = (int64_t)(sl - (unsigned)b * n_strips) * DM_PX;
    };

    // load stream of this wavefront: weight blocks (row blocks MT lw .. MT lw + MT - 1 of both 16-row k steps), or activation blocks
    // 4 lw .. 4 lw + 3 (block xb = rows 2 xb, 2 xb + 1 of the chunk; lane = row (lane >> 5), 8 pixels (lane & 31))
    int iq = slot, ic = 0, isg = 0;                             // next chunk to ask for: tile, chunk, stage
    const unsigned short *sp0 = nullptr, *sp1 = nullptr;        // wavefront-uniform bases of the stream's tile
    int voff = lane * 8;                                        // lane's offset from them, in elements
    auto issue = [&]() -> bool {
        if (iq >= nq) return false;
        if (ic == 0) {
            int ob, b;
            int64_t pw0;
            tile_of(iq, ob, b, pw0);
            if (wload) {
                sp0 = a.W + ((int64_t)(ob * (DM::ROWS / 32) + MT * lw) * nc16) * 512;
            } else {
                sp0 = a.X + (int64_t)b * K1 * a.P;
                sp1 = a.X2 ? a.X2 + (int64_t)b * (a.K - K1) * a.P : sp0;
                voff = (int)min(pw0 + 8 * (lane & 31), a.P - 8);
            }
        }
        if (wload) {
            const unsigned sb = lds0 + isg * DM::ABYTES + MT * lw * 1024;
            const unsigned short* src = sp0 + (int64_t)ic * 1024 + voff;
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int i = 0; i < MT; ++i) dma16(src + ks * 512 + i * wrb, sb + (ks * 4 * MT + i) * 1024);
            isg = (isg == DM_WSTAGES - 1) ? 0 : isg + 1;
        } else {
            const unsigned sb = lds0 + DM::XBASE + isg * DM_XBYTES + 4 * lw * DM_XBLK;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                // rows k0 and k0 + 1 for the two halves of the wavefront; rows past K meet zero weights
                const int k0 = min(ic * DM_CK + 8 * lw + 2 * i, a.K - 1), k1 = min(k0 + 1, a.K - 1);
                const unsigned short* r0 = k0 < K1 ? sp0 + (int64_t)k0 * a.P : sp1 + (int64_t)(k0 - K1) * a.P;
                const unsigned short* r1 = k1 < K1 ? sp0 + (int64_t)k1 * a.P : sp1 + (int64_t)(k1 - K1) * a.P;
                dma16((lane >> 5 ? r1 : r0) + voff, sb + i * DM_XBLK);
            }
            isg = (isg == DM::XSTAGES - 1) ? 0 : isg + 1;
        }
        if (++ic == nchunks) {
            ic = 0;
            iq += nslot;
        }
        return true;
    };

    f32x16 acc[MT][DM_NT];

    if constexpr (TAB)
        for (int i = tid; i < GT_BYTES / 4; i += 512) *reinterpret_cast<float*>(lds + DM::LDS + 4 * i) = phi_neg(__uint_as_float((unsigned)(GT_LO + i) << 16));
    // fill the pipeline: three weight chunks or the activation stages, then chunk 0 must have landed
    bool full = true;
    for (int i = 0; i < (wload ? DM_WSTAGES : DM::XSTAGES); ++i) full = issue() && full;
    if (!full)
        __builtin_amdgcn_s_waitcnt(dm_wait(0));
    else if (wload)
        __builtin_amdgcn_s_waitcnt(dm_wait(2 * 2 * MT));               // the two later weight chunks
    else
        __builtin_amdgcn_s_waitcnt(dm_wait(4 * (DM::XSTAGES - 1)));    // the later activation chunks
    dm_barrier();

    const unsigned char* abase = lds + (MT * wo) * 1024 + lane * 16;
    const unsigned char* xbase = lds + DM::XBASE + (4 * ko) * DM_XBLK + wp * 256 + 8 * q;
    int sw = 0, sx = 0;
    // Operands of a 16-row k step: eight raw words of activations (rw), regrouped by byte permutes into the four B fragments
    // (bf), and three A fragments (af).  The LDS reads of the next k step are issued into rw and af as soon as the current
    // step has consumed them (rw after the permutes, af[mt] after the MFMAs of row tile mt), so they run under the MFMAs.
    u32x2 rw[8];
    u32x4 af[MT], bf[DM_NT];
    auto load_rw = [&](const unsigned char* sxp, int ks) {
#pragma unroll
        for (int r = 0; r < 8; ++r) rw[r] = *reinterpret_cast<const u32x2*>(sxp + (8 * ks + (r >> 1)) * DM_XBLK + (r & 1) * 512);
    };
    auto load_af = [&](const unsigned char* sa, int ks, int mt) { af[mt] = *reinterpret_cast<const u32x4*>(sa + (ks * 4 * MT + mt) * 1024); };
    auto regroup = [&]() {
#pragma unroll
        for (int pp = 0; pp < 2; ++pp)
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                bf[2 * pp][h] = __builtin_amdgcn_perm(rw[2 * h + 1][pp], rw[2 * h][pp], 0x05040100u);
                bf[2 * pp + 1][h] = __builtin_amdgcn_perm(rw[2 * h + 1][pp], rw[2 * h][pp], 0x07060302u);
            }
    };
    // (the first k step of a tile starts its sums from the constant zero: no pass over the 192 accumulators between tiles)
    auto mfma_row = [&](int mt, bool first) {
        const bf16x8 av = __builtin_bit_cast(bf16x8, af[mt]);
        if (first) {
            const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int t = 0; t < DM_NT; ++t)
                acc[mt][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, __builtin_bit_cast(bf16x8, bf[t]), zero, 0, 0, 0);
        } else {
#pragma unroll
            for (int t = 0; t < DM_NT; ++t)
                acc[mt][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, __builtin_bit_cast(bf16x8, bf[t]), acc[mt][t], 0, 0, 0);
        }
    };

    // Epilogue of one tile, a quarter of a row tile (eight rows, of which a lane has the four of its half ko) at a time.
    // Bias and the addend's scale and shift come through the scalar unit, the eight rows in one batch ahead of the four
    // stores: a vector load between the stores would make each store wait for the one before, since the wait for the load
    // covers every store issued before it.  The addend itself is read half a row tile ahead.
    auto epilogue = [&](auto whole, int o0, int ko4, int b, int64_t lane_off) {
        constexpr bool WHOLE = decltype(whole)::value;
        unsigned short* Y = a.Y + lane_off;                                     // (may be the addend itself, as above)
        const unsigned short* R = ADD ? a.addend + lane_off : nullptr;
        auto row_of = [&](int mt, int v) { return 32 * mt + 8 * (v >> 2) + (v & 3); };     // without the lane's 4 ko
        u32x2 rv[2][8];
        auto load_addend = [&](int mh) {
            if constexpr (ADD) {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    int r = row_of(mh >> 1, 8 * (mh & 1) + j);
                    if (!WHOLE) r = min(r, a.O - 1 - o0 - ko4);
                    rv[mh & 1][j] = *reinterpret_cast<const u32x2*>(R + (int64_t)r * a.P);
                }
            }
        };
        // scalar loads one quarter ahead: those of quarter q + 1 are issued once those of quarter q have arrived (the wait of the
        // scalar unit is for all of its loads at once), and are under way while quarter q is converted and stored
        float ub[2][8], usc[2][8], ush[2][8];
        auto load_scalars = [&](int qq) {
            const int oq = o0 + row_of(qq >> 2, 4 * (qq & 3));   // rows oq .. oq + 7 (ko = 0: oq .. oq + 3)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int64_t u = WHOLE ? oq + i : min(oq + i, a.O - 1);
                ub[qq & 1][i] = a.bias ? uniform_load(a.bias, u) : 0.f;
                usc[qq & 1][i] = (AFF && a.add_scale) ? uniform_load(a.add_scale, (int64_t)b * a.O + u) : 1.f;
                ush[qq & 1][i] = (AFF && a.add_shift) ? uniform_load(a.add_shift, (int64_t)b * a.O + u) : 0.f;
            }
        };
        load_addend(0);
        load_scalars(0);
#pragma unroll
        for (int mh = 0; mh < 2 * MT; ++mh) {
            const int mt = mh >> 1;
            if (!WHOLE && o0 + 32 * mt >= a.O) break;
            if (mh + 1 < 2 * MT && (WHOLE || o0 + 32 * ((mh + 1) >> 1) < a.O)) load_addend(mh + 1);
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                const int qq = 2 * mh + g;
                const int v0 = 8 * (mh & 1) + 4 * g;
                const int oq = o0 + row_of(mt, v0);
                asm volatile("" ::"s"(ub[qq & 1][0]), "s"(ub[qq & 1][7]));       // the wait for this quarter's scalars goes here
                __builtin_amdgcn_sched_barrier(0);
                if (qq + 1 < 4 * MT) load_scalars(qq + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) {
                    const int v = v0 + jj;
                    if (!WHOLE && oq + ko4 + jj >= a.O) continue;
                    const float bs = ko4 ? ub[qq & 1][4 + jj] : ub[qq & 1][jj];
                    float y[4];
#pragma unroll
                    for (int t = 0; t < 4; ++t) y[t] = acc[mt][t][v] + bs;
                    if constexpr (EPI & PW_GELU_PRE) {
                        u32x2 z;
                        float e[4];
#pragma unroll
                        for (int pp = 0; pp < 2; ++pp) {
                            z[pp] = bf16_pair(y[2 * pp], y[2 * pp + 1]);
                            if constexpr (TAB) {
                                e[2 * pp] = gelu_look_up(lds + DM::LDS, z[pp] & 0x7fffu);
                                e[2 * pp + 1] = gelu_look_up(lds + DM::LDS, z[pp] >> 16 & 0x7fffu);
                            }
                        }
                        *reinterpret_cast<u32x2*>(a.Z + lane_off + (int64_t)row_of(mt, v) * a.P) = z;
#pragma unroll
                        for (int pp = 0; pp < 2; ++pp) {
                            const float u = __uint_as_float(z[pp] << 16), w = __uint_as_float(z[pp] & 0xffff0000u);
                            y[2 * pp] = TAB ? gelu_from(u, z[pp] & 0x7fffu, e[2 * pp]) : gelu_train(u);
                            y[2 * pp + 1] = TAB ? gelu_from(w, z[pp] >> 16 & 0x7fffu, e[2 * pp + 1]) : gelu_train(w);
                        }
                    } else if constexpr (GELU) {
#pragma unroll
                        for (int t = 0; t < 4; ++t) y[t] = gelu(y[t]);
                    }
                    if constexpr (EPI & PW_GELU_BWD) {
                        const u32x2 r = rv[mh & 1][4 * g + jj];
                        float e[4], x[4];
                        int m[4];
#pragma unroll
                        for (int t = 0; t < 4; ++t) {
                            m[t] = r[t >> 1] >> 16 * (t & 1) & 0x7fffu;
                            x[t] = __uint_as_float(t & 1 ? r[t >> 1] & 0xffff0000u : r[t >> 1] << 16);
                            e[t] = gelu_look_up(lds + DM::LDS, m[t]);
                        }
                        // (one value in two thousand is below the table, one group of 256 in ten has such a value)
                        if (__builtin_amdgcn_ballot_w64(min(min(m[0], m[1]), min(m[2], m[3])) < GT_LO)) {
#pragma unroll
                            for (int t = 0; t < 4; ++t) e[t] = phi_neg(x[t]);
                        }
#pragma unroll
                        for (int t = 0; t < 4; ++t) y[t] *= gelu_grad(x[t], e[t]);
                    }
                    if constexpr (AFF) {
                        const float sc = ko4 ? usc[qq & 1][4 + jj] : usc[qq & 1][jj], sh = ko4 ? ush[qq & 1][4 + jj] : ush[qq & 1][jj];
                        const u32x2 r = rv[mh & 1][4 * g + jj];
#pragma unroll
                        for (int pp = 0; pp < 2; ++pp) {
                            y[2 * pp] += fmaf(sc, __uint_as_float(r[pp] << 16), sh);
                            y[2 * pp + 1] += fmaf(sc, __uint_as_float(r[pp] & 0xffff0000u), sh);
                        }
                    }
                    u32x2 out;
#pragma unroll
                    for (int pp = 0; pp < 2; ++pp) out[pp] = bf16_pair(y[2 * pp], y[2 * pp + 1]);
                    *reinterpret_cast<u32x2*>(Y + (int64_t)row_of(mt, v) * a.P) = out;
                }
            }
        }
    };

    for (int tl = 0; tl < ntl; ++tl) {
        const unsigned char* sa = abase + sw * DM::ABYTES;
        const unsigned char* sxp = xbase + sx * DM_XBYTES;
        load_rw(sxp, 0);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) load_af(sa, 0, mt);
        for (int c = 0; c < nchunks; ++c) {
            // first k step of the chunk; the second one's operands follow it into the registers
            regroup();
            __builtin_amdgcn_sched_barrier(0);
            load_rw(sxp, 1);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                mfma_row(mt, c == 0);
                __builtin_amdgcn_sched_barrier(0);
                load_af(sa, 1, mt);
                __builtin_amdgcn_sched_barrier(0);
            }
            regroup();
            // Every wavefront has read all of this chunk.  The next chunk must have landed for every wavefront before it is
            // read; in flight may stay the loads of one weight chunk (2 MT) or of all but two of the activation chunks (4 each),
            // nothing once the stream has run dry.  Then this chunk's stages take the chunk that many stages further on.
            if (!full)
                __builtin_amdgcn_s_waitcnt(dm_wait(0));
            else if (wload)
                __builtin_amdgcn_s_waitcnt(dm_wait(2 * MT));
            else
                __builtin_amdgcn_s_waitcnt(dm_wait(4 * (DM::XSTAGES - 2)));
            dm_barrier();
            full = issue();
            sw = (sw == DM_WSTAGES - 1) ? 0 : sw + 1;
            sx = (sx == DM::XSTAGES - 1) ? 0 : sx + 1;
            sa = abase + sw * DM::ABYTES;
            sxp = xbase + sx * DM_XBYTES;
            // second k step; the first one of the next chunk follows (after the last chunk of a tile these reads are
            // repeated behind the epilogue, which needs the registers)
            __builtin_amdgcn_sched_barrier(0);
            load_rw(sxp, 0);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                mfma_row(mt, false);
                __builtin_amdgcn_sched_barrier(0);
                load_af(sa, 0, mt);
                __builtin_amdgcn_sched_barrier(0);
            }
        }

        // epilogue: lane holds rows 8 (v / 4) + 4 ko + v % 4 of each 32-row tile and pixels 4 q .. 4 q + 3
        int ob, b;
        int64_t pw0;
        tile_of(slot + tl * nslot, ob, b, pw0);
        // (derived afresh for every tile: hoisted out of the tile loop, the row offsets of a lane and its addresses would
        // occupy registers the accumulators need)
        int lane_ = lane;
        asm volatile("" : "+v"(lane_));
        const int ko4 = (lane_ >> 5) * 4;
        const int o0 = ob * DM::ROWS + wo * 32 * MT;          // first row of the wavefront
        const int64_t px = pw0 + wp * 128 + 4 * (lane_ & 31);
        if (px < a.P && o0 < a.O) {
            const int64_t lane_off = ((int64_t)b * a.O + o0 + ko4) * a.P + px;      // lane's first row
            // whole wavefront tile inside the matrix: no row needs a check or a clamp
            if (o0 + 32 * MT <= a.O)
                epilogue(std::true_type{}, o0, ko4, b, lane_off);
            else
                epilogue(std::false_type{}, o0, ko4, b, lane_off);
        }
    }
}

// packed[rb][c][lane][e] = bf16(w[32 rb + (lane & 31)][16 c + 8 (lane >> 5) + e]), zero outside the O x K weight:
// the A fragment of one wavefront for row block rb and chunk c is 1 KiB of consecutive memory (transposed: w is [K][O])
__device__ __forceinline__ void pack_element(const float* __restrict__ w, unsigned short* __restrict__ packed, int O, int K, int nc, int64_t idx,
                                             int transposed) {
    const int e = (int)(idx & 7), lane = (int)((idx >> 3) & 63);
    const int64_t blk = idx >> 9;
    const int c = (int)(blk % nc), rb = (int)(blk / nc);
    const int o = 32 * rb + (lane & 31), k = 16 * c + 8 * (lane >> 5) + e;
    packed[idx] = (o < O && k < K) ? f_to_bf16(w[transposed ? (int64_t)k * O + o : (int64_t)o * K + k]) : (unsigned short)0;
}
__global__ __launch_bounds__(256) void pointwise_pack_kernel(const float* __restrict__ w, unsigned short* __restrict__ packed, int O, int K, int nc,
                                                             int64_t total, int transposed) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx < total) pack_element(w, packed, O, K, nc, idx, transposed);
}
// A weight and its transpose for a training step: a launch of 3 us instead of two (nothing but launches at these sizes).
__global__ __launch_bounds__(256) void pointwise_pack_both_kernel(const float* __restrict__ w, unsigned short* __restrict__ packed, int nc, int64_t total,
                                                                  unsigned short* __restrict__ packed_t, int nc_t, int64_t total_t, int O, int K) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx < total)
        pack_element(w, packed, O, K, nc, idx, 0);
    else if (idx < total + total_t)
        pack_element(w, packed_t, K, O, nc_t, idx - total, 1);
}

// The merged layer W (scale . m + shift) + W W_skip r + bias of a network's tail (O x K weight W), for every sample b: packed[b], the stream of
// [W diag(scale_b) | W W_skip] as pack_element writes it, and shifted[b] = W shift_b + bias.  The first blocks of a sample pack, the others
// take four output rows each, a wavefront one (lanes over k, sums folded in halves).  grid (pack + ceil(O / 4), samples, at most 256).  Nothing but latency at
// these sizes; as separate products, concatenation, matrix product, sum and packing it was eleven launches and 70 us a call.
__global__ __launch_bounds__(256) void pointwise_merge_kernel(const float* __restrict__ w, const float* __restrict__ ws, const float* __restrict__ scale,
                                                              const float* __restrict__ shift, const float* __restrict__ bias,
                                                              unsigned short* __restrict__ packed, float* __restrict__ shifted, int O, int K, int B,
                                                              int nc, int64_t total, int pack) {
    if ((int)blockIdx.x < pack) {
        const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
        if (idx >= total) return;
        const int e = (int)(idx & 7), lane = (int)((idx >> 3) & 63);
        const int64_t blk = idx >> 9;
        const int c = (int)(blk % nc), rb = (int)(blk / nc);
        const int o = 32 * rb + (lane & 31), k = 16 * c + 8 * (lane >> 5) + e;
        for (int b = blockIdx.y; b < B; b += gridDim.y) {
            float v = 0.f;
            if (o < O && k < K)
                v = scale ? w[(int64_t)o * K + k] * scale[(int64_t)b * K + k] : w[(int64_t)o * K + k];
            else if (o < O && k < 2 * K)
                v = ws[(int64_t)o * K + k - K];
            packed[b * total + idx] = f_to_bf16(v);
        }
        return;
    }
    const int o = 4 * ((int)blockIdx.x - pack) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (o >= O) return;
    for (int b = blockIdx.y; b < B; b += gridDim.y) {
        float sum = 0.f;
        if (shift)
            for (int k = lane; k < K; k += 64) sum = fmaf(w[(int64_t)o * K + k], shift[(int64_t)b * K + k], sum);
#pragma unroll
        for (int d = 32; d; d >>= 1) sum += __shfl_xor(sum, d);
        if (lane == 0) shifted[(int64_t)b * O + o] = bias ? sum + bias[o] : sum;
    }
}

// ---- instance-norm statistics ------------------------------------------------------------------
// partial[row][seg] = (sum d, sum d^2), d = x - x[row][0] (the pivot keeps the variance formula from cancelling)
constexpr int ST_THREADS = 256;
__global__ __launch_bounds__(ST_THREADS) void row_stats_partial_kernel(const unsigned short* __restrict__ x, float2* __restrict__ partial, int64_t P,
                                                                       int nseg) {
    const int64_t row = blockIdx.x;
    const int seg = blockIdx.y;
    const unsigned short* __restrict__ xr = x + row * P;
    const float pivot = bf16_to_f(xr[0]);
    const int64_t ngroups = P / 8;
    const int64_t g0 = ngroups * seg / nseg, g1 = ngroups * (seg + 1) / nseg;
    float s = 0.f, s2 = 0.f;
    for (int64_t g = g0 + threadIdx.x; g < g1; g += ST_THREADS) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(xr + 8 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float lo = __uint_as_float(v[i] << 16) - pivot, hi = __uint_as_float(v[i] & 0xffff0000u) - pivot;
            s += lo + hi;
            s2 = fmaf(lo, lo, fmaf(hi, hi, s2));
        }
    }
    if (seg == nseg - 1)
        for (int64_t i = 8 * ngroups + threadIdx.x; i < P; i += ST_THREADS) {
            const float d = bf16_to_f(xr[i]) - pivot;
            s += d;
            s2 = fmaf(d, d, s2);
        }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        s += __shfl_down(s, off, 64);
        s2 += __shfl_down(s2, off, 64);
    }
    __shared__ float2 red[ST_THREADS / 64];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = make_float2(s, s2);
    __syncthreads();
    if (threadIdx.x == 0) {
        float2 t = red[0];
        for (int w = 1; w < ST_THREADS / 64; ++w) {
            t.x += red[w].x;
            t.y += red[w].y;
        }
        partial[row * nseg + seg] = t;
    }
}

// scale = gamma * rstd, shift = beta - mean * scale  (biased variance, as torch.nn.functional.instance_norm)
__global__ void row_stats_finalize_kernel(const unsigned short* __restrict__ x, const float2* __restrict__ partial, const float* __restrict__ gamma,
                                          const float* __restrict__ beta, float* __restrict__ scale, float* __restrict__ shift,
                                          float2* __restrict__ moments, int64_t rows, int channels, int64_t P, int nseg, float eps) {
    const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= rows) return;
    double s = 0.0, s2 = 0.0;
    for (int i = 0; i < nseg; ++i) {
        s += partial[row * nseg + i].x;
        s2 += partial[row * nseg + i].y;
    }
    const double n = (double)P;
    const double md = s / n;
    const double var = fmax(s2 / n - md * md, 0.0);
    const float mean = bf16_to_f(x[row * P]) + (float)md;
    const float rstd = (float)(1.0 / sqrt(var + (double)eps));
    const int c = (int)(row % channels);
    const float sc = (gamma ? gamma[c] : 1.f) * rstd;
    scale[row] = sc;
    shift[row] = (beta ? beta[c] : 0.f) - mean * sc;
    if (moments) moments[row] = make_float2(mean, rstd);
}

// The same in one kernel for short rows (P <= NORM_SMALL_PIXELS): a wavefront per row, its values in registers, mean first and then the
// moments of the deviations from it.
constexpr int SS_GROUPS = 8;                                  // groups of eight pixels per lane
static_assert(SS_GROUPS * 64 * 8 == NORM_SMALL_PIXELS, "a row fits the registers of a wavefront");
__global__ __launch_bounds__(64) void row_stats_small_kernel(const unsigned short* __restrict__ x, const float* __restrict__ gamma,
                                                             const float* __restrict__ beta, float* __restrict__ scale, float* __restrict__ shift,
                                                             float2* __restrict__ moments, int channels, int P, float eps) {
    const int64_t row = blockIdx.x;
    const u32x4* __restrict__ xr = reinterpret_cast<const u32x4*>(x + row * P);
    const int ngroups = P / 8;
    u32x4 v[SS_GROUPS];
#pragma unroll
    for (int k = 0; k < SS_GROUPS; ++k) {
        const int g = (int)threadIdx.x + 64 * k;
        if (g < ngroups) v[k] = xr[g];
    }
    auto sums = [&](float about, float& s, float& s2) {
        s = s2 = 0.f;
#pragma unroll
        for (int k = 0; k < SS_GROUPS; ++k) {
            if ((int)threadIdx.x + 64 * k >= ngroups) break;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float lo = __uint_as_float(v[k][i] << 16) - about, hi = __uint_as_float(v[k][i] & 0xffff0000u) - about;
                s += lo + hi;
                s2 = fmaf(lo, lo, fmaf(hi, hi, s2));
            }
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            s += __shfl_xor(s, off, 64);
            s2 += __shfl_xor(s2, off, 64);
        }
    };
    float s, s2;
    sums(0.f, s, s2);
    const float about = s / (float)P;
    sums(about, s, s2);
    if (threadIdx.x == 0) {
        const double md = (double)s / P, var = fmax((double)s2 / P - md * md, 0.0);
        const float mean = about + (float)md, rstd = (float)(1.0 / sqrt(var + (double)eps));
        const int c = (int)(row % channels);
        const float sc = (gamma ? gamma[c] : 1.f) * rstd;
        scale[row] = sc;
        shift[row] = (beta ? beta[c] : 0.f) - mean * sc;
        if (moments) moments[row] = make_float2(mean, rstd);
    }
}

// The same coefficients from per-latitude moments of the field (the inverse longitude kernel's by-product):
// stats[row][k] = (a_k, d_k), the mean over longitude of latitude row k and of its squared deviation from a_k.
// mean = avg_k a_k, variance = avg_k ((a_k - mean)^2 + d_k); one wavefront per row, sums in double.
__global__ __launch_bounds__(64) void lat_stats_finalize_kernel(const float2* __restrict__ stats, const float* __restrict__ gamma,
                                                                const float* __restrict__ beta, float* __restrict__ scale, float* __restrict__ shift,
                                                                float2* __restrict__ moments, int channels, int nlat, float eps) {
    const int64_t row = blockIdx.x;
    const float2* __restrict__ sr = stats + row * nlat;
    double s = 0.0;
    for (int k = threadIdx.x; k < nlat; k += 64) s += (double)sr[k].x;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    const double mean = s / nlat;
    double v = 0.0;
    for (int k = threadIdx.x; k < nlat; k += 64) {
        const float2 t = sr[k];
        const double d = (double)t.x - mean;
        v += d * d + (double)t.y;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if (threadIdx.x == 0) {
        const float rstd = (float)(1.0 / sqrt(v / nlat + (double)eps));
        const int c = (int)(row % channels);
        const float sc = (gamma ? gamma[c] : 1.f) * rstd;
        scale[row] = sc;
        shift[row] = (beta ? beta[c] : 0.f) - (float)mean * sc;
        if (moments) moments[row] = make_float2((float)mean, rstd);
    }
}

// y = act(scale[row] * x + shift[row]), bf16 -> bf16, 8 pixels per thread; y may be x
__global__ __launch_bounds__(256) void scale_shift_act_kernel(const unsigned short* x, const float* __restrict__ scale,
                                                              const float* __restrict__ shift, unsigned short* y, int64_t P,
                                                              int64_t groups_per_row, int64_t total_groups, int act) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= total_groups) return;
    const int64_t row = g / groups_per_row;
    const int64_t i0 = row * P + 8 * (g - row * groups_per_row);
    const float sc = scale[row], sh = shift[row];
    const u32x4 v = *reinterpret_cast<const u32x4*>(x + i0);
    u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float lo = fmaf(sc, __uint_as_float(v[i] << 16), sh), hi = fmaf(sc, __uint_as_float(v[i] & 0xffff0000u), sh);
        if (act == SFNO_ACT_GELU) {
            lo = gelu(lo);
            hi = gelu(hi);
        } else if (act == ACT_GELU_TRAIN) {
            lo = gelu_train(lo);
            hi = gelu_train(hi);
        }
        o[i] = bf16_pair(lo, hi);
    }
    *reinterpret_cast<u32x4*>(y + i0) = o;
}

// ---- backward of y = act(scale * x + shift), scale and shift from the row's own statistics (instance norm) ------
// With d = g act'(scale x + shift) and xh = (x - mean) rstd:   dx = scale (d - avg d - xh avg(d xh)),   dgamma = sum d xh,   dbeta = sum d.
// Two passes over (g, x), 8 pixels per thread and step: the first leaves partial[row][seg] = (sum d, sum d xh), the second adds them up per
// row and writes dx; norm_param_grad_kernel adds them up per channel.  Bound by memory: five tensor passes in all (two of them writes
// and reads of nothing else), with the activation's derivative computed twice instead of a tensor written between the passes.
__device__ __forceinline__ void norm_terms(unsigned gw, unsigned xw, bool act, float sc, float sh, float mean, float rstd, float (&d)[2], float (&xh)[2]) {
    const float x[2] = {__uint_as_float(xw << 16), __uint_as_float(xw & 0xffff0000u)};
    d[0] = __uint_as_float(gw << 16);
    d[1] = __uint_as_float(gw & 0xffff0000u);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        xh[i] = (x[i] - mean) * rstd;
        if (act) d[i] *= gelu_grad(fmaf(sc, x[i], sh));
    }
}

template <bool ACT>
__global__ __launch_bounds__(ST_THREADS) void norm_grad_reduce_kernel(const unsigned short* __restrict__ g, const unsigned short* __restrict__ x,
                                                                      const float* __restrict__ scale, const float* __restrict__ shift,
                                                                      const float2* __restrict__ moments, float2* __restrict__ partial, int64_t P, int nseg) {
    const int64_t row = blockIdx.x;
    const int seg = blockIdx.y;
    const float sc = scale[row], sh = shift[row];
    const float2 mo = moments[row];
    const int64_t ngroups = P / 8;
    const int64_t g0 = ngroups * seg / nseg, g1 = ngroups * (seg + 1) / nseg;
    float s = 0.f, s2 = 0.f;
    for (int64_t i = g0 + threadIdx.x; i < g1; i += ST_THREADS) {
        const u32x4 gv = *reinterpret_cast<const u32x4*>(g + row * P + 8 * i), xv = *reinterpret_cast<const u32x4*>(x + row * P + 8 * i);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            float d[2], xh[2];
            norm_terms(gv[w], xv[w], ACT, sc, sh, mo.x, mo.y, d, xh);
            s += d[0] + d[1];
            s2 = fmaf(d[0], xh[0], fmaf(d[1], xh[1], s2));
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        s += __shfl_down(s, off, 64);
        s2 += __shfl_down(s2, off, 64);
    }
    __shared__ float2 red[ST_THREADS / 64];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = make_float2(s, s2);
    __syncthreads();
    if (threadIdx.x == 0) {
        float2 t = red[0];
        for (int w = 1; w < ST_THREADS / 64; ++w) {
            t.x += red[w].x;
            t.y += red[w].y;
        }
        partial[row * nseg + seg] = t;
    }
}

template <bool ACT>
__global__ __launch_bounds__(ST_THREADS) void norm_grad_apply_kernel(const unsigned short* __restrict__ g, const unsigned short* __restrict__ x,
                                                                     const float* __restrict__ scale, const float* __restrict__ shift,
                                                                     const float2* __restrict__ moments, const float2* __restrict__ partial,
                                                                     unsigned short* __restrict__ dx, int64_t P, int nseg) {
    const int64_t row = blockIdx.x;
    const int seg = blockIdx.y;
    __shared__ float2 total;
    if (threadIdx.x < 64) {                      // nseg <= 64
        float2 t = make_float2(0.f, 0.f);
        if ((int)threadIdx.x < nseg) t = partial[row * nseg + threadIdx.x];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            t.x += __shfl_xor(t.x, off, 64);
            t.y += __shfl_xor(t.y, off, 64);
        }
        if (threadIdx.x == 0) total = t;
    }
    __syncthreads();
    const float sc = scale[row], sh = shift[row];
    const float2 mo = moments[row];
    const float m1 = total.x / (float)P, m2 = total.y / (float)P;
    const int64_t ngroups = P / 8;
    const int64_t g0 = ngroups * seg / nseg, g1 = ngroups * (seg + 1) / nseg;
    for (int64_t i = g0 + threadIdx.x; i < g1; i += ST_THREADS) {
        const u32x4 gv = *reinterpret_cast<const u32x4*>(g + row * P + 8 * i), xv = *reinterpret_cast<const u32x4*>(x + row * P + 8 * i);
        u32x4 o;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            float d[2], xh[2];
            norm_terms(gv[w], xv[w], ACT, sc, sh, mo.x, mo.y, d, xh);
            o[w] = bf16_pair(sc * (d[0] - fmaf(xh[0], m2, m1)), sc * (d[1] - fmaf(xh[1], m2, m1)));
        }
        *reinterpret_cast<u32x4*>(dx + row * P + 8 * i) = o;
    }
}

// one wavefront per channel: dgamma and dbeta from the partial sums of its rows
__global__ __launch_bounds__(64) void norm_param_grad_kernel(const float2* __restrict__ partial, float* __restrict__ dgamma, float* __restrict__ dbeta, int batch,
                                                             int channels, int nseg) {
    const int c = blockIdx.x;
    double s = 0.0, s2 = 0.0;
    for (int i = threadIdx.x; i < batch * nseg; i += 64) {
        const float2 t = partial[((int64_t)(i / nseg) * channels + c) * nseg + i % nseg];
        s += t.x;
        s2 += t.y;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        s += __shfl_down(s, off, 64);
        s2 += __shfl_down(s2, off, 64);
    }
    if (threadIdx.x == 0) {
        if (dgamma) dgamma[c] = (float)s2;
        if (dbeta) dbeta[c] = (float)s;
    }
}

#include "pointwise_mlp.h"

}  // namespace

int device_cus() {
    static int cached[64] = {};
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) { (void)hipGetLastError(); return 256; }
    if (cached[dev] > 0) return cached[dev];
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) { (void)hipGetLastError(); return 256; }
    cached[dev] = cus;
    return cus;
}

// the kernel for O > 96 walks K in chunks of 32 rows and takes any number of them; the other one runs whole unrolled loop bodies
int pointwise_kpad(int K, int O) {
    const int align = O > PW_ROWS ? DM_CK : PW_KALIGN;
    return (K + align - 1) / align * align;
}
// 32-row tiles per wavefront of the direct-to-LDS kernel: the fewest multiplied rows, a block of rows counted 96 rows more for
// streaming the activations once more (O = 128: one block of 128, 256: of 256, 384 and 768: of 384, 512: two of 256, 640: two of 384)
static int pointwise_mt(int O) {
    int best = 3, cost = 1 << 30;
    for (int mt = 3; mt >= 1; --mt) {
        const int blocks = (O + 128 * mt - 1) / (128 * mt), c = blocks * (128 * mt + 96);
        if (c < cost) { cost = c; best = mt; }
    }
    return best;
}
// rows are padded to whole workgroup tiles so that no fragment load needs a bound check
int pointwise_opad(int O) {
    const int tile = O > PW_ROWS ? 128 * pointwise_mt(O) : PW_ROWS;
    return (O + tile - 1) / tile * tile;
}

int pointwise_pack_launch(const float* w, unsigned short* packed, int O, int K, int transposed, hipStream_t s) {
    const int nc = pointwise_kpad(K, O) / PW_KC;
    const int64_t total = (int64_t)(pointwise_opad(O) / 32) * nc * 512;
    const int64_t blocks = (total + 255) / 256;
    if (blocks > 0x7fffffffLL) return SFNO_EUNSUPPORTED;
    hipLaunchKernelGGL(pointwise_pack_kernel, dim3((unsigned)blocks), dim3(256), 0, s, w, packed, O, K, nc, total, transposed);
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

int pointwise_pack_both_launch(const float* w, unsigned short* packed, unsigned short* packed_t, int O, int K, hipStream_t s) {
    const int nc = pointwise_kpad(K, O) / PW_KC, nc_t = pointwise_kpad(O, K) / PW_KC;
    const int64_t total = (int64_t)(pointwise_opad(O) / 32) * nc * 512, total_t = (int64_t)(pointwise_opad(K) / 32) * nc_t * 512;
    const int64_t blocks = (total + total_t + 255) / 256;
    if (blocks > 0x7fffffffLL) return SFNO_EUNSUPPORTED;
    hipLaunchKernelGGL(pointwise_pack_both_kernel, dim3((unsigned)blocks), dim3(256), 0, s, w, packed, nc, total, packed_t, nc_t, total_t, O, K);
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

int pointwise_merge_launch(const float* w, const float* ws, const float* scale, const float* shift, const float* bias, unsigned short* packed, float* shifted,
                           int O, int K, int B, hipStream_t s) {
    const int nc = pointwise_kpad(2 * K, O) / PW_KC;
    const int64_t total = (int64_t)(pointwise_opad(O) / 32) * nc * 512, pack = (total + 255) / 256, blocks = pack + (O + 3) / 4;
    if (blocks > 0x7fffffffLL) return SFNO_EUNSUPPORTED;
    hipLaunchKernelGGL(pointwise_merge_kernel, dim3((unsigned)blocks, (unsigned)std::min(B, 256)), dim3(256), 0, s, w, ws, scale, shift, bias, packed, shifted, O, K,
                       B, nc, total, (int)pack);
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

// Whether the GELU of a training convolution takes Phi from the table (its derivative always does).  Not where the formula's instructions already hide behind the
// stores, the faster epilogue is then up to 10 % the slower one: few chunks of 32 input channels and outputs far beyond the memory-side cache
// (256 MB).  Rows that begin inside a 128-byte line are stored longer, so more chunks hide there; rows of the tile past the last channel and a second
// block of rows cost instructions and no stores.  1200 shapes (16 to 768 channels, 2048 pixels to 721 x 1440), table against formula in us: 721 x 1440, 73 -> 384 channels
// 461 / 444, 104 -> 384 472 / 440, 144 -> 384 475 / 457, 208 -> 384 478 / 494, 56 -> 448 513 / 467, 73 -> 448 471 / 495; 720 x 1440, 24 -> 512 422 / 417, 73 -> 384
// 345 / 345, 73 -> 512 444 / 488; 361 x 720, 73 -> 384 139 / 141.  Of 150 shapes that take the formula it is 1.3 % faster on average, 3 % slower at worst; of the others
// the table is 5 % faster on average and loses up to 5 % to it (more with less than 32 input channels).
static bool gelu_table_pays(const PointwiseArgs& a, int mt) {
    if (mt == 1 || 4 * (int64_t)a.B * a.O * a.P < (int64_t)512 << 20) return true;
    const int chunks = (a.K + 31) / 32;
    if (a.P % 64 == 0) return chunks > 1 || a.O < 256;
    return chunks > 7.0 * a.O / (128 * mt * a.n_oblk) - (mt == 3 ? 1.6 : 2.6) - (a.n_oblk > 1 ? 1.0 : 0.0);
}

template <int MT>
static void dma_go(const PointwiseArgs& a, int64_t blocks, int epi, hipStream_t s) {
    const dim3 grid((unsigned)std::min<int64_t>(blocks, std::max(8, DmGeo<MT>::WG_PER_CU * (device_cus() / 8 * 8))));
    switch (epi) {
        case PW_GELU_PRE:
            if constexpr (MT > 1)
                if (!gelu_table_pays(a, MT)) {
                    hipLaunchKernelGGL((pw_gemm_dma_kernel<MT, PW_GELU_PRE | PW_FORMULA>), grid, dim3(512), 0, s, a);
                    break;
                }
            hipLaunchKernelGGL((pw_gemm_dma_kernel<MT, PW_GELU_PRE>), grid, dim3(512), 0, s, a);
            break;
        case PW_GELU_BWD: hipLaunchKernelGGL((pw_gemm_dma_kernel<MT, PW_GELU_BWD>), grid, dim3(512), 0, s, a); break;
        case PW_GELU | PW_ADD: hipLaunchKernelGGL((pw_gemm_dma_kernel<MT, PW_GELU | PW_ADD>), grid, dim3(512), 0, s, a); break;
        case PW_GELU: hipLaunchKernelGGL((pw_gemm_dma_kernel<MT, PW_GELU>), grid, dim3(512), 0, s, a); break;
        case PW_ADD: hipLaunchKernelGGL((pw_gemm_dma_kernel<MT, PW_ADD>), grid, dim3(512), 0, s, a); break;
        default: hipLaunchKernelGGL((pw_gemm_dma_kernel<MT, PW_PLAIN>), grid, dim3(512), 0, s, a);
    }
}

template <int NW>
static void gemm_go(const PointwiseArgs& a, int64_t blocks, int epi, hipStream_t s) {
    const dim3 grid((unsigned)blocks), block(64 * NW);
    switch (epi) {
        case PW_GELU_PRE: hipLaunchKernelGGL((pw_gemm_kernel<NW, PW_GELU_PRE>), grid, block, 0, s, a); break;
        case PW_GELU_BWD: hipLaunchKernelGGL((pw_gemm_kernel<NW, PW_GELU_BWD>), grid, block, 0, s, a); break;
        case PW_GELU | PW_ADD: hipLaunchKernelGGL((pw_gemm_kernel<NW, PW_GELU | PW_ADD>), grid, block, 0, s, a); break;
        case PW_GELU: hipLaunchKernelGGL((pw_gemm_kernel<NW, PW_GELU>), grid, block, 0, s, a); break;
        case PW_ADD: hipLaunchKernelGGL((pw_gemm_kernel<NW, PW_ADD>), grid, block, 0, s, a); break;
        default: hipLaunchKernelGGL((pw_gemm_kernel<NW, PW_PLAIN>), grid, block, 0, s, a);
    }
}

int pointwise_gemm_launch(PointwiseArgs a, hipStream_t s) {
    a.Kpad = pointwise_kpad(a.K, a.O);
    if (a.P % 8 != 0 || a.K < 1 || a.O < 1 || a.B < 1 || a.P < 8) return SFNO_EUNSUPPORTED;
    const bool dma = a.O > PW_ROWS;               // several wavefronts share a pixel strip: direct-to-LDS kernel
    if (a.X2 && (a.K1 < 1 || a.K1 >= a.K)) return SFNO_EINVAL;
    if ((a.Z && (a.act != SFNO_ACT_GELU || a.addend || a.grad)) || (a.grad && (!a.addend || a.act != SFNO_ACT_NONE))) return SFNO_EINVAL;
    int mt = pointwise_mt(a.O), nw = 8;
    const int64_t cus = device_cus();
    const int64_t px_strips = (a.P + (dma ? DM_PX : 512) - 1) / (dma ? DM_PX : 512) * a.B;
    // Smaller tiles where the CUs outnumber the large ones: 50 tiles of 256 x 256 (464 -> 232 channels, 80 x 160 pixels) 22.5 -> 17.3 us
    // with MT = 1, 128 of 384 x 256 (192 -> 384, 2 x 90 x 180, GELU) 23.0 -> 18.5, but 226 of 256 x 256 (512 -> 512, 120 x 240) 26.1 ->
    // 29.4: three blocks of rows each stream the activations.  Two wavefronts per workgroup read no more than eight, only the
    // weights four times as often (64 -> 64, 128 x 256 pixels: 15.2 -> below 10.7).
    if (dma && 3 * px_strips * ((a.O + 128 * mt - 1) / (128 * mt)) < 2 * cus) mt = 1;
    if (!dma && px_strips < cus) nw = 2;
    const int wpx = dma ? DM_PX : 64 * nw;        // pixels per workgroup
    const int rows = dma ? 128 * mt : PW_ROWS;    // output channels per workgroup
    a.n_oblk = (a.O + rows - 1) / rows;
    a.n_strips = (a.P + wpx - 1) / wpx;
    const int64_t strips = a.n_strips * a.B;
    const int64_t blocks = (strips + 7) / 8 * 8 * a.n_oblk;
    if (blocks > 0x7fffffffLL || (dma && a.P > 0x7fffffffLL)) return SFNO_EUNSUPPORTED;
    const int epi = a.Z ? PW_GELU_PRE : a.grad ? PW_GELU_BWD : (a.act == SFNO_ACT_GELU ? PW_GELU : 0) | (a.addend ? PW_ADD : 0);
    if (dma) {     // persistent: as many workgroups as stay resident, the same number on every XCD
        switch (mt) {
            case 1: dma_go<1>(a, blocks, epi, s); break;
            case 2: dma_go<2>(a, blocks, epi, s); break;
            default: dma_go<3>(a, blocks, epi, s); break;
        }
    } else if (nw == 2)
        gemm_go<2>(a, blocks, epi, s);
    else
        gemm_go<8>(a, blocks, epi, s);
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

template <int MT>
static void mlp_go(const MlpArgs& a, bool ragged, hipStream_t s) {
    const dim3 grid((unsigned)std::min<int64_t>(a.n_strips * a.B, device_cus())), block(256);
    if (ragged)
        hipLaunchKernelGGL((pw_mlp_kernel<MT, true>), grid, block, 0, s, a);
    else
        hipLaunchKernelGGL((pw_mlp_kernel<MT, false>), grid, block, 0, s, a);
}

bool pointwise_mlp_supported(int B, int E, int H, int64_t P) {
    if (B < 1 || E < 8 || E > 384 || H < 16 || E % 8 != 0 || H % 16 != 0 || P < 8 || P % 8 != 0) return false;
    // 32-bit byte offsets within a sample and within a packed weight, a 31-bit count of tiles
    return (int64_t)E * P < (1LL << 30) && (int64_t)E * H < (1LL << 28) && (P + 127) / 128 * B < (1LL << 30);
}

// Whether the one kernel is the faster way (both give the same bits): estimates of both in us, fitted to 1669 shapes (E 16 to 384, H E / 2 to 4 E,
// 2 to 8100 tiles, each way timed in a graph on 256 CUs) within 5 and 8 %.  The one kernel takes whole rounds of tiles, each as long as its padded rows
// take: E = 136 pays for 256.  The three have their launches and the depth of one tile, which short calls see, and then bytes and products of
// padded weights.  In us, three / one: E = 384, H = 768 with 900 tiles 221 / 178, with 96 58 / 46, with 16 42 / 45; E = 128, H = 256 58 / 46 with 900;
// E = 64, H = 128 21.5 / 14.9 with 192, 35 / 47 with 900 and 33 / 26 with 512; E = 136 with 2000 and H = 136 87 / 137, H = 272 151 / 167, H = 544 245 / 226;
// E = 264 with 900 and H = 128 70 / 104, H = 528 164 / 162, H = 1056 257 / 244.  Of the 865 shapes past one round 31 lose more than 3 % to
// the three by this rule (at most 10 % with H = 2 E, H = E = 128 up to 25 %); by a line drawn at E > 64 152 did, up to 66 %.
bool pointwise_mlp_preferred(int B, int E, int H, int64_t P) {
    if (!pointwise_mlp_supported(B, E, H, P)) return false;
    const int64_t tiles = (P + 127) / 128 * B, cus = device_cus();
    const int mt = (E + 127) / 128, chunks = std::max(2, (H + 127) / 128);
    constexpr double ROUND[3] = {4.4, 10.0, 16.5}, CHUNK[3] = {2.95, 3.75, 5.05};
    const double one = 4.5 + (double)((tiles + cus - 1) / cus) * (ROUND[mt - 1] + CHUNK[mt - 1] * chunks);
    const double depth = 12.3 + 0.0307 * E + 0.0229 * H;
    const double rate = (0.00936 + 1.25e-4 * E + 7.8e-5 * H + 1.72e-7 * ((double)E * pointwise_opad(H) + (double)H * pointwise_opad(E))) * 256 / (double)cus;
    const double work = rate * (double)tiles;
    // (a call of one round is a few us of a network that waits for its host: two launches less are worth 2 us; the forward of four blocks of 32 channels
    // on a 32 x 64 grid 446 -> 427 us)
    return one <= std::max(depth, work) + 0.86 * std::min(depth, work) + (tiles <= cus ? 2.0 : 0.0);
}

int pointwise_mlp_launch(MlpArgs a, hipStream_t s) {
    if (!pointwise_mlp_supported(a.B, a.E, a.H, a.P)) return SFNO_EUNSUPPORTED;
    a.kpad1 = pointwise_kpad(a.E, a.H);
    a.opad1 = pointwise_opad(a.H);
    a.kpad2 = pointwise_kpad(a.H, a.E);
    a.opad2 = pointwise_opad(a.E);
    a.n_strips = (a.P + 127) / 128;
    const bool ragged = a.E % 128 != 0 || a.H % 128 != 0 || a.H < 256;
    switch ((a.E + 127) / 128) {
        case 1: mlp_go<1>(a, ragged, s); break;
        case 2: mlp_go<2>(a, ragged, s); break;
        default: mlp_go<3>(a, ragged, s); break;
    }
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

int row_stats_segments(int64_t rows, int64_t P) {
    // ~16 K elements per workgroup.  The split depends on the row length only, so that the sums of a row (and with them
    // every value downstream) do not change with the number of rows: a sample gives the same result alone and in a batch.
    (void)rows;
    return (int)std::max<int64_t>(1, std::min<int64_t>(P / 16384, 64));
}

int instance_norm_coeffs_launch(const unsigned short* x, const float* gamma, const float* beta, float* scale, float* shift, float2* partial,
                                int64_t rows, int channels, int64_t P, float eps, hipStream_t s, float2* moments) {
    if (rows < 1 || P < 1 || channels < 1 || rows > 0x7fffffffLL / 64) return SFNO_EUNSUPPORTED;
    if (P % 8 != 0) return SFNO_EUNSUPPORTED;     // 16-byte loads from every row start
    if (P <= NORM_SMALL_PIXELS) {
        hipLaunchKernelGGL(row_stats_small_kernel, dim3((unsigned)rows), dim3(64), 0, s, x, gamma, beta, scale, shift, moments, channels, (int)P, eps);
        return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
    }
    const int nseg = row_stats_segments(rows, P);
    hipLaunchKernelGGL(row_stats_partial_kernel, dim3((unsigned)rows, (unsigned)nseg), dim3(ST_THREADS), 0, s, x, partial, P, nseg);
    hipLaunchKernelGGL(row_stats_finalize_kernel, dim3((unsigned)((rows + 127) / 128)), dim3(128), 0, s, x, partial, gamma, beta, scale, shift, moments,
                       rows, channels, P, nseg, eps);
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

int instance_norm_coeffs_lat_launch(const float2* stats, const float* gamma, const float* beta, float* scale, float* shift, int64_t rows, int channels,
                                    int nlat, float eps, hipStream_t s, float2* moments) {
    if (rows < 1 || rows > 0x7fffffffLL || channels < 1 || nlat < 1) return SFNO_EINVAL;
    hipLaunchKernelGGL(lat_stats_finalize_kernel, dim3((unsigned)rows), dim3(64), 0, s, stats, gamma, beta, scale, shift, moments, channels, nlat,
                       eps);
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

int scale_shift_act_launch(const unsigned short* x, const float* scale, const float* shift, unsigned short* y, int64_t rows, int64_t P, int act,
                           hipStream_t s) {
    if (rows < 1 || P < 8 || P % 8 != 0) return SFNO_EUNSUPPORTED;
    const int64_t gpr = P / 8, total = rows * gpr;
    const int64_t blocks = (total + 255) / 256;
    if (blocks > 0x7fffffffLL) return SFNO_EUNSUPPORTED;
    hipLaunchKernelGGL(scale_shift_act_kernel, dim3((unsigned)blocks), dim3(256), 0, s, x, scale, shift, y, P, gpr, total, act);
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

int norm_grad_launch(const unsigned short* g, const unsigned short* x, const float* scale, const float* shift, const float2* moments, float2* partial,
                     unsigned short* dx, float* dgamma, float* dbeta, int batch, int channels, int64_t P, int act, hipStream_t s) {
    const int64_t rows = (int64_t)batch * channels;
    if (rows < 1 || P < 8 || P % 8 != 0 || rows > 0x7fffffffLL / 64) return SFNO_EUNSUPPORTED;
    const int nseg = row_stats_segments(rows, P);
    const dim3 grid((unsigned)rows, (unsigned)nseg);
    if (act == SFNO_ACT_GELU) {
        hipLaunchKernelGGL(norm_grad_reduce_kernel<true>, grid, dim3(ST_THREADS), 0, s, g, x, scale, shift, moments, partial, P, nseg);
        hipLaunchKernelGGL(norm_grad_apply_kernel<true>, grid, dim3(ST_THREADS), 0, s, g, x, scale, shift, moments, partial, dx, P, nseg);
    } else {
        hipLaunchKernelGGL(norm_grad_reduce_kernel<false>, grid, dim3(ST_THREADS), 0, s, g, x, scale, shift, moments, partial, P, nseg);
        hipLaunchKernelGGL(norm_grad_apply_kernel<false>, grid, dim3(ST_THREADS), 0, s, g, x, scale, shift, moments, partial, dx, P, nseg);
    }
    if (dgamma || dbeta)
        hipLaunchKernelGGL(norm_param_grad_kernel, dim3((unsigned)channels), dim3(64), 0, s, partial, dgamma, dbeta, batch, channels, nseg);
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

}  // namespace sfno
