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
// with rows (m, b) of the spectral layout as A operands (moved to LDS as they are, in whole 128-byte lines, de-interleaved and cut in
// registers; -Xi costs one sign flip per packed pair) and the weights as B operands: the packed stream holds, per
// (degree, block of 32 NTC output channels, chunk of 16 input channels), the image of one LDS stage -- (Wr, Wi) x two
// fp16 planes x output channel x 16 input channels.  The wavefronts move both with global_load_lds_dwordx4, the weights into a
// ring of three stages, the activations into two, two chunks ahead of the matrix instructions.  8 bytes per complex weight, read once.
//
// What bounds it: at one sample the stream of weights (283 of 460 MB for 384 x 384 channels and 240 degrees) and the three rounds that 132 workgroups to an
// XCD take on its 64 places; at four samples the matrix pipe, 425 GFLOP at 1050 TFLOP/s where a large bf16 product reaches 1350 here (the
// clock falls to 1.6 GHz under either).  The vector instructions of a chunk were a third of its time and are 70 for 48 matrix instructions now, and a request
// had one contraction to land where it has two now (activations waited in registers, a lane asking for 64 bytes of its own row in four pieces).
// 384 x 384 channels, 240 degrees, 1 / 2 / 4 samples 160 / 242 / 428 -> 139 / 233 / 404 us; 120 degrees 58 / 85 -> 49 / 66; 128 x 128 channels,
// 90 degrees, 2 samples 22.5 -> 19.2.  Same bits.
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
typedef unsigned int u4 __attribute__((ext_vector_type(4)));

constexpr int DHF_KC = 16;             // complex input channels per chunk: one matrix K step per part
constexpr int DHF_TOP = 14;            // scaled magnitudes stay below 2^(TOP + 1)
constexpr int DHF_HEAD = 3;            // bits of headroom left when a row's exponent bound is raised
constexpr int DHF_SH = DHF_TOP + 127;  // scaled = x * 2^(SH - E), E = biased exponent bound of the row
constexpr int DHF_EMIN = DHF_SH - 127; // smallest bound: its scale is the largest power of two of fp32 (rows below 2^-112 keep 25 bits above 2^-151)
constexpr int DHF_STAGES = 3;          // of weights
constexpr int DHF_XSTAGES = 2, DHF_XBYTES = 32 * 128;      // of activations: 32 rows x 16 complex fp32 per wavefront

// 16 bytes per lane from global memory to LDS base + 16 lane (M0 carries the base; the compiler reserves M0 and does not
// accept it on a clobber list: nothing else in this file may depend on M0 -- no indexed register arrays, no LDS-DMA builtins)
__device__ __forceinline__ void dhf_dma16(const void* g, unsigned lds_byte_addr) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(lds_byte_addr) : "memory");
}
// byte offset, within one (part, plane) of a stage, of the 16-byte piece (output channel o, half kg of the chunk):
// the halves swap places every 8 channels so that the 16-byte reads of 16 consecutive lanes cover all banks
__host__ __device__ constexpr int dhf_piece(int o, int kg) { return o * 32 + ((kg ^ ((o >> 3) & 1)) * 16); }

// One row group of up to 128 rows against one block of CO output channels: this wavefront has 32 rows and T tiles of 32 channels, tile t0 first.
template <int NTC, int T>
__device__ __forceinline__ void dhf_rows(const DhconvArgs& a, unsigned char* lds, int l, int ob, int first, int t0, bool active, int ncols, int wslot) {
    constexpr int CO = 32 * NTC;                     // complex output channels per workgroup
    constexpr int STAGE = 4 * CO * 32;               // bytes: (Wr, Wi) x 2 planes x CO x 16 fp16
    constexpr int ND = STAGE / 4096;                 // weight requests per wavefront and chunk
    constexpr int NX = 4;                            // activation requests per wavefront and chunk
    const int lane = threadIdx.x & 63;
    const int nc = a.nc;                                           // chunks of 16 complex input channels
    const int kg = lane >> 5, cl = lane & 31;
    const unsigned lds0 = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)lds);

    // packed weights of (l, ob): nc stage images; this wavefront moves bytes [ND wslot KiB, ND (wslot + 1) KiB) of each
    const unsigned char* wsrc = reinterpret_cast<const unsigned char*>(a.W) + ((int64_t)l * a.nob + ob) * nc * STAGE + wslot * (ND * 1024) + lane * 16;
    const unsigned wdst = lds0 + wslot * (ND * 1024);
    // Activations: request j brings 8 whole 128-byte lines, chunk c of rows 8 j .. 8 j + 7, into this wavefront's two KiB x 4 of LDS.  Slot s of
    // row r holds piece s ^ (r / 2 % 8) of the line, so that 16 lanes that read the same piece of 16 rows cover all banks.
    const unsigned xdst = lds0 + DHF_STAGES * STAGE + wslot * (DHF_XSTAGES * DHF_XBYTES);
    const unsigned char* xraw = lds + DHF_STAGES * STAGE + wslot * (DHF_XSTAGES * DHF_XBYTES) + cl * 128;
    const int rr = lane >> 3, ps = (lane & 7) ^ (rr >> 1);
    int64_t xoff[NX];          // my piece of chunk 0 of the rows
    const bool aligned = (reinterpret_cast<uintptr_t>(a.X) & 15) == 0;       // (16 bytes at a time go to LDS directly from aligned addresses only)
#pragma unroll
    for (int j = 0; j < NX; ++j) {
        const int n = min(first + 8 * j + rr, ncols - 1);
        const int mm = n / a.B, bb = n - mm * a.B;
        xoff[j] = ((int64_t)mm * a.L + l) * a.ld_in + (int64_t)bb * a.I2 + 4 * (ps ^ (4 * (j & 1)));
    }
    // (pieces past the last channel, in the last chunk only, repeat the last one: the weights are zero there)
    auto x_dma = [&](int c, int stage) {
        const unsigned dst = xdst + stage * DHF_XBYTES;
        if (!aligned) {
            // (these loads retire behind the weights requested before them, so the counted waits below hold)
#pragma unroll
            for (int j = 0; j < NX; ++j) {
                const int k = 4 * (ps ^ (4 * (j & 1)));
                const f4 x = *reinterpret_cast<const f4*>(a.X + xoff[j] + (min(2 * DHF_KC * c + k, a.I2 - 4) - k));
                *reinterpret_cast<f4*>(lds + (dst - lds0) + j * 1024 + 16 * lane) = x;
            }
        } else if (c + 1 < nc) {
            const float* base = a.X + 2 * DHF_KC * c;
#pragma unroll
            for (int j = 0; j < NX; ++j) dhf_dma16(base + xoff[j], dst + j * 1024);
        } else {
#pragma unroll
            for (int j = 0; j < NX; ++j) {
                const int k = 4 * (ps ^ (4 * (j & 1)));
                dhf_dma16(a.X + xoff[j] + (min(2 * DHF_KC * c + k, a.I2 - 4) - k), dst + j * 1024);
            }
        }
    };
    auto w_dma = [&](int c, int stage) {
#pragma unroll
        for (int j = 0; j < ND; ++j) dhf_dma16(wsrc + (int64_t)c * STAGE + j * 1024, wdst + stage * STAGE + j * 1024);
    };

    floatx16 yr[T], yi[T];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            yr[t][v] = 0.0f;
            yi[t][v] = 0.0f;
        }
    int E = DHF_EMIN;          // biased exponent bound of my row (lanes cl and cl + 32 hold the same row and agree)
    const int xs = 4 * kg ^ (cl >> 1 & 7);
    // my 8 complex activations of the chunk in stage `stage`: i = 16c + 8kg .. +7, (re, im) interleaved
    auto x_read = [&](int stage, f4 (&xr)[NX]) {
#pragma unroll
        for (int j = 0; j < NX; ++j) xr[j] = *reinterpret_cast<const f4*>(xraw + stage * DHF_XBYTES + 16 * (xs ^ j));
    };
    // raises the exponent bound of the row to this chunk's values, and the scale of the partial sums with it: D row
    // 8 (v / 4) + 4 kg + v % 4 belongs to the lanes of that number
    auto bound = [&](const f4 (&xr)[NX]) {
        // (written out: the compiler would bring every magnitude to canonical form first)
        float mx;
        asm("v_max3_f32 %0, |%1|, |%2|, |%3|" : "=v"(mx) : "v"(xr[0][0]), "v"(xr[0][1]), "v"(xr[0][2]));
        asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(mx) : "v"(mx), "v"(xr[0][3]), "v"(xr[1][0]));
        asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(mx) : "v"(mx), "v"(xr[1][1]), "v"(xr[1][2]));
        asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(mx) : "v"(mx), "v"(xr[1][3]), "v"(xr[2][0]));
        asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(mx) : "v"(mx), "v"(xr[2][1]), "v"(xr[2][2]));
        asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(mx) : "v"(mx), "v"(xr[2][3]), "v"(xr[3][0]));
        asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(mx) : "v"(mx), "v"(xr[3][1]), "v"(xr[3][2]));
        asm("v_max_f32 %0, %1, |%2|" : "=v"(mx) : "v"(mx), "v"(xr[3][3]));
        const unsigned int mb = __builtin_bit_cast(unsigned int, mx);
        if (__builtin_amdgcn_ballot_w64((int)(mb >> 23) > E) == 0) return;
        // the other half of the row's chunk sits 32 lanes away
        const auto sw = __builtin_amdgcn_permlane32_swap(mb, mb, false, false);
        const int eb = (int)(max(sw[0], sw[1]) >> 23);
        const int en = eb > E ? eb + DHF_HEAD : E;
        const int pend = E - en;
        E = en;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int d = __builtin_amdgcn_ds_bpermute(4 * (8 * (v >> 2) + 4 * kg + (v & 3)), pend);
#pragma unroll
            for (int t = 0; t < T; ++t) {
                yr[t][v] = __builtin_ldexpf(yr[t][v], d);
                yi[t][v] = __builtin_ldexpf(yi[t][v], d);
            }
        }
    };
    // planes of the chunk: pl[0], pl[1] = Xr (upper, lower part), pl[2], pl[3] = Xi; word e of a plane holds the channels
    // 2e, 2e + 1 of the lane's eight.  (The conversions round toward zero, see MODE below.)
    auto cut = [&](const f4 (&xr)[NX], u4 (&pl)[4]) {
        const float sc = __builtin_bit_cast(float, (unsigned)(DHF_SH + 127 - E) << 23);
#pragma unroll
        for (int e = 0; e < NX; ++e)
#pragma unroll
            for (int part = 0; part < 2; ++part) {
                const float u = xr[e][part], v = xr[e][2 + part];
                unsigned hi, lo;
                asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(hi) : "v"(u), "v"(sc));
                asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(hi) : "v"(v), "v"(sc));
                asm("v_fma_mixlo_f16 %0, %1, %2, -%3 op_sel_hi:[0,0,1]" : "=v"(lo) : "v"(u), "v"(sc), "v"(hi));
                asm("v_fma_mixhi_f16 %0, %1, %2, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "+v"(lo) : "v"(v), "v"(sc), "v"(hi));
                pl[2 * part][e] = hi;
                pl[2 * part + 1][e] = lo;
            }
    };
    // one chunk of matrix instructions on stage `stage` with the planes pc
    const int frag = dhf_piece(32 * t0 + cl, kg);
    auto contract = [&](int stage, const u4 (&pc)[4]) {
        const unsigned char* sb = lds + stage * STAGE + frag;
        const f16x8 xr0 = __builtin_bit_cast(f16x8, pc[0]), xr1 = __builtin_bit_cast(f16x8, pc[1]);
        const f16x8 xi0 = __builtin_bit_cast(f16x8, pc[2]), xi1 = __builtin_bit_cast(f16x8, pc[3]);
        // -Xi: one sign flip per packed pair
        const f16x8 ni0 = __builtin_bit_cast(f16x8, pc[2] ^ 0x80008000u), ni1 = __builtin_bit_cast(f16x8, pc[3] ^ 0x80008000u);
#pragma unroll
        for (int t = 0; t < T; ++t) {
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

    // Pipeline, three weight stages and two of activations.  Iteration c: wait for this wavefront's pieces of chunk c (those of chunk c + 1
    // stay in flight), take its activations out of LDS, barrier (every wavefront's pieces of the weights of chunk c have landed and every wavefront
    // is done reading chunk c - 1), request chunk c + 2 into the stages that came free, cut the activations and contract.  A request has two
    // contractions to land.  All requests are written in assembly (the compiler would make every LDS read wait for them) and none has a
    // result register; the explicit waits count them.
    w_dma(0, 0);
    if (active) x_dma(0, 0);
    if (nc > 1) {
        w_dma(1, 1);
        if (active) x_dma(1, 1);
    }
    __builtin_amdgcn_s_setreg((1 << 11) | (2 << 6) | 1, 3);        // MODE[3:2]: conversions to fp16 round toward zero
    for (int c = 0, stage = 0; c < nc; ++c, stage = stage == 2 ? 0 : stage + 1) {
        const bool more1 = c + 1 < nc, more2 = c + 2 < nc;         // uniform over the workgroup
        f4 xc[NX];
        __builtin_amdgcn_sched_barrier(0);
        if (active) {
            if (more1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(ND + NX) : "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            x_read(c & 1, xc);
        } else {
            if (more1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(ND) : "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (more2) w_dma(c + 2, stage == 0 ? 2 : stage - 1);
        if (active) {
            if (more2) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");         // (the stage has been read)
                x_dma(c + 2, c & 1);
            }
            u4 pc[4];
            bound(xc);
            cut(xc, pc);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(1);
            contract(stage, pc);
            __builtin_amdgcn_s_setprio(0);
        }
    }

    if (!active) return;
    // Undo the scales: row by 2^(E - SH) (the partial sums carry the scale of the last cut), column by the factor stored
    // with the weights.
    const int ch0 = CO * ob + 32 * t0;                             // my first channel
    float cinv[T];
#pragma unroll
    for (int t = 0; t < T; ++t) cinv[t] = a.cinv[(int64_t)l * (a.nob * CO) + ch0 + 32 * t + cl];
    // (waited for here and not where they are used: on some way around the uses they would count as on their way in the loops of the other T,
    // whose registers they share, and hold up every iteration there)
    __builtin_amdgcn_s_waitcnt(0x0F70);                            // vmcnt(0)
    const int Efinal = E;
    const int nn0 = first + 4 * kg;                                // my first row; the others are 8 (v / 4) + v % 4 further on
    if (a.B == 1 && first + 32 <= ncols && 2 * (ch0 + 32 * T) <= a.O2) {
        // one sample and no row or channel of my tile outside the tensor: row = order, one address, constant steps
        float* o = a.Y + ((int64_t)nn0 * a.L + l) * a.ld_out + 2 * (ch0 + cl);
        const int64_t rstep = (int64_t)a.L * a.ld_out;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int er = __builtin_amdgcn_ds_bpermute(4 * (8 * (v >> 2) + 4 * kg + (v & 3)), Efinal);
            float* orow = o + (8 * (v >> 2) + (v & 3)) * rstep;
#pragma unroll
            for (int t = 0; t < T; ++t)
                *reinterpret_cast<f2*>(orow + 64 * t) = f2{__builtin_ldexpf(yr[t][v], er - DHF_SH) * cinv[t], __builtin_ldexpf(yi[t][v], er - DHF_SH) * cinv[t]};
        }
        return;
    }
    if ((a.B & (a.B - 1)) == 0 && first + 32 <= ncols && 2 * (ch0 + 32 * T) <= a.O2) {
        // a power-of-two number of samples, whole tile inside: (order, sample) of a row by shift and mask, no checks
        const int lb = 31 - __builtin_clz(a.B);
        float* o = a.Y + (int64_t)l * a.ld_out + 2 * (ch0 + cl);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int er = __builtin_amdgcn_ds_bpermute(4 * (8 * (v >> 2) + 4 * kg + (v & 3)), Efinal);
            const int nn = nn0 + 8 * (v >> 2) + (v & 3);
            float* orow = o + (int64_t)(nn >> lb) * a.L * a.ld_out + (int64_t)(nn & (a.B - 1)) * a.O2;
#pragma unroll
            for (int t = 0; t < T; ++t)
                *reinterpret_cast<f2*>(orow + 64 * t) = f2{__builtin_ldexpf(yr[t][v], er - DHF_SH) * cinv[t], __builtin_ldexpf(yi[t][v], er - DHF_SH) * cinv[t]};
        }
        return;
    }
    // The row slots between the last sample's channels and ld_out, at most 15, become zeros: the transform behind reads whole rows.  The
    // wavefront with the last tile writes them; where there are any, O is no multiple of 16 and that tile comes by here.  (Clearing them
    // in a pass in front: 138 channels, 241 degrees 16 us for the whole tensor, 4 us and a launch for the slots alone.)
    const int npad = a.ld_out - a.B * a.O2;
    const bool pad = npad > 0 && ob == a.nob - 1 && t0 + T == NTC;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int er = __builtin_amdgcn_ds_bpermute(4 * (8 * (v >> 2) + 4 * kg + (v & 3)), Efinal);
        const int nn = nn0 + 8 * (v >> 2) + (v & 3);
        if (nn >= ncols) continue;
        const int m2 = nn / a.B, b2 = nn - m2 * a.B;
        float* orow = a.Y + ((int64_t)m2 * a.L + l) * a.ld_out + (int64_t)b2 * a.O2;
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int oc = 2 * (ch0 + 32 * t + cl);
            if (oc < a.O2)
                *reinterpret_cast<f2*>(orow + oc) = f2{__builtin_ldexpf(yr[t][v], er - DHF_SH) * cinv[t], __builtin_ldexpf(yi[t][v], er - DHF_SH) * cinv[t]};
        }
        if (pad && b2 == a.B - 1 && 2 * cl < npad) *reinterpret_cast<f2*>(orow + a.O2 + 2 * cl) = f2{0.f, 0.f};
    }
}

// grid = dh_blocks workgroups (see dh_map), row groups of 128; a.nob = ceil(O / (32 NTC)); requires 2*I % 4 == 0
template <int NTC>
__global__ __launch_bounds__(256, 2) void dhconv_f16_kernel(DhconvArgs a) {
    __shared__ __align__(16) unsigned char lds[DHF_STAGES * 4 * 32 * NTC * 32 + 4 * DHF_XSTAGES * DHF_XBYTES];
    int l, ob, r0, ncols, rot;
    if (!dh_map(a, 128, l, ob, r0, ncols, rot)) return;
    const int wslot = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wave = (wslot + rot) & 3;
    // A group of at most 32 or 64 rows shares its tiles out to the wavefronts instead of leaving three or two of them idle: the lowest degrees
    // run last and mostly alone, and a wavefront's matrix instructions one after the other (384 x 384 channels, one sample: 32 degrees 35 -> 22 us,
    // 64 degrees and 33 orders 36 -> 26, 34 without the sharing of two blocks; 240 degrees 145 -> 140 of it for two blocks).
    const int blocks = (ncols - r0 + 31) >> 5;
    if (blocks == 1)
        dhf_rows<NTC, 1>(a, lds, l, ob, r0, wave & (NTC - 1), wave < NTC, ncols, wslot);
    else if (blocks == 2)
        dhf_rows<NTC, NTC / 2>(a, lds, l, ob, r0 + 32 * (wave >> 1), (wave & 1) * (NTC / 2), true, ncols, wslot);
    else
        dhf_rows<NTC, NTC>(a, lds, l, ob, r0 + 32 * wave, 0, wave < blocks, ncols, wslot);
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
