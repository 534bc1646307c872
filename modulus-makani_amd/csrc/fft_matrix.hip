// Longitude FFTs of long bfloat16 rows of which only the lowest orders are kept (a sixth of the length at most): half of the work on the
// matrix units, one exchange through LDS instead of three.
//
// The vector kernels of fft_kernels.h move the in-model 1440-point transforms at half of the copy rate: as many cycles of vector
// instructions and of LDS accesses as the whole transform may take.  N = 32 N1, n = n2 + 32 n1, k = k1 + N1 k2:
//   X[k] = sum over n2 of w_32^(n2 k2) w_N^(n2 k1) Y[k1][n2],   Y[k1][n2] = sum over n1 of w_N1^(n1 k1) x[n2 + 32 n1].
// The inner sum is a real DFT of N1 points whose inputs are bfloat16 numbers: a matrix product with cosines and sines (k1 <= N1 / 2), cut into
// three bfloat16 parts each, so that every product is exact and the sums run in fp32 like those of the vector kernels.  Its operand is
// the row as it lies in memory, transposed on its way out of LDS.  The outer one has 12 of 32 outputs, k2 = -6 ... 5: eight-point DFTs in
// registers and their sums over the remaining factor 4; order m = k or, for negative k, m = -k and the conjugate.
// Used for gradients (synthesis_adjoint_launch): the forward transforms keep the rounding of the vector kernels.
#include "fft_fast.h"

#include "fft_kernels.h"

#include <cstring>

namespace sfno {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int FM_THREADS = 192;
constexpr int FM_ROWS = 8;                   // rows of a batch; a tile is two batches: 16 channels, one 128-byte line per order

// wait until this wavefront's LDS accesses (and, VM, its global ones) are done, then for the others
template <bool VM>
__device__ __forceinline__ void fm_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(VM ? 0x0070 : 0xc07f);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
}

// 16 bytes per lane from base + offset to consecutive LDS addresses
__device__ __forceinline__ void fm_dma16(const void* base, unsigned offset, unsigned lds_byte_addr) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(offset), "s"(base), "s"(lds_byte_addr) : "memory");
}

// a + b c
__device__ __forceinline__ float2 cfma(float2 a, float2 b, float2 c) {
    return make_float2(fmaf(b.x, c.x, fmaf(-b.y, c.y, a.x)), fmaf(b.x, c.y, fmaf(b.y, c.x, a.y)));
}

template <int N1>
struct MatGeo {
    static constexpr int N = 32 * N1, KC = N1 / 2 + 1;     // first-stage outputs k1 = 0 ... N1 / 2
    static constexpr int KT = (N1 + 31) / 32;              // matrix steps of 32 inputs
    // floats between rows of Y, so that reads of eight rows fall on 32 banks; odd k1 hold their two halves swapped, on the other 32
    static constexpr int PR = 24 * 64 + 4;
    static constexpr int JN = (N + FM_THREADS - 1) / FM_THREADS;   // pieces of 16 bytes per thread: N in a batch
    static constexpr int ROW = 2 * N;                      // bytes
    static_assert(KC > 16 && KC <= 24, "three tiles of 16 (Re, Im) rows");
};

// Persistent workgroups (two per CU) walk the tiles as in rfft_fast_kernel.  A batch of eight rows goes straight to LDS; the matrix phase
// (a wavefront takes one of the three tiles of 16 (Re, Im) rows) leaves Y there, in the phase after it a thread owns one (row, k1).  The next
// batch is asked for between the two phases; a tile's results are stored when the next one's first batch has landed, so that no wait for a
// batch waits for the stores before it.
// grid = 8 * (workgroups per XCD)
template <int N1>
__global__ __launch_bounds__(FM_THREADS, 2) void rfft_matrix_kernel(const bf16x8* __restrict__ frag, const float2* __restrict__ tw,
                                                                    const unsigned short* __restrict__ x, float* __restrict__ xm, int rows, int nlat,
                                                                    int mmax, int ld, int ngroups) {
    using G = MatGeo<N1>;
    constexpr int N = G::N, KC = G::KC, KT = G::KT, PR = G::PR;
    __shared__ __align__(16) float y[FM_ROWS * PR];
    __shared__ __align__(16) unsigned char stage[G::JN * FM_THREADS * 16];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const TileWalk walk(nlat, ngroups);
    int t = walk.first();
    if (t >= walk.ntiles) return;

    // requests: piece c of a batch is 16 bytes of row c / (N / 8); pieces past the batch and rows past the tensor repeat the last ones
    const unsigned stage0 = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)stage);
    unsigned piece[G::JN];
    auto pieces = [&](int last) {                          // last: the tensor's last row, counted from the batch's first
#pragma unroll
        for (int j = 0; j < G::JN; ++j) {
            const int c = min(j * FM_THREADS + tid, N - 1), row = c / (N / 8);
            piece[j] = (unsigned)(min(row, last) * nlat) * (unsigned)G::ROW + 16 * (c - row * (N / 8));
        }
    };
    pieces(FM_ROWS - 1);
    auto request = [&](int tile, int half) {
        int lat, group;
        walk.locate(tile, lat, group);
        const int r0 = (group * 2 + half) * FM_ROWS, rb = min(r0, rows - 1);
        const uint64_t base = reinterpret_cast<uint64_t>(x) + ((int64_t)rb * nlat + lat) * G::ROW;
        const void* ubase = reinterpret_cast<const void*>((uint64_t)__builtin_amdgcn_readfirstlane((int)(base >> 32)) << 32 |
                                                          (unsigned)__builtin_amdgcn_readfirstlane((int)base));
        const bool whole = r0 + FM_ROWS <= rows;
        if (!whole) pieces(rows - 1 - rb);
#pragma unroll
        for (int j = 0; j < G::JN; ++j) fm_dma16(ubase, piece[j], stage0 + (j * FM_THREADS + wave * 64) * 16);
        if (!whole) pieces(FM_ROWS - 1);
    };

    // matrix phase: the cosines and sines of the wavefront's row tile, and where the lane's four values of a transposing read begin (a
    // group of 16 lanes reads four inputs n1 of 16 columns n2; inputs past N1 repeat others of the row and meet zeros)
    const int mt = wave, g = lane >> 4;
    bf16x8 cs[KT][3];
#pragma unroll
    for (int ks = 0; ks < KT; ++ks)
#pragma unroll
        for (int p = 0; p < 3; ++p) cs[ks][p] = frag[((p * 3 + mt) * KT + ks) * 64 + lane];
    int src[KT][2];
#pragma unroll
    for (int ks = 0; ks < KT; ++ks)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            int n1 = 32 * ks + 8 * g + 4 * e + ((lane & 15) >> 2);
            if (n1 >= N1) n1 -= 32;
            src[ks][e] = n1 * 64 + (lane & 3) * 8;
        }
    const int k1w = 8 * mt + 2 * g;
    float* const yw = y + k1w * 64 + 2 * (lane & 15);
    auto columns = [&](int off, int ks, int e) {
        typedef __attribute__((address_space(3))) s16x4 lds4;
        return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)(stage + src[ks][e] + off));
    };
    // four tiles of 16 columns at a time; between the matrix instructions the next four's operands are read and the previous sums written
    // (one after the other 3.5 k cycles a batch, so 2.5 k)
    s16x4 half[2][4][KT][2];
    auto read = [&](int q, int j) {                        // j-th read of the four tiles q
        const int u = j / (2 * KT), ks = j / 2 % KT, i = 4 * q + u;
        half[q & 1][u][ks][j & 1] = columns((i >> 1) * G::ROW + (i & 1) * 32, ks, j & 1);
    };
    auto write = [&](int q, int j, const f32x4(&acc)[4]) { // j-th write of their sums
        const int u = j / 2, i = 4 * q + u;
        float* dst = yw + (i >> 1) * PR + (j & 1) * 64 + ((i ^ j) & 1) * 32;
        *reinterpret_cast<float2*>(dst) = j & 1 ? make_float2(acc[u][2], acc[u][3]) : make_float2(acc[u][0], acc[u][1]);
    };
    auto matrix_phase = [&]() {
        f32x4 acc[2][4];
#pragma unroll
        for (int j = 0; j < 8 * KT; ++j) read(0, j);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[q & 1][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < 12 * KT; ++j) {            // smallest parts first
                const int p = 2 - j / (4 * KT), ks = j / 4 % KT, u = j & 3;
                const s16x4 lo = half[q & 1][u][ks][0], hi = half[q & 1][u][ks][1];
                acc[q & 1][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cs[ks][p], __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)),
                                                                       acc[q & 1][u], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (q > 0 && j < 8) write(q - 1, j, acc[(q & 1) ^ 1]);
                if (q < 3 && j < 8 * KT) read(q + 1, j);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) write(3, j, acc[1]);
    };

    // vector phase: thread -> row r, k1
    const int r = tid & 7, k1 = tid >> 3, k1r = min(k1, KC - 1);
    float2 w[32];
#pragma unroll
    for (int n2 = 0; n2 < 32; ++n2) w[n2] = tw[k1r * 32 + n2];
    constexpr TwTab<32> w32 = make_tw<32>();
    const float4* const yr = reinterpret_cast<const float4*>(y + r * PR + k1r * 64);
    const float4* const yh[2] = {yr + 8 * (k1r & 1), yr + 8 * (~k1r & 1)};      // columns 0 ... 15, 16 ... 31
    float2 out[2][12];                                    // [batch][orders k1 + N1 s, then N1 (s + 1) - k1 (the conjugate)]
    auto vector_phase = [&](float2(&o)[12]) {
        float2 f[4][8];                                    // columns n2 = 4a + b -> their eight-point DFTs over a
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            const float4 q = yh[c >> 3][c & 7];
            f[2 * (c & 1)][c >> 1] = cmul(make_float2(q.x, q.y), w[2 * c]);
            f[2 * (c & 1) + 1][c >> 1] = cmul(make_float2(q.z, q.w), w[2 * c + 1]);
        }
#pragma unroll
        for (int b = 0; b < 4; ++b) dft<8, 0>(f[b]);
#pragma unroll
        for (int u = 0; u < 12; ++u) {
            const int k2 = u < 6 ? u : 5 - u, q = k2 & 7, i = k2 & 31;
            const float2 wk = make_float2(w32.c[i], w32.s[i]);
            const float2 a = f[0][q];
            if (k2 == 0) {
                o[u] = cadd(cadd(a, f[2][q]), cadd(f[1][q], f[3][q]));
            } else {
                const float2 b = cfma(f[1][q], cfma(f[2][q], f[3][q], wk), wk);
                o[u] = cfma(a, b, wk);
                if (u >= 6) o[u].y = fmaf(-b.x, wk.y, fmaf(-b.y, wk.x, -a.y));
            }
        }
        // (here, and not where the results are used)
#pragma unroll
        for (int u = 0; u < 12; ++u) asm volatile("" : "+v"(o[u].x), "+v"(o[u].y));
    };
    const bool has = k1 < KC, hasn = has && k1 != 0 && 2 * k1 != N1;
    const int64_t mstep = (int64_t)N1 * nlat * ld;
    auto store = [&](int tile) {
        int lat, group;
        walk.locate(tile, lat, group);
        const int row = group * 2 * FM_ROWS + r;
        float* const dp = xm + ((int64_t)k1 * nlat + lat) * ld + 2 * row;
        float* const dn = xm + ((int64_t)(N1 - k1) * nlat + lat) * ld + 2 * row;
        if ((group + 1) * 2 * FM_ROWS <= rows) {
#pragma unroll
            for (int u = 0; u < 12; ++u) {
                if ((u < 6 ? has : hasn) && (u < 6 ? k1 + N1 * u : N1 * (u - 5) - k1) < mmax) {
                    float* const dst = u < 6 ? dp + u * mstep : dn + (u - 6) * mstep;
                    *reinterpret_cast<float2*>(dst) = out[0][u];
                    *reinterpret_cast<float2*>(dst + 2 * FM_ROWS) = out[1][u];
                }
            }
        } else {                                           // the last group: zeros between the rows and ld
#pragma unroll
            for (int u = 0; u < 12; ++u) {
                if ((u < 6 ? has : hasn) && (u < 6 ? k1 + N1 * u : N1 * (u - 5) - k1) < mmax) {
                    float* const dst = u < 6 ? dp + u * mstep : dn + (u - 6) * mstep;
#pragma unroll
                    for (int half = 0; half < 2; ++half) {
                        const int rr = row + half * FM_ROWS;
                        if (2 * rr < ld) *reinterpret_cast<float2*>(dst + 2 * half * FM_ROWS) = rr < rows ? out[half][u] : make_float2(0.f, 0.f);
                    }
                }
            }
        }
    };

    request(t, 0);
    int done = -1;
    for (;;) {
        const int tn = t + walk.step;
        fm_barrier<true>();
        if (done >= 0) store(done);
        matrix_phase();
        fm_barrier<false>();
        request(t, 1);
        vector_phase(out[0]);
        fm_barrier<true>();
        matrix_phase();
        fm_barrier<false>();
        if (tn < walk.ntiles) request(tn, 0);
        vector_phase(out[1]);
        done = t;
        if (tn >= walk.ntiles) break;
        t = tn;
    }
    store(done);
}

// the kernels' N1, 0 if there are none for this length
int mat_n1(int n) {
    const int n1 = n / 32;
    return n % 32 == 0 && (n1 == 45 || n1 == 40 || n1 == 36) ? n1 : 0;
}

template <int N1>
int rfft_go(const FftPlan& p, const void* x, float* xm, int64_t rows, int nlat, int mmax, int ld, hipStream_t s) {
    const int ngroups = (ld / 4 + 7) / 8;
    const int per_xcd = (int)std::min<int64_t>((int64_t)((nlat + 7) / 8) * ngroups, std::max(1, 2 * p.n_cu / 8));
    hipLaunchKernelGGL((rfft_matrix_kernel<N1>), dim3((unsigned)(8 * per_xcd)), dim3(FM_THREADS), 0, s, reinterpret_cast<const bf16x8*>(p.d_mfrag), p.d_mtw,
                       reinterpret_cast<const unsigned short*>(x), xm, (int)rows, nlat, mmax, ld, ngroups);
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

unsigned short to_bf16(double v) {
    const float f = (float)v;
    unsigned u;
    std::memcpy(&u, &f, 4);
    return (unsigned short)((u + 0x7fffu + ((u >> 16) & 1)) >> 16);
}
double from_bf16(unsigned short h) {
    const unsigned u = (unsigned)h << 16;
    float f;
    std::memcpy(&f, &u, 4);
    return f;
}

}  // namespace

int fft_matrix_plan_init(FftPlan& p) {
    const int n1s = mat_n1(p.n);
    if (!n1s) return SFNO_OK;
    const int kc = n1s / 2 + 1, kt = (n1s + 31) / 32;
    // operand fragments: lane holds row 16 mt + lane % 16 (row 2 k1: cos, 2 k1 + 1: -sin), inputs 32 ks + 8 (lane / 16) + 0 ... 7
    std::vector<unsigned short> frag((size_t)3 * 3 * kt * 64 * 8, 0);
    for (int mt = 0; mt < 3; ++mt)
        for (int ks = 0; ks < kt; ++ks)
            for (int lane = 0; lane < 64; ++lane)
                for (int e = 0; e < 8; ++e) {
                    const int row = 16 * mt + lane % 16, k1 = row / 2, n1 = 32 * ks + 8 * (lane / 16) + e;
                    if (k1 >= kc || n1 >= n1s) continue;
                    const int q = k1 * n1 % n1s;
                    const bool zero = row % 2 && (2 * q) % n1s == 0;
                    const double a = kTwoPi * (double)q / (double)n1s;
                    double v = zero ? 0.0 : row % 2 ? -std::sin(a) : std::cos(a);
                    for (int part = 0; part < 3; ++part) {
                        const unsigned short b = to_bf16(v);
                        frag[((((size_t)part * 3 + mt) * kt + ks) * 64 + lane) * 8 + e] = b;
                        v -= from_bf16(b);
                    }
                }
    // twiddles between the stages, with the transform's factor 2 pi / n
    std::vector<float2> tw((size_t)kc * 32);
    for (int k1 = 0; k1 < kc; ++k1)
        for (int n2 = 0; n2 < 32; ++n2) {
            const double a = -kTwoPi * (double)(k1 * n2) / (double)p.n, f = kTwoPi / (double)p.n;
            tw[(size_t)k1 * 32 + n2] = make_float2((float)(f * std::cos(a)), (float)(f * std::sin(a)));
        }
    if (hipMalloc(&p.d_mfrag, sizeof(unsigned short) * frag.size()) != hipSuccess) return SFNO_ENOMEM;
    if (hipMalloc(&p.d_mtw, sizeof(float2) * tw.size()) != hipSuccess) return SFNO_ENOMEM;
    if (hipMemcpy(p.d_mfrag, frag.data(), sizeof(unsigned short) * frag.size(), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(p.d_mtw, tw.data(), sizeof(float2) * tw.size(), hipMemcpyHostToDevice) != hipSuccess)
        return SFNO_EHIP;
    return SFNO_OK;
}

// Bound by HBM latency and bandwidth together: 384 rows of 721 x 1440, 241 orders, 1.33 GB in 352 us (3.8 TB/s) where the vector kernel takes
// 491; 1536 rows, 121 orders 1098 / 1607; 128 rows of 361 x 1280, 200 orders 47 / 73.  (Per tile of a workgroup 5.0 k cycles of matrix phases,
// 5.0 vector phases, 2.5 stores, 3 waiting for rows.  Two threads per (row, k1) that exchange their sums: 424 us, with 60 % more vector
// instructions; asking for the next batch 600 cycles earlier, behind one more barrier: 368.)  Its error against 64 bits is the smaller one,
// 1.0e-7 against 1.1e-7.
bool rfft_matrix_supported(const FftPlan& p, const void* x, int64_t rows, int nlat, int mmax) {
    const int n1 = mat_n1(p.n);
    // orders up to N1 / 2 + 5 N1; 16-byte pieces; offsets within eight rows in 32 bits
    return n1 && mmax <= 5 * n1 + n1 / 2 + 1 && reinterpret_cast<uintptr_t>(x) % 16 == 0 && rows > 0 && rows < (1 << 30) && (int64_t)nlat * p.n < (1 << 27);
}

int rfft_matrix_launch(const FftPlan& p, const void* x, float* xm, int64_t rows, int nlat, int mmax, int ld, hipStream_t s) {
    switch (mat_n1(p.n)) {
        case 45: return rfft_go<45>(p, x, xm, rows, nlat, mmax, ld, s);
        case 40: return rfft_go<40>(p, x, xm, rows, nlat, mmax, ld, s);
        case 36: return rfft_go<36>(p, x, xm, rows, nlat, mmax, ld, s);
    }
    return SFNO_EUNSUPPORTED;
}

}  // namespace sfno
