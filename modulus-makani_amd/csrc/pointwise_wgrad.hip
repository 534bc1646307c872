// Weight gradient of the 1x1 convolution on bf16 NCHW activations:
//
//   dW[o][k] = sum_{b,p} g[b][o][p] x[b][k][p],      db[o] = sum_{b,p} g[b][o][p]
//
// (what autograd derives for nn.Conv2d(kernel_size=1), makani/models/common/layers.py:95-116,160-216).  Both operands are
// pixel-contiguous and the sum runs over the pixels, so a row of g is an A operand and a row of x a B operand of
// v_mfma_f32_32x32x16_bf16 as they lie in memory: 8 consecutive pixels per lane, no transposition.  The bias gradient
// is summed from the A fragments by the wavefronts that hold the first columns: as column K of the
// tiles it took a column of tiles to itself where K is a multiple of 256 (eight instead of six for 768 -> 384 channels with bias:
// 1249 -> 997 us at 721 x 1440).
//
// A workgroup (eight wavefronts, 4 x 2) owns a 256 x 256 tile (small layers: 128 x 128; wide ones: 384 x 192, pw_wgrad_wide_kernel) of dW and a contiguous share of the (sample, 64-pixel chunk)
// sequence.  Per chunk 256 rows of g and 256 rows of x, a whole 128-byte line each (with 64-byte pieces of 32-pixel chunks the
// same bytes were 1.4 times as long on their way, 989 against 704 us without the products for 384 -> 768 channels at 721 x 1440, and
// the kernel took as long as its loads: 1029 -> 902 us in all, 768 -> 384 with bias 997 -> 858),
// go straight from memory into LDS with global_load_lds_dwordx4 (issued from inline assembly with a
// counted wait, as in the forward kernel); a lane fetches the 16-byte piece whose LDS slot it owns, and the pieces of a row
// are permuted by (row >> 1) & 7 so that the 16-byte fragment reads of sixteen consecutive rows cover all banks.  A chunk is two
// halves, its rows of g and its rows of x, and LDS a ring of five of them: three are on their way while two are read.
// Pieces past the end of a sample come from a block of zeros.  Each wavefront multiplies
// 64 x 128 (two A and four B fragments per 16 pixels for eight matrix instructions).  The shares' partial tiles go to a
// workspace [share][O][K (+ 1 with bias)] and a second kernel adds them up in a fixed order: results do not depend on scheduling.
// All tiles of one share run on one XCD (workgroups are dealt to the XCDs round robin by linear id), where they meet
// the share's rows of g and x in L2.
#include "sfno_internal.h"

namespace sfno {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int WG_THREADS = 512;
constexpr int WG_PX = 64;             // pixels per chunk: eight 16-byte pieces per row
constexpr int WG_HALVES = 5;                                  // ring of halves
constexpr int WG_RSTEP = WG_THREADS / (WG_PX / 8);            // rows between a thread's pieces
static_assert(WG_PX == 64, "eight pieces per row: the permutation and the slot arithmetic below");
static_assert(WG_RSTEP % 16 == 0, "a thread's pieces share the permutation of their rows");

// tile of TILE rows (output channels) and columns (input channels) of dW per workgroup: 256, or 128 where the layer has no more or the
// tiles of 256 are few
template <int TILE>
struct WgTile {
    static constexpr int HALF = TILE * 2 * WG_PX;                    // bytes of the rows of g, or of x, of a chunk
    static constexpr int PIECES = HALF / (16 * WG_THREADS);          // 16-byte pieces per thread and half
    static constexpr int PER_CU = TILE == 256 ? 1 : 2;               // resident workgroups
    static constexpr int MT = TILE / 128, NT = TILE / 64;            // 32-row blocks of a wavefront (4 x 2 of them)
    static_assert(PER_CU * WG_HALVES * HALF <= 160 * 1024, "resident workgroups");
};

// source of the pieces that are not read from the tensors
__device__ __align__(16) const unsigned int wg_zero16[4] = {0u, 0u, 0u, 0u};

// 16 bytes per lane from global memory to LDS base + 16 lane (M0 carries the base; the compiler reserves M0 and does not
// accept it on a clobber list: nothing else in this file may depend on M0)
__device__ __forceinline__ void wg_dma16(const void* g, unsigned lds_byte_addr) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(lds_byte_addr) : "memory");
}

// s_waitcnt immediate: at most n vector memory operations in flight, no LDS operation
constexpr int wg_wait(int n) { return (n & 15) | ((n >> 4) << 14) | 0x70; }
// workgroup barrier behind such a wait; no LDS access moves across it
__device__ __forceinline__ void wg_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
}

// the same with a wavefront-uniform base and a 32-bit offset per lane
__device__ __forceinline__ void wg_dma16(const void* base, unsigned offset, unsigned lds_byte_addr) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(offset), "s"(base), "s"(lds_byte_addr) : "memory");
}

// tile of the second kernel: eight wavefronts of 96 x 96, 4 x 2
constexpr int WW_MT = 3, WW_NT = 3, WW_WO = 4, WW_WK = 2;
constexpr int WW_THREADS = 64 * WW_WO * WW_WK;
constexpr int WW_TO = 32 * WW_MT * WW_WO, WW_TK = 32 * WW_NT * WW_WK;

enum WgradKind { WG_SQUARE, WG_SMALL, WG_WIDE, WG_WIDE_SWAP };      // pw_wgrad_kernel<256>, <128>, pw_wgrad_wide_kernel<false>, <true>
struct WgradShape {
    int n_ot, n_kt, splits;
    int64_t cps, chunks;               // chunks per sample, chunks in all
    WgradKind kind;
    int rows() const { return kind == WG_SQUARE ? 512 : WW_TO + WW_TK; }     // that a workgroup asks for
};

// how the launcher and the workspace query divide the work: shares of at least four chunks, one workgroup per CU (all
// workgroups resident at once, the tiles of a share side by side on one XCD; small tiles: see wgrad_shape below)
static WgradShape wgrad_shape(int O, int K, int B, int64_t P, WgradKind kind) {
    const int to = kind == WG_SQUARE ? 256 : kind == WG_SMALL ? 128 : kind == WG_WIDE ? WW_TO : WW_TK;
    const int tk = kind == WG_SQUARE ? 256 : kind == WG_SMALL ? 128 : kind == WG_WIDE ? WW_TK : WW_TO;
    WgradShape s;
    s.kind = kind;
    s.n_ot = (O + to - 1) / to;
    s.n_kt = (K + tk - 1) / tk;
    s.cps = (P + WG_PX - 1) / WG_PX;
    s.chunks = s.cps * B;
    const int tiles = s.n_ot * s.n_kt;
    int64_t want = device_cus() / (kind == WG_SMALL ? ((O + 255) / 256) * ((K + 255) / 256) : tiles) / 8 * 8;
    if (want < 8) want = 8;
    const int64_t most = (s.chunks + 3) / 4;       // at least four chunks per share
    if (want > most) want = most;
    if (want < 1) want = 1;
    s.splits = (int)want;
    return s;
}

// Bytes a CU takes in: the rows its workgroup asks for (whole chunks of the longest share, and some three chunks' time until the first has landed), and
// its part of the partial sums, written and read by a kernel of their own (twice their bytes).  The kernel with fewer is the faster: 256 x 256 where
// both sides are at most 256 and where more shares cost more than fewer rows save (384 -> 192 channels at 4 x 120 x 240 45 us, 51 with
// 192 x 384; 73 -> 384 at 181 x 360 24.8, 28.9 with 384 x 192), else the side of 384 on the output or the input channels (384 -> 384 at 240 x 480
// 65 -> 59 us; more at pw_wgrad_wide_kernel).  Over 2045 shapes (8 to 768 channels, 512 pixels to 721 x 1440) the choice is within 0.9 % of the best
// on average; 35 lose more than 3 % to 256 x 256, 13 % at most, most of them with at most 128 input channels.
static double wgrad_cost(const WgradShape& s, int O, int K) {
    const int64_t share = (s.chunks + s.splits - 1) / s.splits;
    return 2.0 * s.rows() * WG_PX * (double)(share + 3) + 16.0 * O * K * s.splits / device_cus();
}
static WgradShape wgrad_shape(int O, int K, int B, int64_t P) {
    const WgradShape square = wgrad_shape(O, K, B, P, WG_SQUARE);
    WgradShape best = square;
    for (WgradKind kind : {WG_WIDE, WG_WIDE_SWAP}) {
        const WgradShape s = wgrad_shape(O, K, B, P, kind);
        if (wgrad_cost(s, O, K) < wgrad_cost(best, O, K)) best = s;
    }
    // Tiles of 128 x 128 over the shares of the 256 x 256 ones (the same sums in the same order), two workgroups to a CU: a layer of at most 128
    // channels asks for half the rows, and the way to the first chunk and the stores of a short share are spread over twice the workgroups.
    // 1000 shapes (2 to 768 channels, 1024 to 1.5 million pixels), times against the larger tiles: 0.66 where a tile takes the place of one, 0.74 to 0.95
    // for three in place of two, for two in place of one 0.75 with shares of less than 24 chunks and up to 1.19 with longer ones (but 0.7 with at most 64
    // output channels), for four 0.65 to 0.85 with shares of four chunks while all workgroups are resident at once, 0.97 to 1.07 past that and 1.2 with longer
    // shares.  20 % faster on average; of 1600 shapes two are more than 2 % slower (4 %: 250000 pixels and more, two in place of one).
    // 128 channels of 2 x 90 x 180 18.4 -> 12.6 us, 96 of 4 x 128 x 247 51 -> 36.
    const WgradShape small = wgrad_shape(O, K, B, P, WG_SMALL);
    const int n = small.n_ot * small.n_kt, n2 = square.n_ot * square.n_kt;
    const int64_t share = (square.chunks + square.splits - 1) / square.splits;
    const bool few = 2 * n <= 3 * n2;
    if (best.kind == WG_SQUARE ? few || (n <= 2 * n2 && (share < 24 || O <= 64)) || (share < 6 && n2 <= 6 && n * small.splits <= 2 * device_cus()) : few && share < 32) return small;
    return best;
}

struct WgradArgs {
    const unsigned short* G;           // bf16 [B][O][P]
    const unsigned short* X;           // bf16 [B][K][P]
    float* ws;                         // [splits][O][Kext]
    int O, K, Kext, B;
    int64_t P;
    int n_ot, n_kt, splits;
    int64_t cps, chunks;
};

// One stream per operand: the next chunk to ask for lies in sample ib at chunk ic of the sample.  Thread t asks for the piece at
// slot t + THREADS j of the rows' image in LDS (16 bytes a slot, eight to a row), j < PIECES: the thread's rows lie THREADS / 8 apart, a
// multiple of 16, and share their permutation.  Inside a sample the addresses are
// a scalar base and the lane's 32-bit offsets from the tile's first row; they are worked out in 64 bits for the last chunk of a
// sample, whose pieces may lie outside, and where the rows of a tile lie further apart than 32 bits reach.
template <int PIECES, int THREADS>
struct WgStream {
    static_assert(THREADS % 128 == 0, "a thread's pieces share the permutation of their rows");
    static constexpr int ROWS = PIECES * THREADS / 8;
    static_assert(ROWS <= 512, "32-bit offsets");
    static constexpr int64_t NEAR = ROWS <= 256 ? 1 << 23 : 1 << 22;      // ROWS rows of fewer values lie within 2^32 bytes
    const unsigned short* base;
    int r0, last;                  // first row of the tile, last row of the tensor
    int64_t ib, ic;
    unsigned off[PIECES];
    static __device__ __forceinline__ int part(int tid) { return (tid & 7) ^ ((tid >> 4) & 7); }
    __device__ __forceinline__ WgStream(const unsigned short* t, int first, int rows, const WgradArgs& a, int64_t c_begin, int tid)
        : base(t), r0(first), last(rows - 1), ib(c_begin / a.cps), ic(c_begin - ib * a.cps) {
        const unsigned row_bytes = (unsigned)(2 * a.P);
#pragma unroll
        for (int j = 0; j < PIECES; ++j) off[j] = (unsigned)min((tid >> 3) + THREADS / 8 * j, last - r0) * row_bytes + 16 * part(tid);
    }
    // dst: LDS address of the wavefront's first slot
    __device__ __forceinline__ void issue(const WgradArgs& a, unsigned dst, int tid) {
        const unsigned short* b = base + ((ib * (last + 1) + r0) * a.P + ic * WG_PX);
        if (a.P < NEAR && (ic + 1) * WG_PX <= a.P) {
            // (uniform, but the division by the chunks per sample left it in vector registers)
            const uint64_t bits = reinterpret_cast<uint64_t>(b);
            const void* ubase = reinterpret_cast<const void*>((uint64_t)__builtin_amdgcn_readfirstlane((int)(bits >> 32)) << 32 |
                                                              (unsigned)__builtin_amdgcn_readfirstlane((int)bits));
#pragma unroll
            for (int j = 0; j < PIECES; ++j) wg_dma16(ubase, off[j], dst + j * (THREADS * 16));
        } else {
            const bool in = ic * WG_PX + 8 * part(tid) < a.P;      // P is a multiple of 8: a piece lies inside the row or outside
#pragma unroll
            for (int j = 0; j < PIECES; ++j) {
                const unsigned short* p = b + (int64_t)min((tid >> 3) + THREADS / 8 * j, last - r0) * a.P + 8 * part(tid);
                wg_dma16(in ? p : reinterpret_cast<const unsigned short*>(wg_zero16), dst + j * (THREADS * 16));
            }
        }
        if (++ic == a.cps) {
            ic = 0;
            ++ib;
        }
    }
};

// (The comments speak of the 256 x 256 tile.)  grid = 8 * ceil(splits / 8) * n_ot * n_kt workgroups of 512 threads
template <int TILE>
__global__ __launch_bounds__(WG_THREADS, 2 * WgTile<TILE>::PER_CU) void pw_wgrad_kernel(WgradArgs a) {
    constexpr int HALF = WgTile<TILE>::HALF, PIECES = WgTile<TILE>::PIECES, MT = WgTile<TILE>::MT, NT = WgTile<TILE>::NT;
    __shared__ __align__(16) unsigned char lds[WG_HALVES * HALF];
    const int xcd = blockIdx.x & 7, q = blockIdx.x >> 3;
    const int tiles = a.n_ot * a.n_kt;
    const int split = (q / tiles) * 8 + xcd, tile = q % tiles;
    if (split >= a.splits) return;
    const int o0 = (tile % a.n_ot) * TILE, k0 = (tile / a.n_ot) * TILE;
    const int64_t c_begin = (int64_t)split * a.chunks / a.splits, c_end = (int64_t)(split + 1) * a.chunks / a.splits;
    const int nch = (int)(c_end - c_begin);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wo = wave & 3, wk = wave >> 2;
    const unsigned lds0 = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)lds);

    // ---- loads: LDS slot s = 512 j + tid of a half (16 bytes) holds row s >> 3, piece (s & 7) ^ ((row >> 1) & 7).  A thread's
    // slots lie 64 rows apart: same piece, same permutation.  Rows past the matrix are its last row, whose products are never stored.
    WgStream<PIECES, WG_THREADS> sg(a.G, o0, a.O, a, c_begin, tid), sx(a.X, k0, a.K, a, c_begin, tid);
    auto issue = [&](WgStream<PIECES, WG_THREADS>& t, int slot) { t.issue(a, lds0 + slot * HALF + wave * 1024, tid); };

    f32x16 acc[MT][NT];
    float accb[MT] = {}, chunkb[MT] = {};       // sums of the lane's pixels of its two rows: all chunks, this chunk
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[mt][nt][v] = 0.f;

    // fragments of this lane: row (lane & 31) of a 32-row block, pieces 2 ks + (lane >> 5) of the row (pixels 8 (lane >> 5) .. + 7 of
    // the 16-pixel step ks), at their permuted places
    const int sw = (lane >> 1) & 7, kg = lane >> 5;
    const unsigned fa = (wo * 32 * MT + (lane & 31)) * 128, fb = (wk * 32 * NT + (lane & 31)) * 128;

    const bool live = o0 + wo * 32 * MT < a.O && k0 + wk * 32 * NT < a.K;
    const bool bias = a.Kext > a.K && k0 + wk * 32 * NT == 0;
    // Half h (chunk h / 2; g, then x) lives in slot h % 5.  Fragments are read one 16-pixel step ahead of the matrix instructions, those of
    // a chunk's first step under the products of the last step of the chunk before.  In front of that, once a wavefront holds all it
    // needs of chunk i, it waits for its pieces of chunk i + 1 and meets the others: chunk i's slots take halves 2 i + 5 (x of chunk
    // i + 2) and 2 i + 6 (g of chunk i + 3), chunk i + 1 may be read.  The only vector memory operations of the loop are the PIECES loads per
    // wavefront and half, so "at most PIECES outstanding" leaves half 2 i + 4 under way.
    static_assert(WG_HALVES == 5, "the wait counts below");
    bf16x8 af[2][MT], bf[2][NT];               // [step & 1][32-row block]
    auto fragments = [&](int slot_g, int slot_x, int ks) {
        const unsigned pk = (unsigned)(((2 * ks + kg) ^ sw) * 16);
        const unsigned char *pa = lds + slot_g * HALF + fa + pk, *pb = lds + slot_x * HALF + fb + pk;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) af[ks & 1][mt] = *reinterpret_cast<const bf16x8*>(pa + mt * 32 * 128);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) bf[ks & 1][nt] = *reinterpret_cast<const bf16x8*>(pb + nt * 32 * 128);
    };
    auto products = [&](int ks) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[ks & 1][mt], bf[ks & 1][nt], acc[mt][nt], 0, 0, 0);
        if (bias) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const u32x4 p = __builtin_bit_cast(u32x4, af[ks & 1][mt]);
                float lo = 0.f, hi = 0.f;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    lo += __uint_as_float(p[i] << 16);
                    hi += __uint_as_float(p[i] & 0xffff0000u);
                }
                chunkb[mt] += lo + hi;
                if (ks == 3) {
                    accb[mt] += chunkb[mt];
                    chunkb[mt] = 0.f;
                }
            }
        }
    };
    issue(sg, 0);
    issue(sx, 1);
    if (nch > 1) {
        issue(sg, 2);
        issue(sx, 3);
    }
    if (nch > 2) issue(sg, 4);
    __builtin_amdgcn_sched_barrier(0);
    if (nch > 2)
        __builtin_amdgcn_s_waitcnt(wg_wait(3 * PIECES));
    else
        __builtin_amdgcn_s_waitcnt(wg_wait(0));
    wg_barrier();
    int cg = 0, cx = 1;                       // slots of chunk i
    // (a wavefront whose 64 x 128 part of the tile lies outside the matrix only moves data)
    if (live) fragments(cg, cx, 0);
    for (int i = 0; i < nch; ++i) {
        if (live) {
#pragma unroll
            for (int ks = 0; ks < 3; ++ks) {
                fragments(cg, cx, ks + 1);
                __builtin_amdgcn_sched_barrier(0);
                products(ks);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // (the builtin and not inline assembly: the compiler then knows that the fragments have arrived)
        if (i + 3 <= nch)
            __builtin_amdgcn_s_waitcnt(wg_wait(PIECES));
        else
            __builtin_amdgcn_s_waitcnt(wg_wait(0));
        wg_barrier();
        if (i + 2 < nch) issue(sx, cg);
        if (i + 3 < nch) issue(sg, cx);
        cg = cg >= 3 ? cg - 3 : cg + 2;
        cx = cx >= 3 ? cx - 3 : cx + 2;
        if (live) {
            fragments(cg, cx, 0);             // (past the last chunk: whatever those slots hold, and not used)
            __builtin_amdgcn_sched_barrier(0);
            products(3);
        }
    }

    // D layout of the 32x32 MFMA: register v of lane j holds D[8 (v / 4) + 4 (j / 32) + v % 4][j % 32]
    float* out = a.ws + (int64_t)split * a.O * a.Kext;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int kk = k0 + wk * 32 * NT + nt * 32 + (lane & 31);
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int o = o0 + wo * 32 * MT + mt * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                if (o < a.O && kk < a.K) out[(int64_t)o * a.Kext + kk] = acc[mt][nt][v];
            }
        }
    if (bias) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int o = o0 + wo * 32 * MT + mt * 32 + (lane & 31);
            const float b = accb[mt] + __shfl_xor(accb[mt], 32, 64);
            if (lane < 32 && o < a.O) out[(int64_t)o * a.Kext + a.K] = b;
        }
    }
}

// The same with tiles of 384 x 192 and wavefronts of 96 x 96 (3 x 3 matrix instructions from six fragments instead of 2 x 4 from six).
// LDS holds two chunks of 576 rows; the one after next is asked for when the last fragments of a chunk have been read, and has a whole
// chunk's products to land.
// A CU's intake bounds both kernels: memory is read once (2.40 GB for 768 -> 384 channels at 721 x 1440, 736 us), yet a chunk's 72 KiB take 2.7 us
// with nothing else in the loop (694 us), the products alone 425; lines in L2 ahead of their requests, or a share's lines next to
// its neighbours', made it no faster.  So the tile that asks for fewer rows is the better one: four tiles of 576 rows for 384 x 768 where the other
// kernel has six of 512 (384 -> 768 1034 -> 843 us, 768 -> 384 873 -> 736, 384 -> 384 546 -> 407, 384 -> 73 265 -> 198, all at
// 721 x 1440).  Larger tiles (384 x 256) do not fit the registers.
// SWAP: the 384 are input channels, the 192 output channels; a share's partial sums are stored transposed, [K (+ 1 with bias)][O], so that a
// wavefront writes whole lines (written to [O][K] 384 -> 192 at 4 x 120 x 240 took 92 us).
template <bool SWAP>
__global__ __launch_bounds__(WW_THREADS, 2) void pw_wgrad_wide_kernel(WgradArgs a) {
    constexpr int MT = WW_MT, NT = WW_NT, ROW = 2 * WG_PX, BUF = (WW_TO + WW_TK) * ROW;
    constexpr int PA = WW_TO * ROW / (16 * WW_THREADS), PB = WW_TK * ROW / (16 * WW_THREADS);
    static_assert(PA * 16 * WW_THREADS == WW_TO * ROW && PB * 16 * WW_THREADS == WW_TK * ROW && 2 * BUF <= 160 * 1024, "whole pieces, two chunks in LDS");
    __shared__ __align__(16) unsigned char lds[2 * BUF];
    const int xcd = blockIdx.x & 7, q = blockIdx.x >> 3;
    const int tiles = a.n_ot * a.n_kt;
    const int split = (q / tiles) * 8 + xcd, tile = q % tiles;
    if (split >= a.splits) return;
    const int ot = tile % a.n_ot, kt = tile / a.n_ot;
    // rows of the first operand (384 of them) and of the second, and the tile's first ones
    const int RA = SWAP ? a.K : a.O, RB = SWAP ? a.O : a.K;
    const int a0 = (SWAP ? kt : ot) * WW_TO, b0 = (SWAP ? ot : kt) * WW_TK;
    const int64_t c_begin = (int64_t)split * a.chunks / a.splits, c_end = (int64_t)(split + 1) * a.chunks / a.splits;
    const int nch = (int)(c_end - c_begin);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wo = wave % WW_WO, wk = wave / WW_WO;
    const unsigned lds0 = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)lds) + wave * 1024;
    WgStream<PA, WW_THREADS> sa(SWAP ? a.X : a.G, a0, RA, a, c_begin, tid);
    WgStream<PB, WW_THREADS> sb(SWAP ? a.G : a.X, b0, RB, a, c_begin, tid);
    auto issue = [&](int buf) {
        sa.issue(a, lds0 + buf * BUF, tid);
        sb.issue(a, lds0 + buf * BUF + WW_TO * ROW, tid);
    };

    f32x16 acc[MT][NT];
    static_assert(MT == NT, "as many row blocks of g in either order");
    float accb[MT], chunkb[MT];               // sums of the lane's pixels of its rows of g: all chunks, this chunk
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        accb[mt] = chunkb[mt] = 0.f;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[mt][nt][v] = 0.f;
    }
    const int ro = wo * MT * 32, rk = wk * NT * 32;
    const int sw = (lane >> 1) & 7, kg = lane >> 5;
    const unsigned fa = (ro + (lane & 31)) * ROW, fb = (WW_TO + rk + (lane & 31)) * ROW;
    const bool live = a0 + ro < RA && b0 + rk < RB;
    const bool bias = a.Kext > a.K && (SWAP ? a0 + ro : b0 + rk) == 0;
    bf16x8 af[2][MT], bf[2][NT];              // [step & 1][32-row block]
    auto fragments = [&](int buf, int ks) {
        const unsigned char* p = lds + buf * BUF + (unsigned)(((2 * ks + kg) ^ sw) * 16);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) af[ks & 1][mt] = *reinterpret_cast<const bf16x8*>(p + fa + mt * 32 * ROW);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) bf[ks & 1][nt] = *reinterpret_cast<const bf16x8*>(p + fb + nt * 32 * ROW);
    };
    auto products = [&](int ks) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[ks & 1][mt], bf[ks & 1][nt], acc[mt][nt], 0, 0, 0);
        if (bias) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const u32x4 p = __builtin_bit_cast(u32x4, SWAP ? bf[ks & 1][mt] : af[ks & 1][mt]);
                float lo = 0.f, hi = 0.f;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    lo += __uint_as_float(p[i] << 16);
                    hi += __uint_as_float(p[i] & 0xffff0000u);
                }
                chunkb[mt] += lo + hi;
                if (ks == 3) {
                    accb[mt] += chunkb[mt];
                    chunkb[mt] = 0.f;
                }
            }
        }
    };
    issue(0);
    if (nch > 1) issue(1);
    __builtin_amdgcn_sched_barrier(0);
    if (nch > 1)
        __builtin_amdgcn_s_waitcnt(wg_wait(PA + PB));
    else
        __builtin_amdgcn_s_waitcnt(wg_wait(0));
    wg_barrier();
    if (live) fragments(0, 0);
    for (int i = 0; i < nch; ++i) {
        if (live) {
#pragma unroll
            for (int ks = 0; ks < 3; ++ks) {
                fragments(i & 1, ks + 1);
                __builtin_amdgcn_sched_barrier(0);
                products(ks);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // this wavefront holds all it needs of chunk i, and its pieces of chunk i + 1 (all that is under way) have landed
        __builtin_amdgcn_s_waitcnt(wg_wait(0));
        wg_barrier();
        if (i + 2 < nch) issue(i & 1);
        if (live) {
            fragments((i + 1) & 1, 0);        // (past the last chunk: whatever that buffer holds, and not used)
            __builtin_amdgcn_sched_barrier(0);
            products(3);
        }
    }

    float* out = a.ws + (int64_t)split * a.O * a.Kext;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int rb = b0 + rk + nt * 32 + (lane & 31);
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int ra = a0 + ro + mt * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                if (ra < RA && rb < RB) out[(int64_t)ra * (SWAP ? a.O : a.Kext) + rb] = acc[mt][nt][v];
            }
        }
    if (bias) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int o = (SWAP ? b0 + rk : a0 + ro) + mt * 32 + (lane & 31);
            const float b = accb[mt] + __shfl_xor(accb[mt], 32, 64);
            if (lane < 32 && o < a.O) out[SWAP ? (int64_t)a.K * a.O + o : (int64_t)o * a.Kext + a.K] = b;
        }
    }
}

// dW[o][k] = sum over the shares, in a fixed order; column K goes to db.  A workgroup's 16 wavefronts take every 16th share each of
// the same 64 V entries and meet in LDS: latency is what bounds small matrices (up to 256 shares of 73 x 73 entries; one thread per
// four entries walked all shares in turn: both kernels 145 us for 73 -> 73 channels at 2 x 181 x 360, now 20; 128 -> 256 with bias 45 -> 35).  V = 4 entries per lane (16-byte loads; a share must then start on
// 16 bytes) where that still makes 256 workgroups, else one.
constexpr int WR_WAVES = 16;
template <int V>
__global__ __launch_bounds__(64 * WR_WAVES) void pw_wgrad_reduce_kernel(const float* __restrict__ ws, float* __restrict__ dW, float* __restrict__ db, int O,
                                                                        int K, int Kext, int64_t n, int splits, bool swap) {
    typedef float vec __attribute__((ext_vector_type(V)));
    __shared__ __align__(16) float part[WR_WAVES][64 * V];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t base = (int64_t)blockIdx.x * (64 * V), idx = base + V * lane;
    vec acc = (vec)(0.f);
    if (idx < n) {
#pragma unroll 4
        for (int i = wave; i < splits; i += WR_WAVES) acc += *reinterpret_cast<const vec*>(ws + (int64_t)i * n + idx);
    }
    *reinterpret_cast<vec*>(&part[wave][V * lane]) = acc;
    __syncthreads();
    const int64_t e = base + threadIdx.x;
    if (threadIdx.x >= 64 * V || e >= n) return;
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < WR_WAVES; ++w) s += part[w][threadIdx.x];
    const int inner = swap ? O : Kext;             // partial sums lie as [O][Kext] or [Kext][O]
    const int64_t i = e / inner, j = e - i * inner, o = swap ? j : i, k = swap ? i : j;
    if (k < K)
        dW[o * K + k] = s;
    else if (db)
        db[o] = s;
}

size_t pointwise_wgrad_workspace_bytes(int O, int K, int has_bias, int B, int64_t P) {
    const int Kext = K + (has_bias ? 1 : 0);
    const WgradShape s = wgrad_shape(O, K, B, P);
    return sizeof(float) * (size_t)s.splits * (size_t)O * (size_t)Kext;
}

int pointwise_wgrad_launch(const unsigned short* g, const unsigned short* x, float* dW, float* db, int B, int K, int O, int64_t P, float* ws,
                           size_t ws_bytes, hipStream_t s) {
    if (P < 8 || P % 8) return SFNO_EINVAL;
    const int Kext = K + (db ? 1 : 0);
    const WgradShape sh = wgrad_shape(O, K, B, P);
    if (ws_bytes < sizeof(float) * (size_t)sh.splits * (size_t)O * (size_t)Kext) return SFNO_EINVAL;
    WgradArgs a;
    a.G = g; a.X = x; a.ws = ws;
    a.O = O; a.K = K; a.Kext = Kext; a.B = B; a.P = P;
    a.n_ot = sh.n_ot; a.n_kt = sh.n_kt; a.splits = sh.splits; a.cps = sh.cps; a.chunks = sh.chunks;
    const int64_t nwg = 8 * (int64_t)((sh.splits + 7) / 8) * sh.n_ot * sh.n_kt;
    if (nwg > 0x7fffffffLL) return SFNO_EUNSUPPORTED;
    if (sh.kind == WG_WIDE)
        hipLaunchKernelGGL(pw_wgrad_wide_kernel<false>, dim3((unsigned)nwg), dim3(WW_THREADS), 0, s, a);
    else if (sh.kind == WG_WIDE_SWAP)
        hipLaunchKernelGGL(pw_wgrad_wide_kernel<true>, dim3((unsigned)nwg), dim3(WW_THREADS), 0, s, a);
    else if (sh.kind == WG_SMALL)
        hipLaunchKernelGGL(pw_wgrad_kernel<128>, dim3((unsigned)nwg), dim3(WG_THREADS), 0, s, a);
    else
        hipLaunchKernelGGL(pw_wgrad_kernel<256>, dim3((unsigned)nwg), dim3(WG_THREADS), 0, s, a);
    if (hipGetLastError() != hipSuccess) return SFNO_EHIP;
    const int64_t n = (int64_t)O * Kext;
    if (n % 4 == 0 && n >= 256 * 256)
        hipLaunchKernelGGL(pw_wgrad_reduce_kernel<4>, dim3((unsigned)((n + 255) / 256)), dim3(64 * WR_WAVES), 0, s, ws, dW, db, O, K, Kext, n, sh.splits, sh.kind == WG_WIDE_SWAP);
    else
        hipLaunchKernelGGL(pw_wgrad_reduce_kernel<1>, dim3((unsigned)((n + 63) / 64)), dim3(64 * WR_WAVES), 0, s, ws, dW, db, O, K, Kext, n, sh.splits, sh.kind == WG_WIDE_SWAP);
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

}  // namespace sfno
