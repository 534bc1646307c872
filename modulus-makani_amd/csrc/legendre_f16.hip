// Equator-folded Legendre contractions with fp32 accuracy on the fp16 matrix pipe of gfx950 (the default fp32 path):
//
//   analysis : spec[m][l][n] = sum_k W[m][l][k] xm[m][k][n]     (RealSHT.forward, Legendre stage)
//   synthesis: xm[m][k][n]   = sum_l P[m][l][k] spec[m][l][n]   (InverseRealSHT.forward, Legendre stage)
//
// Work decomposition, table streams, equator fold and the omitted polar chunks are those of legendre_fold.hip: a
// workgroup has four wavefronts = 2 parities x 2 row blocks of 32 table rows, owns NT 32-wide column tiles and walks K
// in chunks of 16.  What differs is the arithmetic.  An fp32 number scaled by a power of two into the range of fp16 is,
// to 22 of its 24 significant bits, the sum of two fp16 numbers; with both operands cut that way a product needs three
// v_mfma_f32_32x32x16_f16 (t0 q0 + t0 q1 + t1 q0; t1 q1 is below 2^-21 of the product), each exact in the fp32
// accumulator, where three exact bf16 parts need six.
//   table: cut on the host from the float64 value (both parts rounded to nearest, so 23 bits are kept), one power-of-two
//          scale per table row that brings the row's largest entry to [2^14, 2^15); 4 bytes per entry in the stream;
//   panel: cut once per workgroup by the wavefronts that stage it -- sums and differences of mirrored latitude rows
//          (analysis) or the degree rows of the two parities (synthesis) go to LDS as two fp16 planes in the order the
//          matrix instruction wants its B operand (16-byte fragment reads, no arithmetic in the matrix phase) -- with one
//          power-of-two scale per column.  The scale of a column is found while the column streams by: the staging
//          wavefronts keep a bound on its exponent, raise it (leaving a few bits of headroom) when a chunk exceeds it and
//          publish the bound with the chunk; a wavefront whose column's bound moved rescales that column's partial sums,
//          which is exact.
// What bounds it: the panels' way from L2.  With the panel loads left out a kernel of 200 us took 157 (no matrix
// instructions: 180; no cut: 180; loads two chunks ahead: no gain), so a lane asks for four columns at once and a
// wavefront for whole 128-byte pieces of a row (a float per lane before): analysis of 384 rows, 721 latitudes, 240
// degrees 162 -> 134 us, synthesis 199 -> 171; 240 latitudes 62 -> 55 and 76 -> 62; 73 rows, 721 degrees 196 -> 185
// and 200 -> 205, before the choice of tiles (see launch_f16).
// Entries more than 2^17 below the largest entry of their column (row) keep fewer bits, so the error bound is
// 2^-21 |t q| + 2^-38 max|t| max|q| per product where fp32 arithmetic has 2^-24 |t q|; the transform's own longitude
// FFT has an error of that second kind already (relative to the largest value of a latitude row).
#include "sfno_internal.h"

namespace sfno {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef int i4 __attribute__((ext_vector_type(4)));

constexpr int LH_TOP = 14;             // scaled magnitudes stay below 2^(TOP + 1)
constexpr int LH_HEAD = 3;             // bits of headroom left when a column's exponent bound is raised
constexpr int LH_SH = LH_TOP + 127;    // scaled = x * 2^(SH - E), E = biased exponent bound of the column
constexpr int LH_EMIN = LH_SH - 127;   // smallest bound: its scale is the largest power of two of fp32 (columns below 2^-112 keep 25 bits above 2^-151)

// resident workgroups per CU: set by the 16 NT accumulator registers and the staged rows held across the matrix phase
constexpr int lh_occupancy(int nt) { return nt <= 4 ? 4 : 3; }

// COEFFS: the spectral side is the reference layout, complex [rows][lmax][mmax] (zeros above the diagonal included), and no layout pass
// runs: an order's values lie 8 mmax bytes apart there, eight bytes at a time, so this is for small transforms only (legendre_coeffs_fit).
template <int NT, bool ANALYSIS, bool COEFFS>
__global__ __launch_bounds__(256, lh_occupancy(NT)) void legendre_f16_kernel(PgemmArgs a) {
    constexpr int TN = 32 * NT;            // columns per workgroup
    constexpr int QN = TN / 4;             // column quads
    // LDS image of one (buffer, panel, plane): column c = 4 j + cc lives in class cc at slot j; a slot is the column's 16 k
    // values (32 bytes); classes are CS bytes apart with CS = 128 mod 256, and the two 16-byte halves of a slot swap places in
    // classes 2 and 3, so that the 16-byte fragment reads of 16 consecutive columns cover all banks
    constexpr int CS = QN * 32 + 128;
    constexpr int PLANE = 4 * CS;
    constexpr int PLANES = 2 * 2 * 2 * PLANE < 18432 ? 18432 : 2 * 2 * 2 * PLANE;      // [buffer][panel][plane]; at least the four tiles of 32 x 36 floats of the parity exchange
    __shared__ __align__(16) unsigned char planes[PLANES];
    __shared__ __align__(16) int expo[2][2][TN];   // [buffer][panel][column]: exponent bound the chunk was cut with

    // Workgroups go to the 8 XCDs round-robin by linear id and entry 8 i + x of the work list is meant for XCD x: the
    // column tiles of one entry run back to back on that XCD, where they share the entry's table fragments in L2.
    const int nct = (a.ld + TN - 1) / TN;
    const int qid = blockIdx.x >> 3;
    const int ct = qid % nct;
    // (the record is read through the scalar unit: one 64-byte request, wavefront-uniform)
    const __attribute__((address_space(4))) int64_t* wrec =
        reinterpret_cast<const __attribute__((address_space(4))) int64_t*>(reinterpret_cast<uintptr_t>(a.wrec)) + (int64_t)((qid / nct) * 8 + (blockIdx.x & 7)) * PG_WREC;
    int64_t rec[PG_WREC];
#pragma unroll
    for (int i = 0; i < PG_WREC; ++i) rec[i] = wrec[i];
    const int m = (int)rec[PG_WREC_M];
    if (m < 0) return;
    // (leading row blocks of the order that its consumer takes for zero)
    const int dropped = !ANALYSIS && a.drop ? (int)(rec[PG_WREC_M] >> 32) : 0;
    if (!ANALYSIS && (int)rec[PG_WREC_RB] + 2 <= dropped) return;
    const int2 wi = make_int2(m, (int)rec[PG_WREC_RB]);
    __builtin_amdgcn_s_setreg((1 << 11) | (2 << 6) | 1, 3);      // MODE[3:2]: conversions to fp16 round toward zero
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    // wavefront w runs on SIMD w; alternate which SIMDs get the (possibly absent) second row block
    // and the (one row shorter) odd parity from workgroup to workgroup
    const int wslot = (wave + qid) & 3;
    const int par = wslot >> 1, rb = wi.y + (wslot & 1);
    const int n0 = ct * TN;
    const int ld = a.ld, nlat = a.nlat, lmax = a.lmax;
    if (n0 >= ld) return;
    const int K2 = (nlat + 1) >> 1;
    const int nl0 = (lmax - m > 0) ? (lmax - m + 1) >> 1 : 0;          // degrees of parity 0: l = m, m+2, ...
    const int nl1 = (lmax - m - 1 > 0) ? (lmax - m) >> 1 : 0;          // parity 1: l = m+1, m+3, ...
    const int nlp = par ? nl1 : nl0;

    const int nrows = ANALYSIS ? nlp : K2;
    const int nrb = (nrows + PG_ROWS - 1) / PG_ROWS;
    const int nc = ANALYSIS ? (K2 + PG_KC - 1) / PG_KC : (nl0 + PG_KC - 1) / PG_KC;
    const bool active = rb < nrb && rb >= dropped;

    const float* xm_m = (ANALYSIS ? a.Q : a.Out) + (int64_t)m * nlat * ld;     // Fourier panel of order m
    const float* sp_m = (ANALYSIS ? a.Out : a.Q) + (COEFFS ? 2 * (int64_t)m : (int64_t)m * lmax * ld);     // spectral panel of order m
    const int nval = COEFFS ? a.ncol : ld;         // columns with values on the spectral side
    const uint32_t srow = COEFFS ? 2u * a.mmax : (uint32_t)ld;       // floats from degree to degree, and the column's offset
    const int live = min(NT, (ld - n0 + 31) >> 5);         // tiles with columns
    auto scolumn = [&](int n) { return COEFFS ? (uint32_t)(n >> 1) * (uint32_t)lmax * srow + (uint32_t)(n & 1) : (uint32_t)n; };
    // Index entry of a row block: first block of its stream | leading chunks left out << 48 (their entries are negligible:
    // towards the poles the table falls off like sin^m(theta)).  The K loop of the workgroup starts at the smallest such
    // count of its (up to) four row blocks; a wavefront joins in at its own.
    constexpr int APB = 128;               // 16-byte pieces per block: two planes x 64 lanes
    // (the work record holds the entries of the four streams -- nc << 48 for one that does not exist: an order without
    // degrees, synthesis with mmax > lmax, has none, its rows are zero-filled below -- and the parities' first positions)
    auto entry_pos = [&](int p_, int rb_) { return (p_ ? rec[PG_WREC_POS + 1] : rec[PG_WREC_POS]) + rb_; };
    int cstart = nc;
#pragma unroll
    for (int s_ = 0; s_ < 4; ++s_) cstart = min(cstart, (int)(rec[PG_WREC_ENTRY + s_] >> 48));
    const int64_t my_entry = par ? ((wslot & 1) ? rec[PG_WREC_ENTRY + 3] : rec[PG_WREC_ENTRY + 2]) : ((wslot & 1) ? rec[PG_WREC_ENTRY + 1] : rec[PG_WREC_ENTRY]);
    cstart = max(cstart, 0);
    const int c0w = min(max((int)(my_entry >> 48), 0), nc);   // nc for a wavefront without a row block or with nothing but negligible entries
    const f4* apv = reinterpret_cast<const f4*>(a.A) + ((c0w < nc ? my_entry & (((int64_t)1 << 48) - 1) : (int64_t)0) * APB + lane);

    floatx16 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[t][v] = 0.0f;
    int erun[NT];                          // exponent bound my partial sums of tile t are scaled with (per lane = column)
#pragma unroll
    for (int t = 0; t < NT; ++t) erun[t] = LH_EMIN;

    // ---- staging: a wavefront takes a column tile, a lane four columns and RPL consecutive rows of the chunk in both panels: eight
    // lanes ask for one 128-byte piece of a row.  Up to four tiles there is a wavefront for each; of five the first wavefront takes
    // two, 32 lanes and four rows each.
    constexpr int RPL = NT <= 4 ? 2 : 4;   // rows per lane
    constexpr int RG = PG_KC / RPL;        // row groups: lanes that share a column
    const int stile = NT <= 4 ? wave : lane < 32 ? wave : wave + 4;
    const bool stager = stile < live;
    const int rg = (lane >> 3) & (RG - 1);
    const int slot = min(stile, NT - 1) * 8 + (lane & 7);      // column quad of the tile
    float q[2][RPL][4];
    const char* qpanel = reinterpret_cast<const char*>(ANALYSIS ? xm_m : sp_m);
    const uint32_t qstep = (ANALYSIS ? (uint32_t)ld : srow) * 4u;
    const int sn = n0 + 4 * slot;
    constexpr bool PAIRS = COEFFS && !ANALYSIS;                // columns come as (re, im) pairs of a row
    const int sna = PAIRS ? min(sn, nval - 2) : min(sn, ld - 4), snb = PAIRS ? min(sn + 2, nval - 2) : 0;
    const uint32_t qca = (PAIRS ? scolumn(sna) : (uint32_t)sna) * 4u, qcb = PAIRS ? scolumn(snb) * 4u : 0u;
    // offsets of my first row in chunk 0 and of the last row walked; a wavefront without a tile reads row 0 only
    const uint32_t qfirst = (uint32_t)(ANALYSIS ? RPL * rg : m + 2 * RPL * rg) * qstep, qlast = stager ? (uint32_t)(ANALYSIS ? K2 - 1 : lmax - 1) * qstep : 0u;
    const uint32_t qtop = (uint32_t)(nlat - 1) * qstep;
    auto q_at = [&](uint32_t off, float (&v)[4]) {
        if constexpr (PAIRS) {
            const float2 x = *reinterpret_cast<const float2*>(qpanel + (size_t)(off + qca)), y = *reinterpret_cast<const float2*>(qpanel + (size_t)(off + qcb));
            v[0] = x.x; v[1] = x.y; v[2] = y.x; v[3] = y.y;
        } else {
            const float4 x = *reinterpret_cast<const float4*>(qpanel + (size_t)(off + qca));
            v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
        }
    };
    auto q_load = [&](int c) {
        const uint32_t off = qfirst + (uint32_t)((ANALYSIS ? PG_KC : 2 * PG_KC) * c) * qstep;
#pragma unroll
        for (int r = 0; r < RPL; ++r) {
            if (ANALYSIS) {
                const uint32_t o = min(off + r * qstep, qlast);
                q_at(o, q[0][r]);
                q_at(qtop - o, q[1][r]);
            } else {
                q_at(min(off + 2 * r * qstep, qlast), q[0][r]);
                q_at(min(off + (2 * r + 1) * qstep, qlast), q[1][r]);
            }
        }
    };
    // largest exponent of my values of a column; an excess over the bound of any column of the wavefront is rare
    auto exponents = [&](const float (&v)[RPL][4], int (&eb)[4]) {
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) {
            float mx;
            asm("v_max_f32 %0, |%1|, |%2|" : "=v"(mx) : "v"(v[0][cc]), "v"(v[1][cc]));
#pragma unroll
            for (int r = 2; r < RPL; ++r) asm("v_max_f32 %0, %1, |%2|" : "=v"(mx) : "v"(mx), "v"(v[r][cc]));
            eb[cc] = __builtin_bit_cast(int, mx) >> 23;
        }
    };
    auto raise = [&](const int (&eb_)[4], i4& E) {
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) {
            int eb = eb_[cc];
#pragma unroll
            for (int d = 8; d < 8 * RG; d <<= 1) eb = max(eb, __shfl_xor(eb, d, 64));
            E[cc] = eb > E[cc] ? eb + LH_HEAD : E[cc];
        }
    };
    const uint32_t dpos = slot * 32 + (RPL == 2 ? (rg & 3) * 4 : (rg & 1) * 8), dhalf = (RPL == 2 ? rg >> 2 : rg >> 1) * 16;
    const uint32_t dst01 = dpos + dhalf, dst23 = dpos + (dhalf ^ 16);
    // one panel's values of my columns: scale, cut, write
    auto cut_store = [&](unsigned char* pl0, const float (&v)[RPL][4], const i4& E) {
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) {
            const float sc = __builtin_bit_cast(float, (unsigned)(LH_SH + 127 - E[cc]) << 23);
            unsigned char* dst = pl0 + cc * CS + (cc < 2 ? dst01 : dst23);
            unsigned hi[RPL / 2], lo[RPL / 2];
#pragma unroll
            for (int e = 0; e < RPL / 2; ++e) {
                asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(hi[e]) : "v"(v[2 * e][cc]), "v"(sc));
                asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(hi[e]) : "v"(v[2 * e + 1][cc]), "v"(sc));
                asm("v_fma_mixlo_f16 %0, %1, %2, -%3 op_sel_hi:[0,0,1]" : "=v"(lo[e]) : "v"(v[2 * e][cc]), "v"(sc), "v"(hi[e]));
                asm("v_fma_mixhi_f16 %0, %1, %2, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "+v"(lo[e]) : "v"(v[2 * e + 1][cc]), "v"(sc), "v"(hi[e]));
            }
            if constexpr (RPL == 2) {
                *reinterpret_cast<unsigned*>(dst) = hi[0];
                *reinterpret_cast<unsigned*>(dst + PLANE) = lo[0];
            } else {
                *reinterpret_cast<uint2*>(dst) = make_uint2(hi[0], hi[RPL / 2 - 1]);
                *reinterpret_cast<uint2*>(dst + PLANE) = make_uint2(lo[0], lo[RPL / 2 - 1]);
            }
        }
    };
    auto q_store = [&](int buf, int c) {
        if (!stager) return;
        // chunks that touch neither end of the K range need no masks
        const bool plain = ANALYSIS ? (c + 1) * PG_KC < K2 : m + 2 * (c + 1) * PG_KC < lmax;
        if (PAIRS && sn + 2 >= nval) {
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int r = 0; r < RPL; ++r)
#pragma unroll
                    for (int cc = 0; cc < 4; ++cc)
                        if (sn + cc >= nval) q[p][r][cc] = 0.f;
        }
        if constexpr (ANALYSIS) {
            // i = latitude k; panel 0 = X[k] + X[k'], panel 1 = X[k] - X[k']; the equator row is its own mirror
            if (!plain) {
#pragma unroll
                for (int r = 0; r < RPL; ++r) {
                    const int i = c * PG_KC + RPL * rg + r;
                    const bool ok = i < K2, mirror = (nlat - 1 - i) != i;
#pragma unroll
                    for (int cc = 0; cc < 4; ++cc) {
                        q[0][r][cc] = ok ? q[0][r][cc] : 0.f;
                        q[1][r][cc] = ok && mirror ? q[1][r][cc] : 0.f;
                    }
                }
            }
#pragma unroll
            for (int r = 0; r < RPL; ++r)
#pragma unroll
                for (int cc = 0; cc < 4; ++cc) {
                    const float a_ = q[0][r][cc], b_ = q[1][r][cc];
                    q[0][r][cc] = a_ + b_;
                    q[1][r][cc] = a_ - b_;
                }
            if (!plain) {
#pragma unroll
                for (int r = 0; r < RPL; ++r) {
                    const int i = c * PG_KC + RPL * rg + r;
#pragma unroll
                    for (int cc = 0; cc < 4; ++cc) q[1][r][cc] = (nlat - 1 - i) != i ? q[1][r][cc] : 0.f;
                }
            }
        } else if (!plain) {
            // i = index within a parity; panel 0 = degree m+2i, panel 1 = degree m+2i+1
#pragma unroll
            for (int r = 0; r < RPL; ++r) {
                const int i = c * PG_KC + RPL * rg + r;
#pragma unroll
                for (int cc = 0; cc < 4; ++cc) {
                    q[0][r][cc] = m + 2 * i < lmax ? q[0][r][cc] : 0.f;
                    q[1][r][cc] = m + 2 * i + 1 < lmax ? q[1][r][cc] : 0.f;
                }
            }
        }
        // the bounds live in the other buffer's array between chunks: they would cost eight registers across the matrix phase
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            i4 E = *reinterpret_cast<const i4*>(&expo[buf ^ 1][p][4 * slot]);
            int eb[4];
            exponents(q[p], eb);
            const int over = max(max(eb[0] - E[0], eb[1] - E[1]), max(eb[2] - E[2], eb[3] - E[3]));
            if (__builtin_amdgcn_ballot_w64(over > 0) != 0) raise(eb, E);
            cut_store(planes + ((buf * 2 + p) * 2) * PLANE, q[p], E);
            if (rg == 0) *reinterpret_cast<i4*>(&expo[buf][p][4 * slot]) = E;
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // ---- matrix phase --------------------------------------------------------------------------------------------------------
    const int kg = lane >> 5, cl = lane & 31;
    const int frag = (cl & 3) * CS + (cl >> 2) * 32 + ((kg ^ ((cl & 3) >> 1)) * 16);      // my fragment of tile 0 within a plane
    auto compute = [&](int buf, const f4 (&ar)[2]) {
        // follow the scales of my columns
        int enew[NT];
        bool moved = false;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            enew[t] = expo[buf][par][32 * t + cl];
            moved |= enew[t] != erun[t];
        }
        if (__builtin_amdgcn_ballot_w64(moved) != 0) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int d = erun[t] - enew[t];
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[t][v] = __builtin_ldexpf(acc[t][v], d);
                erun[t] = enew[t];
            }
        }
        const f16x8 a0 = __builtin_bit_cast(f16x8, ar[0]), a1 = __builtin_bit_cast(f16x8, ar[1]);
        const unsigned char* pb = planes + ((buf * 2 + par) * 2) * PLANE + frag;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const f16x8 b0 = *reinterpret_cast<const f16x8*>(pb + t * 256), b1 = *reinterpret_cast<const f16x8*>(pb + PLANE + t * 256);
            // smallest terms first
            acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1, b0, acc[t], 0, 0, 0);
            acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a0, b1, acc[t], 0, 0, 0);
            acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a0, b0, acc[t], 0, 0, 0);
        }
    };
    auto a_load = [&](int c, f4 (&ar)[2]) {
        // (chunks past the end repeat the last one: the stream of the next row block, or the end of the buffer, follows)
#pragma unroll
        for (int p = 0; p < 2; ++p) ar[p] = apv[(int64_t)min(max(c - c0w, 0), max(nc - 1 - c0w, 0)) * APB + 64 * p];
    };

    // Software pipeline, one chunk deep: the panel rows of the next chunk are requested before the matrix instructions of the current
    // one and its table fragments after them (into the same registers); the rows are cut once those instructions are issued.
    // The analysis walks the latitudes from the equator to the pole: Fourier coefficients of order m fall off towards the
    // poles like sin^m(theta), so the first chunk sets the column scales and later ones rarely move them; the synthesis
    // walks the degrees upwards, the direction in which spectra decay.
    constexpr int cstep = ANALYSIS ? -1 : 1;
    const int cfirst = ANALYSIS ? nc - 1 : cstart;
    f4 acur[2];
    if (cstart < nc) {
        if (stager && rg == 0) {
            const i4 e0 = {LH_EMIN, LH_EMIN, LH_EMIN, LH_EMIN};
            *reinterpret_cast<i4*>(&expo[(cfirst & 1) ^ 1][0][4 * slot]) = e0;
            *reinterpret_cast<i4*>(&expo[(cfirst & 1) ^ 1][1][4 * slot]) = e0;
        }
        q_load(cfirst);
        a_load(cfirst, acur);
        q_store(cfirst & 1, cfirst);
    }
    __syncthreads();
    for (int c = cfirst, left = nc - cstart; left > 0; --left, c += cstep) {
        const int buf = c & 1;
        const bool more = left > 1;
        q_load(c + cstep);      // (past the end: the nearest row; unconditional, so that what is waited for can be counted)
        __builtin_amdgcn_sched_barrier(0);
        if (c >= c0w) compute(buf, acur);
        __builtin_amdgcn_sched_barrier(0);
        a_load(c + cstep, acur);
        __builtin_amdgcn_sched_barrier(0);
        if (more) q_store(buf ^ 1, c + cstep);
        __syncthreads();
    }

    // ---- epilogue: undo the scales (row factor stored with the table, column bound erun), store ------------------------------
    // D layout of the 32x32 MFMA: register v of lane j holds D[8*(v/4) + 4*(j/32) + v%4][j%32].
    f4 rinv[4];
    if (active) {
        const float* rp = a.rinv + (entry_pos(par, rb) - 2 * (int64_t)a.mmax) * PG_ROWS + 4 * kg;
#pragma unroll
        for (int q = 0; q < 4; ++q) rinv[q] = *reinterpret_cast<const f4*>(rp + 8 * q);
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[t][v] = __builtin_ldexpf(acc[t][v], erun[t] - LH_SH) * rinv[v >> 2][v & 3];
    }
    if (ANALYSIS && COEFFS) {
        float* out = a.Out + 2 * (int64_t)m;
        if (rb - (wslot & 1) == 0) {
            // the order's first workgroups write its zeros, those of the last order with degrees also the orders past it
            for (int i = tid; i < m * TN; i += 256) {
                const int n = n0 + i % TN;
                if (n < nval) out[scolumn(n) + (uint32_t)(i / TN) * srow] = 0.f;
            }
            if (m == min(lmax, a.mmax) - 1)
                for (int i = tid; i < (a.mmax - 1 - m) * lmax * TN; i += 256) {
                    const int n = n0 + i % TN, l = i / TN % lmax, mm = 1 + i / TN / lmax;
                    if (n < nval) out[scolumn(n) + (uint32_t)l * srow + 2 * mm] = 0.f;
                }
        }
        if (!active) return;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int n = n0 + 32 * t + cl;
            float* o = out + scolumn(n);
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int r = PG_ROWS * rb + 8 * (v >> 2) + 4 * kg + (v & 3);
                if (r < nrows && n < nval) o[(uint32_t)(m + par + 2 * r) * srow] = acc[t][v];
            }
        }
    } else if (ANALYSIS) {
        if (!active) return;
        const int ldo = a.ldo, split = a.split;
        const int second = n0 >= split ? split : 0;             // (a tile of columns may also have both, see the checks below)
        if (PG_ROWS * (rb + 1) <= nrows && n0 + TN - second <= ldo && (second || n0 + TN <= split)) {
            // no row or column of my tile needs a check: one address per row, the tiles at constant offsets from it
            float* o = (second ? a.Out2 : a.Out) + (int64_t)m * lmax * ldo + (int64_t)(m + par + 2 * (PG_ROWS * rb + 4 * kg)) * ldo + (n0 - second) + cl;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                float* orow = o + (int64_t)(2 * (8 * (v >> 2) + (v & 3))) * ldo;
#pragma unroll
                for (int t = 0; t < NT; ++t) orow[32 * t] = acc[t][v];
            }
            return;
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            int n = n0 + 32 * t + cl;
            float* out = (n >= split ? a.Out2 : a.Out) + (int64_t)m * lmax * ldo;
            n -= n >= split ? split : 0;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int r = PG_ROWS * rb + 8 * (v >> 2) + 4 * kg + (v & 3);
                if (r < nrows && n < ldo) out[(int64_t)(m + par + 2 * r) * ldo + n] = acc[t][v];
            }
        }
    } else {
        // X[k] = E[k] + O[k] and X[k'] = E[k] - O[k]: the two wavefronts of a row block leave their sums in LDS, TB column tiles at a
        // time, and each stores one of the two rows -- the even-parity wavefront the northern row k, the odd-parity one the mirrored
        // row k' -- so that all four wavefronts share the stores; read back by rows, four columns to a lane
        constexpr int TP = 32 * 36;                   // floats of a tile: rows 36 apart keep the 16-byte reads aligned and off each other's banks
        constexpr int TB = NT >= 2 && PLANES >= 2 * 4 * TP * 4 ? 2 : 1;
        static_assert(TB * 4 * TP * 4 <= PLANES, "the parity exchange reuses the plane buffers");
        float* exch = reinterpret_cast<float*>(planes);
        float* mine = exch + wslot * (TB * TP) + 4 * kg * 36 + cl;
        const int er = lane >> 3, ec = 4 * (lane & 7);
        const float* pe = exch + (wslot & 1) * (TB * TP) + er * 36 + ec;
        const float* po = pe + 2 * (TB * TP);
        float* out = a.Out + (int64_t)m * nlat * ld;
        const int k0 = PG_ROWS * rb;
#pragma unroll
        for (int t0 = 0; t0 < NT; t0 += TB) {
            if (t0 > 0) __syncthreads();               // the previous tiles have been read
            if (active) {
#pragma unroll
                for (int t = t0; t < t0 + TB && t < NT; ++t)
#pragma unroll
                    for (int v = 0; v < 16; ++v) mine[(t - t0) * TP + (8 * (v >> 2) + (v & 3)) * 36] = acc[t][v];
            }
            __syncthreads();
            if (active) {
#pragma unroll
                for (int t = t0; t < t0 + TB && t < NT; ++t) {
                    const int n = n0 + 32 * t + ec;
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const int k = k0 + 8 * u + er;
                        const f4 e = *reinterpret_cast<const f4*>(pe + (t - t0) * TP + 8 * u * 36), o = *reinterpret_cast<const f4*>(po + (t - t0) * TP + 8 * u * 36);
                        const int row = par ? nlat - 1 - k : k;
                        // even parity: E + O to row k; odd parity: E - O to row k' (the equator row is its own mirror and has O = 0)
                        if (k < K2 && n < ld && !(par && row == k)) *reinterpret_cast<f4*>(out + (int64_t)row * ld + n) = par ? e - o : e + o;
                    }
                }
            }
        }
    }
}

// Column tiles per workgroup (1 to 5).  Wide workgroups read the table once for more columns and spread the cut of the panels, narrow
// ones are more in number (small grids leave CUs idle) and pad less.  Estimated time in us: a launch, and the longer of one workgroup
// alone (longest chunk loop and epilogue) and a CU's share of all of them, the coefficients fitted to 4000 measured shapes per
// direction (8 to 720 latitudes, 2 to 720 degrees, 1 to 3072 rows, all five tile counts): the choice is 0.6 % (analysis) and 0.8 % (synthesis) from the
// best tile count on average, 11 % at worst above 30 us.  By the least padding alone it was 10 % and 85 %: 74 rows of 160 x 320 went
// 14.4 -> 11.4 us and 17.2 -> 12.7, 384 rows of 721 latitudes and 240 degrees keep four tiles.
int legendre_f16_tiles(bool analysis, int64_t ncols, int64_t items, int64_t chunks, int longest, int cus) {
    static const double alone[2][4] = {{0.626, 0.139, 0.0, 0.328}, {0.619, 0.161, 0.0, 0.294}};      // per chunk: + per tile; epilogue: + per tile
    static const double per_chunk[2][5] = {{0.259, 0.291, 0.297, 0.278, 0.377}, {0.247, 0.348, 0.435, 0.480, 0.673}};
    static const double per_item[2][5] = {{0.673, 1.338, 2.152, 2.769, 3.901}, {0.488, 0.871, 1.352, 1.920, 3.060}};
    int best = 1;
    double best_t = 0.0;
    for (int nt = 1; nt <= 5; ++nt) {
        const double groups = (double)((ncols + 32 * nt - 1) / (32 * nt));
        const double one = longest * (alone[analysis][0] + alone[analysis][1] * nt) + alone[analysis][2] + alone[analysis][3] * nt;
        const double all = groups * ((double)chunks * per_chunk[analysis][nt - 1] + (double)items * per_item[analysis][nt - 1]) / cus;
        const double one2 = one * one, all2 = all * all, t = one2 * one2 + all2 * all2;      // (the time's fourth power: 0.3 us of a launch less than with std::pow)
        if (nt == 1 || t < best_t) { best_t = t; best = nt; }
    }
    return best;
}

template <bool ANALYSIS, bool COEFFS>
static int launch_f16(const PgemmArgs& a, int n_work, hipStream_t s) {
    const int64_t ncols = a.ld;
    if (n_work <= 0 || ncols <= 0) return SFNO_OK;
    if (!a.rinv || !a.wrec) return SFNO_EINVAL;
    // the kernel addresses a panel (one order: nlat or lmax rows of ld floats) with 32-bit byte offsets
    if ((int64_t)(a.nlat > a.lmax ? a.nlat : a.lmax) * a.ld >= ((int64_t)1 << 30)) return SFNO_EUNSUPPORTED;
    const int best = legendre_f16_tiles(ANALYSIS, ncols, a.items, a.chunks, a.longest, device_cus());
#define LH_CASE(NT_)                                                                             \
    case NT_: {                                                                                  \
        const int64_t nwg = (int64_t)n_work * ((ncols + 32 * NT_ - 1) / (32 * NT_));             \
        if (nwg > 0x7fffffffLL) return SFNO_EUNSUPPORTED;                                        \
        dim3 grid((unsigned)nwg);                                                                \
        hipLaunchKernelGGL((legendre_f16_kernel<NT_, ANALYSIS, COEFFS>), grid, dim3(256), 0, s, a); \
        break;                                                                                   \
    }
    switch (best) {
        LH_CASE(1) LH_CASE(2) LH_CASE(3) LH_CASE(4) LH_CASE(5)
        default: return SFNO_EINVAL;
    }
#undef LH_CASE
    return hipGetLastError() == hipSuccess ? SFNO_OK : SFNO_EHIP;
}

int legendre_f16_launch(bool analysis, const PgemmArgs& a, int n_work, hipStream_t s) {
    return analysis ? launch_f16<true, false>(a, n_work, s) : launch_f16<false, false>(a, n_work, s);
}

// A launch less against eight-byte accesses.  Coefficients of 0.06 MiB (32 x 64, 8 rows): analysis 9.6 -> 7.5 us, synthesis 10.6 -> 7.5; 0.64 MiB
// (20 degrees, 200 rows) 13.9 -> 11.4 and 14.6 -> 11.2; 1.3 MiB (64 x 128, 40 rows) 13.8 -> 15.1 and 16.2 -> 14.2; 1.6 MiB (91 x 180, 26 rows) 15.0 -> 14.0
// and 16.1 -> 13.3; 3.9 MiB (160 x 320, 20 rows) 21.6 -> 23.7 and 24.3 -> 22.5; 14.5 MiB 32 -> 51 and 37 -> 43.  (One workgroup writes the zeros of the orders
// past the last degree: there may be one such order, not many.)
bool legendre_coeffs_fit(bool analysis, int format, int64_t rows, int lmax, int mmax) {
    return format == PG_FORMAT_F16X2 && mmax <= lmax + 1 && 8 * rows * lmax * mmax <= (analysis ? 1 << 20 : 2 << 20);
}

int legendre_coeffs_launch(bool analysis, PgemmArgs a, int64_t rows, int n_work, hipStream_t s) {
    a.ncol = (int)(2 * rows);
    return analysis ? launch_f16<true, true>(a, n_work, s) : launch_f16<false, true>(a, n_work, s);
}

}  // namespace sfno
