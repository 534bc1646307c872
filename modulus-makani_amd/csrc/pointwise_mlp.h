// MLP of the SFNO block in one kernel (inference, bf16 NCHW activations; included by pointwise.hip):
//   y[b][o][p] = b2[o] + sum_h W2[o][h] gelu(b1[h] + sum_c W1[h][c] gelu(scale[b][c] x[b][c][p] + shift[b][c]))
// Same sums in the same order and same roundings as scale_shift_act_kernel and two pw_gemm kernels, which write and read the normalised
// field and the hidden one (the larger by the MLP ratio); here neither leaves the CU.
//
// A workgroup is four wavefronts, one per SIMD with all 512 registers, on a tile of 128 pixels; it stays resident and walks its tiles.  The
// activated input of the tile lies in LDS as operands of the first product (up to 96 KiB), the hidden channels pass through in chunks of 128
// (two buffers of 32 KiB).  Wavefronts split the rows of both products (32 hidden and up to 96 output channels each), so every weight
// is read once per tile and CU, from L2 into registers, and feeds four matrix instructions (32 bytes per clock, half of what L1
// gives); the shared operands come from LDS (128 bytes per clock under the first product: its bound).  The lane that holds a hidden channel's
// sums holds them as operand of the second product, because the rows of W1 are dealt out for that; they only pass through LDS
// to reach the other wavefronts.  Output and hidden sums take all 256 accumulation registers.
//
// With one wavefront per SIMD a vector instruction issues every 5.4 clocks and eight of them fit behind a matrix instruction (46 clocks
// where they take 34 and 43 by themselves), so the GELU of chunk c - 1 is cut into slices between the matrix instructions of the second product
// of chunk c - 2 and the first of chunk c.  384 -> 768 -> 384 at 720 x 1440, one sample: 1.43 ms (855 TFLOP/s) where the three kernels take
// 1.96; 240 x 480 180 us against 218, four samples 655 against 883.  87 k clocks per tile, of which 40 k of matrix pipe and 49 k of vector issue;
// 17 k of the latter (norm and GELU of the next tile's input, with the stores between) find no matrix instruction to hide behind.
// The clock falls from 2.05 to 1.8 GHz as the two overlap better: 110 k clocks took only 13 % longer.
#pragma once

// Memory behind a wavefront-uniform base: a lane's 32-bit offset and a scalar one, both in bytes (no address arithmetic per load)
struct Buf {
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ Buf(const void* p, unsigned bytes) : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00027000)) {}
    __device__ __forceinline__ u32x4 load16(unsigned lane, unsigned uniform) const {
        return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, lane, uniform, 0));
    }
    __device__ __forceinline__ u32x2 load8(unsigned lane, unsigned uniform) const {
        return __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, lane, uniform, 0));
    }
    __device__ __forceinline__ void store8(u32x2 v, unsigned lane, unsigned uniform) const { __builtin_amdgcn_raw_buffer_store_b64(v, r, lane, uniform, 0); }
};

// f(0), f(1), ... f(N - 1) with constants for arguments: register arrays are indexed by them
template <class F, int... I>
__device__ __forceinline__ void unrolled_(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void unrolled(F&& f) {
    unrolled_(f, std::make_integer_sequence<int, N>{});
}

// A value out of the accumulation registers, here and not where the sum is complete: read ahead, a tile's sums would take the ordinary
// registers of everything else.  The last matrix instruction that wrote it must be behind acc_settle().
__device__ __forceinline__ float from_acc(float x) {
    float y;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(y) : "a"(x));
    return y;
}
// more wait states than any matrix instruction here needs between its result and a vector instruction that reads it
__device__ __forceinline__ void acc_settle() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 15\n\ts_nop 15");
    __builtin_amdgcn_sched_barrier(0);
}

// gelu() of eight values in twelve slices of about eight instructions, which fit between matrix instructions; w: the results in bf16
struct Gelu8 {
    static constexpr int SLICES = 12;
    float x[8], t[8], q[8];
    u32x4 w;
    __device__ __forceinline__ void slice(int s) {
        float inf = __builtin_inff();                // (opaque: max(x, 0) would canonicalise x first)
        asm("" : "+s"(inf));
        constexpr float C[6] = {-5.615057212e-04f, 6.880626770e-03f, -5.027262948e-02f, -4.624537704e-01f, -1.149621597e+00f, -1.000106287211f};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (s == 0) t[i] = __builtin_amdgcn_fmed3f(fabsf(x[i]), 0.f, 6.5f);
            if (s == 1) q[i] = fmaf(t[i], 2.008575651e-05f, C[0]);
            if (s >= 2 && s <= 6) q[i] = fmaf(t[i], q[i], C[s - 1]);
            if ((s == 7 && i < 4) || (s == 8 && i >= 4)) q[i] = __builtin_amdgcn_exp2f(q[i]);
            if (s == 9) t[i] = __builtin_amdgcn_fmed3f(x[i], 0.f, inf);
            if (s == 10) t[i] = fmaf(-fabsf(x[i]), q[i], t[i]);
        }
        if (s == 11) {
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = bf16_pair(t[2 * i], t[2 * i + 1]);
        }
    }
    __device__ __forceinline__ void all() {
#pragma unroll
        for (int s = 0; s < SLICES; ++s) slice(s);
    }
};

template <int MT>
struct MlpGeo {
    static constexpr int PX = 128;                   // pixels per tile
    static constexpr int CHUNK = 128;                // hidden channels per pass
    static constexpr int CSTEPS = CHUNK / 16;        // steps of 16 rows in a chunk
    static constexpr int ROWS = 128 * MT;            // input and output channels at most
    static constexpr int XBYTES = ROWS * PX * 2;
    static constexpr int HBYTES = CHUNK * PX * 2;    // one of two buffers of hidden channels
    static constexpr int LDS = XBYTES + 2 * HBYTES;
    static constexpr int KSTEPS = 8 * MT;            // steps over the input channels
    static constexpr int RING1 = 8, RING2 = 4;       // how many steps ahead the weights of the two products are asked for
    static constexpr int UNITS = 2 * MT;             // groups of 64 input channels
    static_assert(LDS <= 160 * 1024, "one workgroup fits the CU");
};

template <int MT, bool RAGGED>
__global__ __launch_bounds__(256, 1) void pw_mlp_kernel(MlpArgs a) {
    using G = MlpGeo<MT>;
    using T = std::true_type;
    using F = std::false_type;
    constexpr int R1 = G::RING1, R2 = G::RING2, CS = G::CSTEPS, KS = G::KSTEPS;
    constexpr int KB = G::PX * 16;                   // bytes of a group of eight rows in LDS
    __shared__ __align__(16) unsigned char lds[G::LDS];
    unsigned char* const xl = lds;
    unsigned char* const hl = lds + G::XBYTES;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane & 31, ko = lane >> 5;
    const int E = a.E;
    const unsigned P2 = 2 * (unsigned)a.P;           // bytes of a row
    const int nchunks = max(2, (a.H + G::CHUNK - 1) / G::CHUNK);
    const int nk1p = a.kpad1 / 16, nk2p = a.kpad2 / 16;
    const int rb1max = a.opad1 / 32 - 1, rb2max = a.opad2 / 32 - 1;   // last row blocks of the packed weights
    // rows of a hidden tile are dealt out so that a lane's sums of rows 8 g + 4 ko + j are the operand of the second product
    // for its own column: matrix row 16 s + 8 a + 4 b + j stands for hidden channel 16 s + 8 b + 4 a + j
    const int prow = (q & 19) | ((q & 4) << 1) | ((q & 8) >> 1);
    const unsigned off1 = (unsigned)(prow + 32 * ko) * 16, off2 = (unsigned)lane * 16;
    const unsigned char* const bx = xl + ko * KB + q * 16;
    const unsigned char* const bh = hl + ko * KB + q * 16;
    unsigned char* const hput = hl + (4 * wave + ko) * KB + q * 16;

    const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    f32x16 out[MT][4], acc[4], bias1;
    float hv[4][16];                                 // a chunk's sums on their way through the GELU
    u32x4 r1[R1], r2[R2][MT], bf[2][4];

    auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
    // fragments are 1 KiB each, those of a row block one after the other
    const Buf w1(a.W1, (unsigned)a.opad1 / 32 * nk1p * 1024), w2(a.W2, (unsigned)a.opad2 / 32 * nk2p * 1024);
    const Buf b1(a.b1, a.b1 ? a.H * 4 : 0), b2(a.b2, a.b2 ? E * 4 : 0);      // (no bias: nothing in range, the loads return zeros)
    // (`here` makes a scalar opaque: hoisted out of the loops, the offsets of all loads would not fit the scalar registers)
    auto here = [](unsigned s) __attribute__((always_inline)) {
        asm volatile("" : "+s"(s));
        return s;
    };
    auto load1 = [&](int c, int k) {                 // step k of chunk c
        const unsigned s = here(min(4 * c + wave, rb1max) * nk1p + (RAGGED ? min(k, nk1p - 1) : 0)) * 1024 + (RAGGED ? 0 : (k & ~3) * 1024);
        r1[k % R1] = w1.load16(off1 + (RAGGED ? 0 : (k & 3) * 1024), s);
    };
    auto load2 = [&](int c, int k) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const unsigned s = here(min(MT * wave + i, rb2max) * nk2p) + (RAGGED ? min(c * CS + k, nk2p - 1) : here(c * CS) + (k & ~3));
            r2[k % R2][i] = w2.load16(off2 + (RAGGED ? 0 : (k & 3) * 1024), s * 1024);
        }
    };
    // (past the packed matrix the loads repeat its last step: zeros in their place)
    auto frag = [&](const u32x4& r, bool valid) {
        if (!RAGGED) return __builtin_bit_cast(bf16x8, r);
        const unsigned m = valid ? ~0u : 0u;
        const u32x4 v = {r[0] & m, r[1] & m, r[2] & m, r[3] & m};
        return __builtin_bit_cast(bf16x8, v);
    };
    auto rows_to = [&](const unsigned char* base, int k, u32x4 (&dst)[4]) {
#pragma unroll
        for (int t = 0; t < 4; ++t) dst[t] = *reinterpret_cast<const u32x4*>(base + k * 2 * KB + t * 512);
    };
    // bias of a chunk's hidden rows in the order of a lane's sums
    auto ask_bias = [&](int c) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            // (groups of 16 rows are inside or outside as a whole)
            const u32x4 v = b1.load16(32 * ko, 4 * (min(G::CHUNK * c + 32 * wave + 16 * (g >> 1), a.H - 16) + 4 * (g & 1)));
#pragma unroll
            for (int j = 0; j < 4; ++j) bias1[4 * g + j] = __uint_as_float(v[j]);
        }
    };

    const int ntiles = (int)(a.n_strips * a.B);
    auto tile_at = [&](int t, int& b, int64_t& px) {
        b = __builtin_amdgcn_readfirstlane((int)((unsigned)t / (unsigned)a.n_strips));     // (the division leaves it in a vector register)
        px = (int64_t)(t - b * (int)a.n_strips) * G::PX + 4 * q;
    };
    int b;
    int64_t px;
    // Staging of a tile: unit u is 64 channels, of which a half wavefront takes 8 x 128 pixels: raw rows, then affine, GELU and into LDS
    u32x2 raw[G::UNITS][8];
    Gelu8 g;
    float sc[8], sh[8];
    auto channel = [&](int u) { return min(8 * (8 * u + 2 * wave + ko), E - 8); };
    auto ask_raw = [&](int b, int64_t px, int n, unsigned bytes) {    // n = 8 unit + row; bytes: of a sample, 0 asks for nothing
        const int u = n >> 3, i = n & 7;
        const Buf x(a.X + (int64_t)b * E * a.P, bytes);
        // (channels past the last one repeat others and meet zero weights; whole units of them where E is a multiple of 64)
        const unsigned s = (RAGGED ? i : here(min(64 * u, E - 64)) + i) * here(P2);
        raw[u][i] = x.load8((unsigned)(RAGGED ? channel(u) : 16 * wave + 8 * ko) * P2 + 2 * (unsigned)min(px, a.P - 4), s);
    };
    // (through the scalar unit: vector loads would queue up behind the rows)
    auto ask_affine = [&](int b, int u) {
        const int64_t c0 = (int64_t)b * E + min(8 * (8 * u + 2 * wave), E - 8), c1 = (int64_t)b * E + min(8 * (8 * u + 2 * wave + 1), E - 8);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float s0 = uniform_load(a.scale, c0 + i), s1 = uniform_load(a.scale, c1 + i), t0 = uniform_load(a.shift, c0 + i), t1 = uniform_load(a.shift, c1 + i);
            sc[i] = ko ? s1 : s0;
            sh[i] = ko ? t1 : t0;
        }
    };
    // n = 4 unit + t: eight channels of pixel t of the lane's four
    auto stage_unit = [&](int b, auto n_) __attribute__((always_inline)) {
        constexpr int u = decltype(n_)::value / 4, t = decltype(n_)::value % 4;
        if constexpr (t == 0) ask_affine(b, u);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const unsigned w = raw[u][i][t >> 1];
            g.x[i] = fmaf(sc[i], __uint_as_float(t & 1 ? w & 0xffff0000u : w << 16), sh[i]);
        }
    };
    auto put_x = [&](int n, const Gelu8& g) {
        const int u = n / 4, t = n % 4;
        const int kg = 8 * u + 2 * wave + ko;
        const unsigned m = 8 * kg < E ? ~0u : 0u;
        const u32x4 o = {g.w[0] & m, g.w[1] & m, g.w[2] & m, g.w[3] & m};
        *reinterpret_cast<u32x4*>(xl + kg * KB + t * 512 + q * 16) = o;
    };
    // a lane's u-th eight values of the hidden tile: column tile u / 2, half u % 2
    auto put_hidden = [&](int c, int u, const Gelu8& g) { *reinterpret_cast<u32x4*>(hput + (c & 1) * G::HBYTES + 2 * (u & 1) * KB + (u >> 1) * 512) = g.w; };
    // Work dealt out between matrix instructions: units of twelve slices, `take` before a unit's first and `put` behind its last.
    // after(m) runs behind the m-th of n matrix instructions.
    auto dealt = [&](auto m_, auto n_, auto units_, auto&& take, auto&& put) __attribute__((always_inline)) {
        constexpr int M = decltype(m_)::value, N = decltype(n_)::value, UNITS = decltype(units_)::value, S = Gelu8::SLICES;
        constexpr int FROM = M * UNITS * S / N, TO = (M + 1) * UNITS * S / N;
        fence();
        unrolled<TO - FROM>([&](auto j) __attribute__((always_inline)) {
            constexpr int s = FROM + decltype(j)::value;
            if constexpr (s % S == 0) take(std::integral_constant<int, s / S>{});
            g.slice(s % S);
            if constexpr (s % S == S - 1) put(std::integral_constant<int, s / S>{});
        });
        fence();
    };
    auto hidden_unit = [&](auto u_) __attribute__((always_inline)) {
        constexpr int u = decltype(u_)::value;
#pragma unroll
        for (int i = 0; i < 8; ++i) g.x[i] = hv[u >> 1][8 * (u & 1) + i];
    };
    auto sums_unit = [&](auto u_) __attribute__((always_inline)) {      // the same straight from the sums
        constexpr int u = decltype(u_)::value;
#pragma unroll
        for (int i = 0; i < 8; ++i) g.x[i] = from_acc(acc[u >> 1][8 * (u & 1) + i]) + bias1[8 * (u & 1) + i];
    };
    // first product of chunk c; `after`: work behind each matrix instruction, `more`: loads to ask for behind a step
    auto product1 = [&](int c, auto&& after, auto&& more) __attribute__((always_inline)) {
        rows_to(bx, 0, bf[0]);
        unrolled<KS>([&](auto k_) __attribute__((always_inline)) {
            constexpr int k = decltype(k_)::value;
            if constexpr (k + 1 < KS) rows_to(bx, k + 1, bf[(k + 1) & 1]);
            fence();
            const bf16x8 av = frag(r1[k % R1], k < nk1p);
            unrolled<4>([&](auto t_) __attribute__((always_inline)) {
                constexpr int t = decltype(t_)::value;
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, __builtin_bit_cast(bf16x8, bf[k & 1][t]), k == 0 ? zero : acc[t], 0, 0, 0);
                after(std::integral_constant<int, 4 * k + t>{});
            });
            if constexpr (k + R1 < KS) load1(c, k + R1);
            more(k_);
            fence();
        });
#pragma unroll
        for (int t = 0; t < 4; ++t) asm volatile("" : "+a"(acc[t]));        // (the sums stay in this block)
    };
    // second product of chunk c
    auto product2 = [&](int c, bool ragged, auto&& after, auto&& more) __attribute__((always_inline)) {
        const unsigned char* const bc = bh + (c & 1) * G::HBYTES;
        rows_to(bc, 0, bf[0]);
        unrolled<CS>([&](auto k_) __attribute__((always_inline)) {
            constexpr int k = decltype(k_)::value;
            if constexpr (k + 1 < CS) rows_to(bc, k + 1, bf[(k + 1) & 1]);
            fence();
            unrolled<4 * MT>([&](auto m_) __attribute__((always_inline)) {
                constexpr int m = decltype(m_)::value, i = m / 4, t = m % 4;
                out[i][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag(r2[k % R2][i], !ragged || c * CS + k < nk2p), __builtin_bit_cast(bf16x8, bf[k & 1][t]), out[i][t], 0, 0, 0);
                after(std::integral_constant<int, 4 * MT * k + m>{});
            });
            if constexpr (k + R2 < CS) load2(c, k + R2);
            more(k_);
            fence();
        });
#pragma unroll
        for (int i = 0; i < 4 * MT; ++i) asm volatile("" : "+a"(out[i / 4][i % 4]));
    };
    auto take_sums = [&]() {
        acc_settle();
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) hv[t][v] = from_acc(acc[t][v]) + bias1[v];
        fence();
    };
    const auto nothing = [](auto) {};
    constexpr std::integral_constant<int, 4 * KS> N1{};          // matrix instructions of the products
    constexpr std::integral_constant<int, 4 * MT * CS> N2{};
    constexpr std::integral_constant<int, CS> ALL{};             // units of a chunk's GELU
    // of which under the next chunk's first product; the others under the second product of the chunk before
    constexpr std::integral_constant<int, CS / 2> UA{};
    constexpr std::integral_constant<int, CS - UA> UB{};

    if ((int)blockIdx.x >= ntiles) return;
    tile_at(blockIdx.x, b, px);
#pragma unroll
    for (int n = 0; n < 8 * G::UNITS; ++n) ask_raw(b, px, n, (unsigned)E * P2);
    unrolled<4 * G::UNITS>([&](auto n) {
        stage_unit(b, n);
        g.all();
        put_x(n, g);
        fence();
    });
    ask_bias(0);
#pragma unroll
    for (int k = 0; k < R1; ++k) load1(0, k);
    __syncthreads();
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int next = tile + gridDim.x;
        int nb = b;
        int64_t npx = px;
        if (next < ntiles) tile_at(next, nb, npx);
        const unsigned nbytes = next < ntiles ? (unsigned)E * P2 : 0;
        // chunks 0 and 1: the first product of chunk 1 takes the whole GELU of chunk 0
        product1(0, nothing, [&](auto k) { if (k >= KS - R1) load1(1, k - (KS - R1)); });
        take_sums();
        ask_bias(1);
        product1(1, [&](auto m) { dealt(m, N1, ALL, hidden_unit, [&](auto u) { put_hidden(0, u, g); }); },
                 [&](auto k) { if (k >= KS - R2) load2(0, k - (KS - R2)); });
#pragma unroll
        for (int i = 0; i < 4 * MT; ++i) out[i / 4][i % 4] = zero;
        __syncthreads();
        for (int c = 2; c < nchunks; ++c) {
            // second product of chunk c - 2, first of chunk c, GELU of chunk c - 1
            take_sums();
            ask_bias(c);
            product2(c - 2, false,
                     [&](auto m) {
                         dealt(m, N2, UB, [&](auto u) { hidden_unit(std::integral_constant<int, UA + decltype(u)::value>{}); },
                               [&](auto u) { put_hidden(c - 1, UA + u, g); });
                     },
                     [&](auto k) {
                         unrolled<(decltype(k)::value + 1) * R1 / CS - decltype(k)::value * R1 / CS>([&](auto j) { load1(c, k * R1 / CS + j); });
                     });
            product1(c, [&](auto m) { dealt(m, N1, UA, hidden_unit, [&](auto u) { put_hidden(c - 1, u, g); }); },
                     [&](auto k) { if (k >= KS - R2) load2(c - 1, k - (KS - R2)); });
            __syncthreads();
        }
        // The next tile's rows are asked for a few at a time: a CU takes in no more than about 10 bytes per clock from beyond L2, and
        // whatever waits for weights asked for later waits for these rows too (the memory counter retires in order).
        acc_settle();
        product2(nchunks - 2, true, [&](auto m) { dealt(m, N2, ALL, sums_unit, [&](auto u) { put_hidden(nchunks - 1, u, g); }); },
                 [&](auto k) {
                     if (k >= CS - R2) load2(nchunks - 1, k - (CS - R2));
                     unrolled<MT>([&](auto n) { ask_raw(nb, npx, MT * k + n, nbytes); });
                 });
        __syncthreads();
        // (whole units of 64 channels under the second product: those whose rows were asked for before it)
        constexpr std::integral_constant<int, 4 * (G::UNITS / 3)> EARLY{};
        product2(nchunks - 1, true, [&](auto m) { dealt(m, N2, EARLY, [&](auto n) { stage_unit(nb, n); }, [&](auto n) { put_x(n, g); }); },
                 [&](auto k) { unrolled<MT>([&](auto n) { ask_raw(nb, npx, MT * (CS + k) + n, nbytes); }); });
        ask_bias(0);
#pragma unroll
        for (int k = 0; k < R1; ++k) load1(0, k);
        // (all of the bias ahead of the stores, which a later load would wait for)
        u32x4 bias2[MT][4];
#pragma unroll
        for (int i = 0; i < 4 * MT; ++i) bias2[i / 4][i % 4] = b2.load16(16 * ko, 4 * min(32 * MT * wave + 8 * i, E - 8));
        // Results out, the rest of the next tile in.  Lane: rows 8 (v / 4) + 4 ko + v % 4 of each 32-row tile, pixels 4 q .. 4 q + 3.
        acc_settle();
        const Buf y(a.Y + (int64_t)b * E * a.P, (unsigned)E * P2);
        const unsigned yoff = px < a.P ? 4 * ko * P2 + 2 * (unsigned)px : 0xffffffffu;       // (past the buffer: not stored)
        auto store = [&](auto r_) __attribute__((always_inline)) {
            constexpr int i = decltype(r_)::value / 16, v = decltype(r_)::value % 16;
            const int row = 32 * (MT * wave + i) + 8 * (v / 4);
            const float bs = __uint_as_float(bias2[i][v / 4][v % 4]);
            const u32x2 w = {bf16_pair(from_acc(out[i][0][v]) + bs, from_acc(out[i][1][v]) + bs), bf16_pair(from_acc(out[i][2][v]) + bs, from_acc(out[i][3][v]) + bs)};
            if (row < E) y.store8(w, yoff, (here(row) + v % 4) * here(P2));
        };
        constexpr int LATE = 4 * G::UNITS - EARLY, ROWS = 16 * MT;
        if (next < ntiles) {
            unrolled<LATE>([&](auto n_) __attribute__((always_inline)) {
                constexpr int n = decltype(n_)::value, from = n * ROWS / LATE, to = (n + 1) * ROWS / LATE;
                stage_unit(nb, std::integral_constant<int, EARLY + n>{});
                g.all();
                put_x(EARLY + n, g);
                unrolled<to - from>([&](auto r) { store(std::integral_constant<int, from + decltype(r)::value>{}); });
                fence();
            });
        } else {
            unrolled<ROWS>(store);
        }
        b = nb;
        px = npx;
        __syncthreads();
    }
}
