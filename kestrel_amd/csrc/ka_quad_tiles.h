// Matrix products of some hundred rows by four waves, one on every SIMD, each with a quarter of the tile: the loop over K, the ends of a tile, and the kernel of
// one linear or of two that read the same rows.
//
// A wave of a quarter reads the least from LDS per product, and nothing has to be timed against a second wave: products are issued one after the other, and among
// them, at fixed places, the reads of the slice of channels behind this one and the loads of a K-step NS further on. One barrier a K-step.
//
// Cycles a K-step of 64 (the products alone in brackets), us on 256 CUs; the phased tiles in turn: 128 x 128 840 to 900 (512), 0.43 us, phased 1,310 to 1,380; 128 x 256
// 1,350 to 1,480 (1,024), 0.82, phased 1,790 to 1,860; 160 x 256 1,570 to 1,740 (1,280), 0.98. The clock gives way as products get denser, with any loop: 2.4 GHz with few
// workgroups, 1.6 to 1.9 with one of these on every CU. 192 x 256 and 256 x 256 leave LDS for two stages, wait for their loads (2,500 and 3,100 cycles) and stay with
// the phased tiles (ka_phased_tiles.h).
#pragma once

#include "ka_dma_tiles.h"

// TW, TX: MFMA tiles of 16 that a wave has of W and X; two by two waves. NS: K-steps in LDS.
template <int TW, int TX, int NS>
struct KqTile {
    static constexpr int BN = 32 * TW, BM = 32 * TX, WAVE_N = 16 * TW, WAVE_M = 16 * TX;
    static constexpr int STAGE = (BN + BM) * 128, SMEM = NS * STAGE;        // a K-step: the rows of W, then of X
    static constexpr int WL = BN / 32, XL = BM / 32, LOADS = WL + XL;       // loads of 1 KB per wave and K-step
    static_assert(SMEM <= 160 * 1024 && NS >= 3, "the stages fit, and a load has two K-steps to land");
    // What this lane asks for in load i of the wave's loads of W (X): the row of the tile; the first channel of the K-step follows from the row.
    static __device__ __forceinline__ int w_row(int i, int wave, int lane) { return kd_load_row<8>(wave * WL + i, lane); }
    static __device__ __forceinline__ int x_row(int i, int wave, int lane) { return kd_load_row<8>(wave * XL + i, lane); }
};

// acc[a][b] += the products of this wave's MFMA tiles (a of W, its rows the product's rows, b of X) over `steps` >= 1 K-steps. wsrc(i, t), xsrc(i, t): this lane's
// address of its load i at K-step t. The whole workgroup takes part; LDS is free again behind a barrier.
template <int TW, int TX, int NS, typename Weight, typename Row>
__device__ __forceinline__ void kq_product(unsigned char* lds, int wave, int lane, int steps, Weight wsrc, Row xsrc, floatx4 (&acc)[TW][TX]) {
    using T = KqTile<TW, TX, NS>;
    constexpr int PRODUCTS = TW * TX, READS = TW + TX, LOADS = T::LOADS, LATE = LOADS / 2;
    const int wn = wave / 2, wm = wave % 2, col = lane % 16, quarter = lane / 16;
    auto fetch = [&](int i, int stage, int t) {
        unsigned char* const base = lds + stage * T::STAGE;
        if (i < T::WL) __builtin_amdgcn_global_load_lds((const GD_GLOBAL void*)wsrc(i, t), (GD_LDS void*)(base + (wave * T::WL + i) * 1024), 16, 0, 0);
        else __builtin_amdgcn_global_load_lds((const GD_GLOBAL void*)xsrc(i - T::WL, t), (GD_LDS void*)(base + T::BN * 128 + (wave * T::XL + i - T::WL) * 1024), 16, 0, 0);
    };
    const int swz = kd_swizzle<8>(col), place[2] = {(quarter ^ swz) * 16, ((quarter + 4) ^ swz) * 16};
    const int wrow = (wn * T::WAVE_N + col) * 128, xrow = T::BN * 128 + (wm * T::WAVE_M + col) * 128;
    bf16x8 w[2][TW], x[2][TX];                                  // the operands of either half of a K-step
    auto read = [&](auto half_c, auto j_c, int stage) {
        constexpr int half = decltype(half_c)::value, j = decltype(j_c)::value;
        const unsigned char* const base = lds + stage * T::STAGE + place[half];
        if constexpr (j < TX) x[half][j] = *reinterpret_cast<const bf16x8*>(base + xrow + j * 2048);
        else w[half][j - TX] = *reinterpret_cast<const bf16x8*>(base + wrow + (j - TX) * 2048);
    };
    // The products of a half, and among them the reads of the other one (of stage `from`; in the first three quarters) and loads [first, first + count) of K-step t into
    // stage `into`. Everything stays where it is written.
    auto half_step = [&](auto half_c, auto first_c, auto count_c, auto reads_c, int from, int into, int t) {
        constexpr int half = decltype(half_c)::value, first = decltype(first_c)::value, count = decltype(count_c)::value, span = (PRODUCTS * 3 + 3) / 4;
        gd_static_for<0, PRODUCTS>([&](auto i_c) {
            constexpr int i = decltype(i_c)::value, a = i / TX, b = i % TX;
            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[half][a], x[half][b], acc[a][b], 0, 0, 0);
            if constexpr (decltype(reads_c)::value && i < span)
                gd_static_for<i * READS / span, (i + 1) * READS / span>([&](auto j_c) { read(std::integral_constant<int, 1 - half>{}, j_c, from); });
            gd_static_for<first + i * count / PRODUCTS, first + (i + 1) * count / PRODUCTS>([&](auto l_c) { fetch(decltype(l_c)::value, into, t); });
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    using C0 = std::integral_constant<int, 0>;
    using C1 = std::integral_constant<int, 1>;
    using Early = std::integral_constant<int, LOADS - LATE>;    // a K-step's loads beside the second half, and its last ones beside the first half behind that
    using Late = std::integral_constant<int, LATE>;
    using Yes = std::integral_constant<bool, true>;
    using No = std::integral_constant<bool, false>;
#pragma unroll
    for (int s = 0; s < NS; ++s)
        if (s < steps)
#pragma unroll
            for (int i = 0; i < LOADS; ++i) fetch(i, s, s);
    gd_wait_younger<LOADS, NS - 1>(min(NS - 1, steps - 1));
    gd_barrier();
    gd_static_for<0, READS>([&](auto j_c) { read(C0{}, j_c, 0); });
    int stage = 0, t = 0;
    auto behind = [&](int s) { return s + 1 == NS ? 0 : s + 1; };
    half_step(C0{}, C0{}, C0{}, Yes{}, 0, 0, 0);
    // Between the halves of a K-step: this wave's reads of its stage are in registers, and its loads of the next one have landed; behind the barrier everybody's, so
    // the next stage may be read and this one's memory written.
    for (; t + NS < steps;) {
        gd_wait_lds();
        gd_wait_loads<(NS - 2) * LOADS>();
        gd_barrier();
        const int before = stage;
        stage = behind(stage);
        half_step(C1{}, C0{}, Early{}, Yes{}, stage, before, t + NS);
        half_step(C0{}, Early{}, Late{}, Yes{}, stage, before, t + NS);
        ++t;
    }
#pragma unroll 1
    for (; t + 1 < steps; ++t) {
        gd_wait_lds();
        gd_wait_younger<LOADS, NS - 2>(min(NS - 2, steps - 2 - t));
        gd_barrier();
        stage = behind(stage);
        half_step(C1{}, C0{}, C0{}, Yes{}, stage, 0, 0);
        half_step(C0{}, C0{}, C0{}, Yes{}, stage, 0, 0);
    }
    gd_wait_lds();
    half_step(C1{}, C0{}, C0{}, No{}, 0, 0, 0);
}

// A wave's outputs as whole rows, a block of 16 rows at a time through the wave's share of LDS: take(a, b) gives four neighbouring columns of one row; store(row,
// column, from) then gets the wave's row and first column of 16 bytes of E at `from`. (Behind a barrier: the last K-step has been read by everybody.)
template <typename E, int TW, int TX, int NS, typename Take, typename Store>
__device__ __forceinline__ void kq_rows_out(unsigned char* lds, int wave, int lane, Take take, Store store) {
    using T = KqTile<TW, TX, NS>;
    constexpr int RB = T::WAVE_N * (int)sizeof(E), RS = RB + 16, SHARE = T::SMEM / 4;       // (padded: the lanes' writes spread over the banks)
    static_assert(2 * 16 * RS <= SHARE, "two blocks in a wave's share: the one before may still be on its way out");
    constexpr int CH = RB / 16, RPI = KA_WAVE / CH;                                         // chunks of a row, rows of a store instruction
    unsigned char* const mine = lds + wave * SHARE;
    const int col = lane % 16, quarter = lane / 16;
    gd_static_for<0, TX>([&](auto b_c) {
        constexpr int b = decltype(b_c)::value;
        unsigned char* const slot = mine + b % 2 * 16 * RS;
        gd_static_for<0, TW>([&](auto a_c) {
            constexpr int a = decltype(a_c)::value;
            const floatx4 v = take(a_c, b_c);
            unsigned char* const at = slot + col * RS + (a * 16 + quarter * 4) * (int)sizeof(E);
            if constexpr (sizeof(E) == 2) *reinterpret_cast<bf16x4*>(at) = bf16x4{(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
            else *reinterpret_cast<floatx4*>(at) = v;
        });
        at_epilogue_wave_sync();
#pragma unroll
        for (int r0 = 0; r0 < 16; r0 += RPI) {
            const int r = r0 + lane / CH, c = lane % CH;
            if (lane < RPI * CH && r < 16) store(b * 16 + r, c * (int)(16 / sizeof(E)), slot + r * RS + c * 16);
        }
        at_epilogue_wave_sync();
    });
}

// out[s] = act[s](A W[s]^T + bias[s]), s = 0, 1 (N[1] = 0: one linear), in bf16; or, one linear alone, in fp32, added to what is there if `accumulate`. The tiles of the second
// linear follow those of the first.
struct KqLinears {
    const bf16_t* A;        // [M, K]
    long lda;
    int M, K, tiles_m, tiles_n[2], accumulate;
    const bf16_t* W[2];     // [N[s], K]
    const float* bias[2];   // may be null
    void* out[2];           // [M, N[s]]
    long ldw[2], ldo[2];
    int N[2], act[2];
};

template <int TW, int TX, int NS, bool F32>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
quad_tiles_kernel(KqLinears p) {
    using T = KqTile<TW, TX, NS>;
    using E = std::conditional_t<F32, float, bf16_t>;
    extern __shared__ __attribute__((aligned(16))) unsigned char kq_lds[];
    const int total = (p.tiles_n[0] + p.tiles_n[1]) * p.tiles_m, per_xcd = (total + 7) / 8;
    const int logical = blockIdx.x % 8 * per_xcd + blockIdx.x / 8;      // an XCD's tiles: neighbours in N, whose rows of W they share
    if (logical >= total || (int)blockIdx.x / 8 >= per_xcd) return;
    const int m0 = logical % p.tiles_m * T::BM, tile = logical / p.tiles_m;
    const bool second = tile >= p.tiles_n[0];
    const int n0 = (second ? tile - p.tiles_n[0] : tile) * T::BN;
    const char* const W = (const char*)(second ? p.W[1] : p.W[0]);
    const long ldw = second ? p.ldw[1] : p.ldw[0], ldo = second ? p.ldo[1] : p.ldo[0];
    const int N = second ? p.N[1] : p.N[0], act = second ? p.act[1] : p.act[0];
    const float* const bias = second ? p.bias[1] : p.bias[0];
    E* const out = (E*)(second ? p.out[1] : p.out[0]);
    const char* const A = (const char*)p.A;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KA_WAVE), lane = threadIdx.x % KA_WAVE;
    // (bytes from the operand's start, which the host has checked to fit in 32 bits; rows past the end are read from the last row, and never stored)
    unsigned woff[T::WL], xoff[T::XL];
#pragma unroll
    for (int i = 0; i < T::WL; ++i) {
        const int r = T::w_row(i, wave, lane);
        woff[i] = (unsigned)(min(n0 + r, N - 1) * ldw + kd_load_channel<8>(r, lane)) * 2u;
    }
#pragma unroll
    for (int i = 0; i < T::XL; ++i) {
        const int r = T::x_row(i, wave, lane);
        xoff[i] = (unsigned)(min(m0 + r, p.M - 1) * p.lda + kd_load_channel<8>(r, lane)) * 2u;
    }
    floatx4 acc[TW][TX];
#pragma unroll
    for (int a = 0; a < TW; ++a)
#pragma unroll
        for (int b = 0; b < TX; ++b) acc[a][b] = floatx4{0.f, 0.f, 0.f, 0.f};
    asm volatile("" ::"s"(bias), "s"(out), "s"(ldo), "s"(act), "s"(p.M), "s"(N), "s"(p.accumulate));      // (no scalar load later, on the counter of the LDS reads)
    kq_product<TW, TX, NS>(kq_lds, wave, lane, p.K / 64, [&](int i, int t) { return W + (size_t)t * 128 + woff[i]; },
                           [&](int i, int t) { return A + (size_t)t * 128 + xoff[i]; }, acc);
    gd_barrier();                                        // the last K-step has been read by everybody
    const int n_wave = n0 + wave / 2 * T::WAVE_N, m_wave = m0 + wave % 2 * T::WAVE_M, quarter = lane / 16;
    // (N is a multiple of 8: four columns of a tile are inside it or past it together, and so are the eight, or four, of a store)
    floatx4 add[TW];
#pragma unroll
    for (int a = 0; a < TW; ++a) {
        const int n = n_wave + a * 16 + quarter * 4;
        add[a] = bias && n < N ? *reinterpret_cast<const floatx4*>(bias + n) : floatx4{0.f, 0.f, 0.f, 0.f};
    }
    auto rows_out = [&](auto activate) {
        kq_rows_out<E, TW, TX, NS>(
            kq_lds, wave, lane,
            [&](auto a, auto b) {
                floatx4 v = acc[a.value][b.value] + add[a.value];
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = activate(v[i]);
                return v;
            },
            [&](int r, int c, const unsigned char* from) {
                const int m = m_wave + r, n = n_wave + c;
                if (m >= p.M || n >= N) return;
                floatx4* const at = reinterpret_cast<floatx4*>(out + (size_t)m * ldo + n);
                const floatx4 v = *reinterpret_cast<const floatx4*>(from);
                if constexpr (F32) *at = p.accumulate ? *at + v : v;
                else *at = v;
            });
    };
    // (the two activations that matter have an epilogue of their own: chosen per value, an activation costs a branch a value)
    if (act == KA_ACT_NONE) rows_out([](float x) { return x; });
    else if (act == KA_ACT_GELU_TANH) rows_out([](float x) { return ka_gelu_tanh_fast(x); });
    else rows_out([&](float x) { return ka_activate_fast(act, x); });
}

template <int TW, int TX, int NS, bool F32>
static int launch_quad(KqLinears p, hipStream_t stream) {
    using T = KqTile<TW, TX, NS>;
    static bool configured = false;
    auto kernel = quad_tiles_kernel<TW, TX, NS, F32>;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, T::SMEM);
        KA_CHECK(e == hipSuccess, "linears by tiles: cannot reserve %d bytes of LDS: %s", T::SMEM, hipGetErrorString(e));
        configured = true;
    }
    p.tiles_m = ka_cdiv(p.M, T::BM);
    for (int s = 0; s < 2; ++s) p.tiles_n[s] = ka_cdiv(p.N[s], T::BN);
    const long total = ((long)(p.tiles_n[0] + p.tiles_n[1]) * p.tiles_m + 7) / 8 * 8;
    KA_CHECK(total < (1L << 31), "linears by tiles: too many tiles");
    hipLaunchKernelGGL(kernel, dim3((unsigned)total), dim3(256), T::SMEM, stream, p);
    KA_LAUNCH_CHECK();
    return 0;
}

// Tiles by their code (gemm_quad_bf16.hip, gemm_quad_f32_bf16.hip); 1, 2 and 4 are the phased tiles' (gemm_phased_bf16.hip).
int ka_quad_bf16(const KqLinears& p, int code, hipStream_t stream);
int ka_quad_f32(const KqLinears& p, int code, hipStream_t stream);

#define KQ_TILES(LAUNCH)   \
    switch (code) {        \
        case 6: return LAUNCH(2, 4, 4); \
        case 7: return LAUNCH(3, 4, 4); \
        case 8: return LAUNCH(4, 4, 4); \
        case 5: return LAUNCH(5, 4, 4); \
        case 3: return LAUNCH(4, 6, 4); \
        case 9: return LAUNCH(3, 8, 3); \
        case 10: return LAUNCH(5, 6, 3); \
        case 11: return LAUNCH(4, 8, 3); \
        case 12: return LAUNCH(5, 8, 3); \
    }
