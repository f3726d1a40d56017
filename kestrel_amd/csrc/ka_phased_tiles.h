// The loop over K of matrix products with enough rows for tiles of 128 rows and more: products and everything else in turns.
//
// Eight waves (GW x GX), two on every SIMD, and a tile of BN rows of W by BM rows of X, either in two halves. A K-step of 64 is four
// phases, each a quarter of the tile (half of W by half of X): its operands from LDS, a half of a later K-step on its way from
// memory into LDS, a barrier, its products, a barrier. The second four waves run half a phase behind the first four, so that of the two
// waves of a SIMD one always multiplies while the other reads. The halves of a K-step are asked for six phases before they are read (about
// 1.3 us) and waited for by count, never all of them.
//
// On every CU at once this is bound by the clock under load, not by a wait: 256 x 256 takes 1.42 us a K-step on 256 CUs and 1.04 on 64,
// 1.21 without a load in the loop (1.6 PFLOP/s at the most that way; 0.85 us at the nominal clock). The lockstep loop of ka_dma_tiles.h at
// 256 x 256 by the same eight waves takes about 1.9.
#pragma once

#include "ka_dma_tiles.h"

// QW0, QW1, QX0, QX1: MFMA tiles of 16 that a wave has of either half of W and X. Rows of a wave's W halves are neighbours in the
// output: tile row (wave, half, j) is row (wave * (QW0 + QW1) + half * QW0) * 16 + j of the tile, and likewise X.
template <int QW0, int QW1, int QX0, int QX1, int GW, int GX>
struct KpTile {
    static_assert(GW * GX == 8, "eight waves");
    static constexpr int QW = QW0 > QW1 ? QW0 : QW1, QX = QX0 > QX1 ? QX0 : QX1;
    static constexpr int W0 = 16 * QW0 * GW, W1 = 16 * QW1 * GW, X0 = 16 * QX0 * GX, X1 = 16 * QX1 * GX;      // rows of the halves
    static constexpr int BN = W0 + W1, BM = X0 + X1;
    static constexpr int LW0 = W0 / 64, LW1 = W1 / 64, LX0 = X0 / 64, LX1 = X1 / 64;                          // loads of 1 KB per wave and half
    static_assert(LW0 * 64 == W0 && LW1 * 64 == W1 && LX0 * 64 == X0 && LX1 * 64 == X1, "halves in steps of 64 rows");
    static_assert(LW0 > 0 && LW1 > 0 && LX0 > 0 && LX1 > 0, "two halves of either operand");
    static constexpr int LOADS = LW0 + LW1 + LX0 + LX1;
    static constexpr int STAGE = (BN + BM) * 128;       // bytes of a K-step: both halves of W, then of X
    static constexpr int SMEM = 2 * STAGE;
    static constexpr int WAVE_N = 16 * (QW0 + QW1), WAVE_M = 16 * (QX0 + QX1);                                // a wave's outputs

    // What this lane asks for in load i of the wave's loads of W (X): the row of the tile, and the first channel of the K-step.
    static __device__ __forceinline__ int w_row(int i, int wave, int lane) { return row<QW0, QW1, LW0>(w_place(i, wave, lane), i); }
    static __device__ __forceinline__ int x_row(int i, int wave, int lane) { return row<QX0, QX1, LX0>(x_place(i, wave, lane), i); }
    static __device__ __forceinline__ int w_channel(int i, int wave, int lane) { return kd_load_channel<8>(w_place(i, wave, lane), lane); }
    static __device__ __forceinline__ int x_channel(int i, int wave, int lane) { return kd_load_channel<8>(x_place(i, wave, lane), lane); }

   private:
    // the row of the half as it lies in LDS
    static __device__ __forceinline__ int w_place(int i, int wave, int lane) { return kd_load_row<8>(i >= LW0 ? wave * LW1 + i - LW0 : wave * LW0 + i, lane); }
    static __device__ __forceinline__ int x_place(int i, int wave, int lane) { return kd_load_row<8>(i >= LX0 ? wave * LX1 + i - LX0 : wave * LX0 + i, lane); }
    template <int Q0, int Q1, int L0>
    static __device__ __forceinline__ int row(int place, int i) {
        const bool second = i >= L0;
        const int per = 16 * (second ? Q1 : Q0);
        return place / per * 16 * (Q0 + Q1) + (second ? 16 * Q0 : 0) + place % per;
    }
};

// acc[h][g][a][b] += the products of this wave's MFMA tiles: tile a of half h of W (its rows the product's rows) by tile b of half g of X.
// wsrc(i, t), xsrc(i, t): this lane's address of its load i at K-step t (the row of w_row / x_row, clamped to what is there, its chunk). steps >= 2.
// The whole workgroup takes part; LDS is free again when the last wave returns (a barrier is the caller's).
template <int QW0, int QW1, int QX0, int QX1, int GW, int GX, typename Weight, typename Row>
__device__ __forceinline__ void kp_product(unsigned char* lds, int wave, int lane, int steps, Weight wsrc, Row xsrc,
                                           floatx4 (&acc)[2][2][QW0 > QW1 ? QW0 : QW1][QX0 > QX1 ? QX0 : QX1]) {
    using T = KpTile<QW0, QW1, QX0, QX1, GW, GX>;
    const int wn = wave / GX, wm = wave % GX, col = lane % 16, quarter = lane / 16;
    constexpr int OFF_W1 = T::W0 * 128, OFF_X0 = T::BN * 128, OFF_X1 = OFF_X0 + T::X0 * 128;
    using C0 = std::integral_constant<int, 0>;
    using C1 = std::integral_constant<int, 1>;
    auto fetch_w = [&](auto half_c, auto buf_c, int t) {
        constexpr int half = decltype(half_c)::value, n = half ? T::LW1 : T::LW0;
        unsigned char* base = lds + decltype(buf_c)::value * T::STAGE + (half ? OFF_W1 : 0);
#pragma unroll
        for (int i = 0; i < n; ++i)
            __builtin_amdgcn_global_load_lds((const GD_GLOBAL void*)wsrc(half ? T::LW0 + i : i, t), (GD_LDS void*)(base + (wave * n + i) * 1024), 16, 0, 0);
    };
    auto fetch_x = [&](auto half_c, auto buf_c, int t) {
        constexpr int half = decltype(half_c)::value, n = half ? T::LX1 : T::LX0;
        unsigned char* base = lds + decltype(buf_c)::value * T::STAGE + (half ? OFF_X1 : OFF_X0);
#pragma unroll
        for (int i = 0; i < n; ++i)
            __builtin_amdgcn_global_load_lds((const GD_GLOBAL void*)xsrc(half ? T::LX0 + i : i, t), (GD_LDS void*)(base + (wave * n + i) * 1024), 16, 0, 0);
    };
    // (an MFMA tile starts at a multiple of 16 rows, so the swizzle of a row is that of its lane)
    const int swz = kd_swizzle<8>(col);
    const int place[2] = {(quarter ^ swz) * 16, ((quarter + 4) ^ swz) * 16};
    bf16x8 wr[2][T::QW], xr[2][2][T::QX];
    auto read_w = [&](auto half_c, auto buf_c) {
        constexpr int half = decltype(half_c)::value, n = half ? QW1 : QW0;
        const unsigned char* base = lds + decltype(buf_c)::value * T::STAGE + (half ? OFF_W1 : 0) + (wn * n * 16 + col) * 128;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int a = 0; a < n; ++a) wr[u][a] = *reinterpret_cast<const bf16x8*>(base + a * 2048 + place[u]);
    };
    auto read_x = [&](auto half_c, auto buf_c, auto set_c) {
        constexpr int half = decltype(half_c)::value, n = half ? QX1 : QX0, set = decltype(set_c)::value;
        const unsigned char* base = lds + decltype(buf_c)::value * T::STAGE + (half ? OFF_X1 : OFF_X0) + (wm * n * 16 + col) * 128;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int b = 0; b < n; ++b) xr[set][u][b] = *reinterpret_cast<const bf16x8*>(base + b * 2048 + place[u]);
    };
    auto multiply = [&](auto hw_c, auto hx_c, auto set_c) {
        constexpr int hw = decltype(hw_c)::value, hx = decltype(hx_c)::value, set = decltype(set_c)::value;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int a = 0; a < (hw ? QW1 : QW0); ++a)
#pragma unroll
                for (int b = 0; b < (hx ? QX1 : QX0); ++b)
                    acc[hw][hx][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wr[u][a], xr[set][u][b], acc[hw][hx][a][b], 0, 0, 0);
    };
    // Between a phase's reads and its products, and behind them. The wait for the wave's own LDS reads stands in front of the products of
    // every phase: when two phases later a load writes over what was read here, no wave's read can still be on its way.
    auto begin = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        gd_barrier();
        gd_wait_lds();
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
    };
    auto end = [&]() {
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
        gd_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    // Waits until the half that the next phase reads has landed; A, B, C: how many of this wave's loads are younger than it with two or
    // more K-steps behind this one, with one, with none.
    auto landed = [&](auto a_c, auto b_c, auto c_c, bool two, bool one) {
        if (two) gd_wait_loads<decltype(a_c)::value>();
        else if (one) gd_wait_loads<decltype(b_c)::value>();
        else gd_wait_loads<decltype(c_c)::value>();
    };
#define KP_N(x) std::integral_constant<int, (x)>{}
    constexpr int L = T::LOADS;
    // One K-step, its number's parity PAR. A half's memory is written again two phases after it was last read, for the K-step after
    // next: X0 (read in the fourth phase of the K-step before) in the second phase, W0 in the third, X1 in the fourth, W1 in the first of the next.
    auto step = [&](auto par_c, int t) {
        constexpr int par = decltype(par_c)::value;
        using P = std::integral_constant<int, par>;
        using O = std::integral_constant<int, par ^ 1>;
        const bool one = t + 1 < steps, two = t + 2 < steps;
        read_w(C0{}, P{});
        if (one) fetch_w(C1{}, O{}, t + 1);
        landed(KP_N(L + T::LW1), KP_N(L + T::LW1), KP_N(T::LW1), two, one);
        begin();
        multiply(C0{}, C0{}, P{});
        end();
        read_x(C1{}, P{}, O{});
        if (two) fetch_x(C0{}, P{}, t + 2);
        landed(KP_N(L + T::LX0), KP_N(L), KP_N(0), two, one);
        begin();
        multiply(C0{}, C1{}, O{});
        end();
        read_w(C1{}, P{});
        if (two) fetch_w(C0{}, P{}, t + 2);
        landed(KP_N(L + T::LW0), KP_N(L - T::LX0), KP_N(0), two, one);
        begin();
        multiply(C1{}, C1{}, O{});
        end();
        read_x(C0{}, O{}, O{});                         // (behind the last K-step: of memory that nobody needs)
        if (two) fetch_x(C1{}, P{}, t + 2);
        landed(KP_N(L + T::LX1), KP_N(T::LX1 + T::LW1), KP_N(0), two, one);
        begin();
        multiply(C1{}, C0{}, P{});
        end();
    };
#undef KP_N
    fetch_x(C0{}, C0{}, 0);
    fetch_w(C0{}, C0{}, 0);
    fetch_x(C1{}, C0{}, 0);
    fetch_w(C1{}, C0{}, 0);
    fetch_x(C0{}, C1{}, 1);
    fetch_w(C0{}, C1{}, 1);
    fetch_x(C1{}, C1{}, 1);
    gd_wait_loads<T::LX1 + T::LW1 + T::LX0 + T::LW0 + T::LX1>();
    gd_barrier();
    if (wave >= 4) gd_barrier();                        // half a phase behind
    read_x(C0{}, C0{}, C0{});
#pragma unroll 1
    for (int t = 0;; t += 2) {
        step(C0{}, t);
        if (t + 1 >= steps) break;
        step(C1{}, t + 1);
        if (t + 2 >= steps) break;
    }
    if (wave < 4) gd_barrier();
}

// A wave's outputs as whole rows. For each of its 16 WAVE_M / 16 blocks of 16 rows: take(h, g, a, b) gives four neighbouring columns of one row
// (value of MFMA tile a of half h by tile b of half g), which pass through the wave's share of LDS; store(row, column, from) then gets the
// wave's row and first column of 16 bytes of E at `from`. E: float or bf16_t.
template <typename E, int QW0, int QW1, int QX0, int QX1, int GW, int GX, typename Take, typename Store>
__device__ __forceinline__ void kp_rows_out(unsigned char* lds, int wave, int lane, Take take, Store store) {
    using T = KpTile<QW0, QW1, QX0, QX1, GW, GX>;
    constexpr int RB = T::WAVE_N * sizeof(E), RS = RB + 16;     // bytes of a row, and its place: padded so that the lanes' writes spread over the banks
    constexpr int SHARE = T::SMEM / 8;
    static_assert(16 * RS <= SHARE, "a block of rows in a wave's share");
    constexpr int SLOTS = 2 * 16 * RS <= SHARE ? 2 : 1;         // (two: the block before may still be on its way out)
    constexpr int CH = RB / 16, RPI = KA_WAVE / CH;             // chunks of a row, rows of a store instruction
    unsigned char* const mine = lds + wave * SHARE;
    const int col = lane % 16, quarter = lane / 16;
    gd_static_for<0, QX0 + QX1>([&](auto block_c) {
        constexpr int block = decltype(block_c)::value, g = block >= QX0, b = g ? block - QX0 : block;
        unsigned char* const slot = mine + block % SLOTS * 16 * RS;
        gd_static_for<0, QW0 + QW1>([&](auto tile_c) {
            constexpr int tile = decltype(tile_c)::value, h = tile >= QW0, a = h ? tile - QW0 : tile;
            const floatx4 v = take(std::integral_constant<int, h>{}, std::integral_constant<int, g>{}, std::integral_constant<int, a>{}, std::integral_constant<int, b>{});
            unsigned char* const at = slot + col * RS + (tile * 16 + quarter * 4) * sizeof(E);
            if constexpr (sizeof(E) == 2) *reinterpret_cast<bf16x4*>(at) = bf16x4{(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
            else *reinterpret_cast<floatx4*>(at) = v;
        });
        at_epilogue_wave_sync();
#pragma unroll
        for (int r0 = 0; r0 < 16; r0 += RPI) {
            const int r = r0 + lane / CH, c = lane % CH;
            if (lane < RPI * CH && r < 16) store(block * 16 + r, c * (int)(16 / sizeof(E)), slot + r * RS + c * 16);
        }
        at_epilogue_wave_sync();
    });
}
