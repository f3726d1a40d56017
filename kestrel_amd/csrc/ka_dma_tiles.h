// The loop over K of the large-tile matrix products: operands go from global memory straight into LDS.
//
// Four or eight waves (GN x GM), each with WN x WM MFMA tiles of 32 x 32: a tile of BN = 32 WN GN rows of the row operand W by
// BM = 32 WM GM rows of the column operand X. K-steps of BK come by global_load_lds_dwordx4 (no registers, no ds_write)
// into NS stages, one barrier per step. Chunk c (16 bytes) of tile row r lies at place c ^ kd_swizzle(r) of its row, chosen by
// which chunk each lane of the load asks for, so that the rows that one pass of a 16-byte LDS read touches fall on
// different banks without padding. K must be a multiple of BK. Which rows of memory the tile's rows are is the caller's
// business (an address per load and lane), so they may as well be gathered.
#pragma once

#include "ka_common.h"

#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(16))) float floatx16;
typedef __attribute__((ext_vector_type(4))) float floatx4;

constexpr int gd_smem(int bn, int bm, int bk, int ns) { return ns * (bn + bm) * bk * 2; }

// A loop whose index is a compile-time constant in every round (the accumulators are up to 256
// registers: an index the compiler does not resolve would put them in memory).
template <int I, int N, typename F>
__device__ __forceinline__ void gd_static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        gd_static_for<I + 1, N>(f);
    }
}

#define GD_GLOBAL __attribute__((address_space(1)))
#define GD_LDS __attribute__((address_space(3)))

// s_waitcnt vmcnt(n) alone (gfx9 encoding: vmcnt in bits 3:0 and 15:14, the other counters at their maximum)
template <int N>
__device__ __forceinline__ void gd_wait_loads() {
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0f70);
}

// Waits until at most `younger` x LPW of this wave's loads are still in flight (the count of an
// s_waitcnt is an immediate: one instruction per value that can occur, at most MAX).
template <int LPW, int MAX>
__device__ __forceinline__ void gd_wait_younger(int younger) {
    static_assert(LPW * (MAX > 0 ? MAX : 0) <= 63, "more loads in flight than the counter holds");
    if constexpr (MAX <= 0) {
        gd_wait_loads<0>();
    } else {
        if (younger >= MAX) gd_wait_loads<LPW * MAX>();
        else gd_wait_younger<LPW, MAX - 1>(younger);
    }
}

// s_waitcnt lgkmcnt(0) alone: this wave's LDS reads have all arrived in its registers
__device__ __forceinline__ void gd_wait_lds() { __builtin_amdgcn_s_waitcnt(0xc07f); }

// The barrier alone, without the fence that __syncthreads() puts before it: that fence waits
// for every load in flight, the younger stages' too. What must be ordered here is ordered by
// hand: a wave has waited for its own loads of the stage (vmcnt) and for its LDS reads of the
// stage before (their values were used) when it arrives.
__device__ __forceinline__ void gd_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Orders the LDS traffic of one wave: what its lanes wrote before is seen by its lanes after.
__device__ __forceinline__ void at_epilogue_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The sizes that follow from a tile's shape; EDGE: rows and columns of an MFMA tile.
template <int WN, int WM, int GN, int GM, int BK, int NS, int EDGE = 32>
struct KdTile {
    static_assert(BK == 32 || BK == 64, "K-steps of 32 or 64");
    static_assert(NS >= 2 && NS <= 8, "two to eight stages");
    static_assert(GN * GM == 4 || GN * GM == 8, "four or eight waves");
    static constexpr int WAVES = GN * GM;
    static constexpr int BN = EDGE * WN * GN, BM = EDGE * WM * GM;
    static constexpr int ROW = BK * 2;                          // bytes of a tile row
    static constexpr int CPR = BK / 8;                          // 16-byte chunks of a tile row
    static constexpr int RPL = KA_WAVE / CPR;                   // rows that one load of 1 KB brings
    static constexpr int STAGE = (BN + BM) * ROW;               // bytes of one stage: W rows, then X rows
    static constexpr int W_LOADS = BN / RPL / WAVES, X_LOADS = BM / RPL / WAVES;   // loads per wave and stage
    static_assert(W_LOADS * RPL * WAVES == BN && X_LOADS * RPL * WAVES == BM, "the tile does not divide over the waves' loads");
    static constexpr int LPW = W_LOADS + X_LOADS;
    static constexpr int SMEM = gd_smem(BN, BM, BK, NS);
};

// One pass of a 16-byte LDS read serves 16 lanes, which here read the same chunk of 16 consecutive rows, and the 64 banks
// hold 256 bytes: two rows of 128 bytes, so rows of the same parity must differ in their place ((r >> 1) & 7), or four rows
// of 64 bytes ((r >> 2) & 3). (Measured with r & 7: half of the LDS cycles were bank conflicts, rows r and r + 8 meeting
// in one pass.)
template <int CPR>
__device__ __forceinline__ int kd_swizzle(int r) { return CPR == 8 ? ((r >> 1) & 7) : ((r >> 2) & 3); }

// The tile row whose piece this lane asks for in load `i` of the wave's loads of one operand, and the first channel of the
// piece within a K-step.
template <int CPR>
__device__ __forceinline__ int kd_load_row(int load, int lane) { return load * (KA_WAVE / CPR) + lane / CPR; }
template <int CPR>
__device__ __forceinline__ int kd_load_channel(int row, int lane) { return ((lane % CPR) ^ kd_swizzle<CPR>(row)) * 8; }

// acc[a][b] += the products of this wave's tiles over K. wsrc[i], xsrc[i]: this lane's address at K-step 0 of the wave's load i
// (rows wave * W_LOADS + i and so on, kd_load_row; valid whatever the row is). The whole workgroup takes part.
// HALVES: which channels of a K-step meet in a product: slice j takes eight from place 8 j of either half of the step, as
// kl_tile_product does (ka_listed_tiles.h), and the sums have its bits; without it sixteen neighbours. Both cost the same.
template <int WN, int WM, int GN, int GM, int BK, int NS, int SL, bool HALVES = false>
__device__ __forceinline__ void kd_product(unsigned char* lds, int wave, int lane, int K,
                                           const bf16_t* const (&wsrc)[KdTile<WN, WM, GN, GM, BK, NS>::W_LOADS],
                                           const bf16_t* const (&xsrc)[KdTile<WN, WM, GN, GM, BK, NS>::X_LOADS], floatx16 (&acc)[WN][WM]) {
    using T = KdTile<WN, WM, GN, GM, BK, NS>;
    constexpr int BN = T::BN, ROW = T::ROW, CPR = T::CPR, RPL = T::RPL, STAGE = T::STAGE, W_LOADS = T::W_LOADS, X_LOADS = T::X_LOADS, LPW = T::LPW;
    const int wn = wave / GM, wm = wave % GM;
    const int li = lane % 32, lg = lane / 32;
    auto fetch = [&](int stage, int k0) {
        unsigned char* base = lds + stage * STAGE;
#pragma unroll
        for (int i = 0; i < W_LOADS; ++i)
            __builtin_amdgcn_global_load_lds((const GD_GLOBAL void*)(wsrc[i] + k0),
                                             (GD_LDS void*)(base + (wave * W_LOADS + i) * RPL * ROW), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < X_LOADS; ++i)
            __builtin_amdgcn_global_load_lds((const GD_GLOBAL void*)(xsrc[i] + k0),
                                             (GD_LDS void*)(base + BN * ROW + (wave * X_LOADS + i) * RPL * ROW), 16, 0, 0);
    };

    // operand addresses inside a stage: tile row li of each of this wave's tiles; the k-chunk
    // of slice ks is ks * 2 + lg, by halves lg * CPR / 2 + ks
    int wrow_off[WN], xrow_off[WM];
#pragma unroll
    for (int a = 0; a < WN; ++a) wrow_off[a] = (wn * 32 * WN + a * 32 + li) * ROW;
#pragma unroll
    for (int b = 0; b < WM; ++b) xrow_off[b] = BN * ROW + (wm * 32 * WM + b * 32 + li) * ROW;
    const int swz = kd_swizzle<CPR>(li);

    // The K-steps' operands are read from LDS a group of SL k-slices (of 16) at a time, one group
    // ahead of the group that is being multiplied, also across the edge of a K-step: the MFMAs of a
    // stage's last group run while the first group of the next stage is on its way from LDS, so the
    // matrix pipes do not stand still at every K-step while both waves of a SIMD wait for LDS
    // together. For that the barrier of a K-step stands before the last group's MFMAs: a wave
    // arrives when its own loads of the next stage have landed and its own reads of this stage are
    // in its registers. After the barrier everybody's have, so the next stage may be read and this
    // stage's memory may be written: the load of stage s + NS goes out, and has NS - 1 K-steps to land.
    constexpr int G = BK / 16 / SL;                      // groups per K-step
    static_assert(G * SL * 16 == BK, "the groups of slices do not divide a K-step");
    const int steps = K / BK;
    // NS stages go out at once; the first has to be there before anything can be read
#pragma unroll
    for (int st = 0; st < NS; ++st)
        if (st < steps) fetch(st, st * BK);
    {
        const int younger = min(NS - 1, steps - 1);
        gd_wait_younger<LPW, NS - 1>(younger);
        gd_barrier();
    }
    bf16x8 wa[2][SL][WN], xb[2][SL][WM];
    auto operands = [&](auto slot_c, int stage, int g) {
        constexpr int slot = decltype(slot_c)::value;
        const unsigned char* base = lds + (stage % NS) * STAGE;
#pragma unroll
        for (int i = 0; i < SL; ++i) {
            const int slice = g * SL + i, place = ((HALVES ? lg * (CPR / 2) + slice : slice * 2 + lg) ^ swz) * 16;
#pragma unroll
            for (int a = 0; a < WN; ++a) wa[slot][i][a] = *reinterpret_cast<const bf16x8*>(base + wrow_off[a] + place);
#pragma unroll
            for (int b = 0; b < WM; ++b) xb[slot][i][b] = *reinterpret_cast<const bf16x8*>(base + xrow_off[b] + place);
        }
    };
    const int groups = steps * G;
    // group t (stage t / G, its group t % G) is multiplied from the registers of slot t & 1
    auto group = [&](auto slot_c, int t) {
        constexpr int slot = decltype(slot_c)::value;
        const int st = t / G, g = t % G;
        if (g == G - 1 && st + 1 < steps) {
            // own loads of stage st + 1 landed (the stages after it may stay in flight), own reads of
            // stage st done (they are the operands of this group, needed below in any case)
            const int younger = min(NS - 2, steps - 2 - st);
            gd_wait_younger<LPW, NS - 2>(younger);
            gd_wait_lds();
            gd_barrier();
            if (st + NS < steps) fetch(st % NS, (st + NS) * BK);
        }
        // (always, also after the last group, whose "next" is read from memory nobody needs: a read
        // under a condition makes the compiler wait for every read in flight before the MFMAs,
        // the ones just asked for included)
        operands(std::integral_constant<int, slot ^ 1>{}, (t + 1) / G, (t + 1) % G);
#pragma unroll
        for (int i = 0; i < SL; ++i)
#pragma unroll
            for (int a = 0; a < WN; ++a)
#pragma unroll
                for (int b = 0; b < WM; ++b)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wa[slot][i][a], xb[slot][i][b], acc[a][b], 0, 0, 0);
        // The reads of the next group go out behind this group's second MFMA, into registers of
        // their own, and have the rest of the group's MFMAs to arrive. (Left to itself the compiler
        // gives both groups the same registers and asks for the next operands only after the
        // MFMAs that use the present ones, three MFMAs before they are needed. Asked for ahead of
        // the group's first MFMA they would be waited for at once: the compiler waits for every
        // read in flight where this loop needs the older ones only.)
        constexpr int FIRST = SL * WN * WM > 2 ? 2 : 1;
        __builtin_amdgcn_sched_group_barrier(0x008, FIRST, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, SL * (WN + WM), 0);
        __builtin_amdgcn_sched_group_barrier(0x008, SL * WN * WM - FIRST, 0);
    };
    // (Nothing but LDS reads may be in flight on the counter they share with scalar loads when the
    // loop is entered: with a scalar load among them the compiler can no longer count on arrival
    // in order and waits, in every round, for all reads, the ones just asked for included.)
    gd_wait_lds();
    operands(std::integral_constant<int, 0>{}, 0, 0);
    int t = 0;
    for (; t + 1 < groups; t += 2) {
        group(std::integral_constant<int, 0>{}, t);
        group(std::integral_constant<int, 1>{}, t + 1);
    }
    if (t < groups) group(std::integral_constant<int, 0>{}, t);
}

// The same on MFMA tiles of 16 x 16 by 32 channels, two products a K-step of 64, for sums that have to have the order (and so the bits) of a
// kernel that streams weights through registers, whatever the number of rows:
//  * KD_HALVES: the first product takes channels 0 .. 31 of a step, the second 32 .. 63, each into sums of its own (skinny_wide_kernel);
//  * KD_FOURTHS: the four lane groups hold sixteen neighbours each, the first product takes eight of each, and every fourth K-step goes
//    into the same sums (ef_columns).
// acc[c][a][b], c the set of sums; weight(i, step), row(i, step): this lane's address of load i at that K-step (as wsrc and xsrc above).
enum { KD_HALVES = 2, KD_FOURTHS = 4 };

template <int WN, int WM, int GN, int GM, int NS, int ORDER, typename Weight, typename Row>
__device__ __forceinline__ void kd_product_16(unsigned char* lds, int wave, int lane, int steps, Weight weight, Row row, floatx4 (&acc)[ORDER][WN][WM]) {
    using T = KdTile<WN, WM, GN, GM, 64, NS, 16>;
    constexpr int BN = T::BN, ROW = T::ROW, CPR = T::CPR, RPL = T::RPL, STAGE = T::STAGE, W_LOADS = T::W_LOADS, X_LOADS = T::X_LOADS, LPW = T::LPW;
    const int wn = wave / GM, wm = wave % GM, col = lane % 16, quarter = lane / 16;
    auto fetch = [&](int stage, int step) {
        unsigned char* base = lds + stage * STAGE;
#pragma unroll
        for (int i = 0; i < W_LOADS; ++i)
            __builtin_amdgcn_global_load_lds((const GD_GLOBAL void*)weight(i, step), (GD_LDS void*)(base + (wave * W_LOADS + i) * RPL * ROW), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < X_LOADS; ++i)
            __builtin_amdgcn_global_load_lds((const GD_GLOBAL void*)row(i, step), (GD_LDS void*)(base + BN * ROW + (wave * X_LOADS + i) * RPL * ROW), 16, 0, 0);
    };
    int wrow_off[WN], xrow_off[WM];
#pragma unroll
    for (int a = 0; a < WN; ++a) wrow_off[a] = ((wn * WN + a) * 16 + col) * ROW;
#pragma unroll
    for (int b = 0; b < WM; ++b) xrow_off[b] = (BN + (wm * WM + b) * 16 + col) * ROW;
    const int swz = kd_swizzle<CPR>(col);
    // As in kd_product, a group being a whole K-step: the operands of the next step are read from LDS behind the first products of this one.
#pragma unroll
    for (int st = 0; st < NS; ++st)
        if (st < steps) fetch(st, st);
    gd_wait_younger<LPW, NS - 1>(min(NS - 1, steps - 1));
    gd_barrier();
    bf16x8 wa[2][2][WN], xb[2][2][WM];
    auto operands = [&](auto slot_c, int stage) {
        constexpr int slot = decltype(slot_c)::value;
        const unsigned char* base = lds + (stage % NS) * STAGE;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int place = ((ORDER == KD_HALVES ? u * 4 + quarter : quarter * 2 + u) ^ swz) * 16;
#pragma unroll
            for (int a = 0; a < WN; ++a) wa[slot][u][a] = *reinterpret_cast<const bf16x8*>(base + wrow_off[a] + place);
#pragma unroll
            for (int b = 0; b < WM; ++b) xb[slot][u][b] = *reinterpret_cast<const bf16x8*>(base + xrow_off[b] + place);
        }
    };
    auto step = [&](auto place_c, int st) {             // st % 4 == place
        constexpr int place = decltype(place_c)::value, slot = place & 1;
        if (st + 1 < steps) {
            gd_wait_younger<LPW, NS - 2>(min(NS - 2, steps - 2 - st));
            gd_wait_lds();
            gd_barrier();
            if (st + NS < steps) fetch(st % NS, st + NS);
        }
        operands(std::integral_constant<int, slot ^ 1>{}, st + 1);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            constexpr int fourth = place;
            const int c = ORDER == KD_HALVES ? u : fourth;
#pragma unroll
            for (int a = 0; a < WN; ++a)
#pragma unroll
                for (int b = 0; b < WM; ++b) acc[c][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[slot][u][a], xb[slot][u][b], acc[c][a][b], 0, 0, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * (WN + WM), 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 2 * WN * WM - 2, 0);
    };
    gd_wait_lds();
    operands(std::integral_constant<int, 0>{}, 0);
    int st = 0;
    for (; st + 3 < steps; st += 4) {
        step(std::integral_constant<int, 0>{}, st);
        step(std::integral_constant<int, 1>{}, st + 1);
        step(std::integral_constant<int, 2>{}, st + 2);
        step(std::integral_constant<int, 3>{}, st + 3);
    }
    if (st < steps) step(std::integral_constant<int, 0>{}, st);
    if (st + 1 < steps) step(std::integral_constant<int, 1>{}, st + 1);
    if (st + 2 < steps) step(std::integral_constant<int, 2>{}, st + 2);
}
