// Linears of 17 to 64 rows by tiles that have all of K each: no parts of K, no launch that adds them up, and the activations in LDS beside the weights.
//
// Bound by the weights' way from HBM. A tile is BN = 16 TW weight rows by all rows, K in steps of 64 straight into swizzled LDS, a wave per 16 rows; what
// decides is that no CU gets more weight rows than another, so BN comes in steps of 16. In their loop all tiles read 4.7 to 5 TB/s, whatever their stages (four to
// nine), their waves and the rows beside the weights (10 to 64); the rest is some 4 us of start and end.
#include "ka_dma_tiles.h"
#include "ka_partials.h"
#include "ka_skinny.h"

// The order of a sum is that of the kernel that streams weights through registers, whose bits these are:
//  * FW_EIGHTHS, skinny_persistent_kernel: its wave w takes K-steps w, w + 8, ..., the first and second 32 channels of each apart; a sum starts with the bias and
//    takes the waves' in turn. The eight waves' sums are registers of their own here (64 TW a lane; with four and five sixteens
//    all 512 are taken, and 16 and 20 spill), so that K is read in its order (in the waves' order, with
//    one set of sums: 21.3 instead of 17.8 us, 64 rows, 14,336 of 2,048).
//  * FW_HALVES, skinny_wide_kernel with K in one part: all K-steps, the first and second 32 channels apart; the bias behind.
enum { FW_EIGHTHS = 0, FW_HALVES = 1 };

struct FwArgs {
    const bf16_t* A;        // [M, K]
    long lda;
    int M, K, tiles_a;
    SkinnyTarget a, b;      // b.W null: one target; the tiles of the second follow those of the first
};

template <int TW, int GX>
struct FwTile {
    static constexpr int BN = 16 * TW, BM = 16 * GX;
    static constexpr int STAGE = (BN + BM) * 128;
    static constexpr int NS = 81920 / STAGE < 6 ? 81920 / STAGE : 6;            // stages in half of a CU's LDS: two workgroups where there are as many
    static constexpr int WL = (BN / 8 + GX - 1) / GX, LPW = WL + 2;             // loads of 1 KB per wave and K-step (where W's do not divide, the last ones twice)
    static constexpr int SMEM = NS * STAGE;
    static __device__ __forceinline__ int w_load(int i, int wave) { return min(wave * WL + i, BN / 8 - 1); }
};

template <int TW, int GX, int ORDER>
__global__ void __launch_bounds__(64 * GX)
few_whole_kernel(FwArgs p) {
    using T = FwTile<TW, GX>;
    constexpr int NS = T::NS, SUMS = ORDER == FW_EIGHTHS ? SP_WAVES : 1;
    extern __shared__ __attribute__((aligned(16))) unsigned char fw_lds[];
    const int per_xcd = (p.tiles_a + (p.b.W ? (p.b.N + T::BN - 1) / T::BN : 0) + 7) / 8;
    const int tile = blockIdx.x % 8 * per_xcd + blockIdx.x / 8;        // an XCD's tiles: neighbours
    const bool second = tile >= p.tiles_a;
    const int n0 = (second ? tile - p.tiles_a : tile) * T::BN;
    const SkinnyTarget& tg = second ? p.b : p.a;
    if (!tg.W || n0 >= tg.N) return;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KA_WAVE), lane = threadIdx.x % KA_WAVE, col = lane % 16, quarter = lane / 16;
    const int N = tg.N, blocks = p.K / 64;
    const char* wsrc[T::WL];
    const char* xsrc[2];
#pragma unroll
    for (int i = 0; i < T::WL; ++i) {
        const int r = kd_load_row<8>(T::w_load(i, wave), lane);
        wsrc[i] = (const char*)(tg.W + (size_t)min(n0 + r, N - 1) * tg.ldw + kd_load_channel<8>(r, lane));
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = kd_load_row<8>(wave * 2 + i, lane);
        xsrc[i] = (const char*)(p.A + (size_t)min(r, p.M - 1) * p.lda + kd_load_channel<8>(r, lane));
    }
    auto fetch = [&](int stage, int t) {
        unsigned char* const base = fw_lds + stage * T::STAGE;
        const size_t at = (size_t)t * 128;
#pragma unroll
        for (int i = 0; i < T::WL; ++i)
            __builtin_amdgcn_global_load_lds((const GD_GLOBAL void*)(wsrc[i] + at), (GD_LDS void*)(base + T::w_load(i, wave) * 1024), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < 2; ++i)
            __builtin_amdgcn_global_load_lds((const GD_GLOBAL void*)(xsrc[i] + at), (GD_LDS void*)(base + T::BN * 128 + (wave * 2 + i) * 1024), 16, 0, 0);
    };
    const int swz = kd_swizzle<8>(col);
    bf16x8 w[2][2][TW], x[2][2];
    auto operands = [&](auto set_c, int stage) {
        constexpr int set = decltype(set_c)::value;
        const unsigned char* const base = fw_lds + stage * T::STAGE;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int place = ((u * 4 + quarter) ^ swz) * 16;
            x[set][u] = *reinterpret_cast<const bf16x8*>(base + (T::BN + wave * 16 + col) * 128 + place);
#pragma unroll
            for (int a = 0; a < TW; ++a) w[set][u][a] = *reinterpret_cast<const bf16x8*>(base + (a * 16 + col) * 128 + place);
        }
    };
    const floatx4 zero = floatx4{0.f, 0.f, 0.f, 0.f};
    floatx4 acc[SUMS][2][TW], sum[TW];
#pragma unroll
    for (int e = 0; e < SUMS; ++e)
#pragma unroll
        for (int a = 0; a < TW; ++a) acc[e][0][a] = acc[e][1][a] = zero;
    asm volatile("" ::"s"(p.M), "s"(N), "s"(tg.out), "s"(tg.ldo), "s"(tg.act), "s"(tg.out_dtype), "s"(tg.accumulate));
    // The bias comes before everything else, by loads that nothing decides upon (a branch around them would wait for them): without one the weights' first bytes.
    const float* const bias = tg.bias ? tg.bias : reinterpret_cast<const float*>(tg.W);
#pragma unroll
    for (int a = 0; a < TW; ++a) sum[a] = *reinterpret_cast<const floatx4*>(bias + (tg.bias ? min(n0 + a * 16 + quarter * 4, N - 4) : 0));
    __builtin_amdgcn_sched_barrier(0);
    for (int s = 0; s < NS; ++s)
        if (s < blocks) fetch(s, s);
    gd_wait_younger<T::LPW, NS - 1>(min(NS - 1, blocks - 1));
    gd_barrier();
#pragma unroll
    for (int a = 0; a < TW; ++a)
        if (!tg.bias) sum[a] = zero;
    int stage = 0;
    auto step = [&](auto place_c, int t) {               // t % 8 == place
        constexpr int place = decltype(place_c)::value, set = place & 1, e = place % SUMS;
        const int now = stage;
        stage = stage + 1 == NS ? 0 : stage + 1;
        if (t + 1 < blocks || (ORDER == FW_EIGHTHS && place < 7)) {
            // the next K-step has landed, and everybody's reads of this one: its memory is written next
            gd_wait_younger<T::LPW, NS - 2>(min(NS - 2, blocks - 2 - t));
            gd_wait_lds();
            gd_barrier();
            if (t + NS < blocks) fetch(now, t + NS);
            operands(std::integral_constant<int, set ^ 1>{}, stage);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int a = 0; a < TW; ++a) acc[e][u][a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[set][u][a], x[set][u], acc[e][u][a], 0, 0, 0);
    };
    operands(std::integral_constant<int, 0>{}, 0);
#pragma unroll 1
    for (int t = 0; t < blocks; t += 8)
        gd_static_for<0, 8>([&](auto place_c) {
            if (ORDER == FW_EIGHTHS || t + decltype(place_c)::value < blocks) step(place_c, t + decltype(place_c)::value);
        });
    if constexpr (ORDER == FW_EIGHTHS) {
#pragma unroll
        for (int e = 0; e < SUMS; ++e)
#pragma unroll
            for (int a = 0; a < TW; ++a) sum[a] += acc[e][0][a] + acc[e][1][a];
    } else {
#pragma unroll
        for (int a = 0; a < TW; ++a) sum[a] = (acc[0][0][a] + acc[0][1][a]) + sum[a];
    }
    // A wave's sums leave through LDS as rows (written once per value where they are computed, every activation was code TW x 4 times over).
    gd_wait_lds();
    gd_barrier();                                                       // the last K-step is in everybody's registers
    constexpr int PITCH = T::BN + 4;
    static_assert(GX * 16 * PITCH * 4 <= T::SMEM, "the sums of all waves");
    float* const rows = reinterpret_cast<float*>(fw_lds) + wave * 16 * PITCH;
#pragma unroll
    for (int a = 0; a < TW; ++a)
        *reinterpret_cast<floatx4*>(rows + col * PITCH + a * 16 + quarter * 4) = sum[a];
    at_epilogue_wave_sync();
#pragma unroll 1
    for (int i = lane; i < 16 * 4 * TW; i += KA_WAVE) {
        const int r = i / (4 * TW), c = i % (4 * TW) * 4, m = wave * 16 + r, n = n0 + c;
        if (m >= p.M || n >= N) continue;
        floatx4 s = *reinterpret_cast<const floatx4*>(rows + r * PITCH + c);
        if (ka_act_gated(tg.act)) {
            const float v[4] = {s[0], s[1], s[2], s[3]};
            ka_gated_store<true, 4>(tg.out, tg.out_dtype, tg.ldo, m, n, N, v, tg.act);
            continue;
        }
        if (tg.act) {
#pragma unroll
            for (int j = 0; j < 4; ++j) s[j] = ka_activate_fast(tg.act, s[j]);
        }
        const size_t o = (size_t)m * tg.ldo + n;
        if (tg.out_dtype == KA_F32) {
            floatx4* const at = reinterpret_cast<floatx4*>(reinterpret_cast<float*>(tg.out) + o);
            *at = tg.accumulate ? *at + s : s;
        } else {
            *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16_t*>(tg.out) + o) = bf16x4{(bf16_t)s[0], (bf16_t)s[1], (bf16_t)s[2], (bf16_t)s[3]};
        }
    }
}

template <int TW, int GX, int ORDER>
static int launch_whole(FwArgs p, hipStream_t stream) {
    using T = FwTile<TW, GX>;
    static bool configured = false;
    auto kernel = few_whole_kernel<TW, GX, ORDER>;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, T::SMEM);
        KA_CHECK(e == hipSuccess, "linear of few rows: cannot reserve %d bytes of LDS: %s", T::SMEM, hipGetErrorString(e));
        configured = true;
    }
    p.tiles_a = ka_cdiv(p.a.N, T::BN);
    const int tiles = p.tiles_a + (p.b.W ? ka_cdiv(p.b.N, T::BN) : 0);
    hipLaunchKernelGGL(kernel, dim3(ka_cdiv(tiles, 8) * 8), dim3(64 * GX), T::SMEM, stream, p);
    KA_LAUNCH_CHECK();
    return 0;
}

// The tile, in sixteens of weight rows, 0: not by these tiles. Measured against the kernels of before over 1,046 sizes of 17 to 64 rows, weights from HBM.
//  * FW_EIGHTHS (K in steps of 512 up to 2,560, against skinny_persistent_kernel): one tile a CU, of at most 80 weight rows, the registers being what they are. From
//    49 rows on, where that kernel has a strip at a time (us: 14,336 of 2,048 20.1 and 19.0, 14,336 of 2,560 28.6 and 22.6, 4,096 of 2,560 14.4 and 11.4), but more than
//    64 weight rows a CU with K of 1,537 to 2,048 (17,920: 23.7 and 25.0). Up to 48 rows from 3,072 outputs on (2,048: level; 1,024: up to 16 % behind), to
//    16,384 with K up to 1,536 (32 rows, 7,680 of 1,024: 9.1 and 7.1), else to 10,240 (7,680 of 2,048: 12.8 and 10.9; 14,336: 17.8 and 18.5; 17,920 of 2,560 23.5 and 27.8).
//  * FW_HALVES (where the kernel with parts of K has one, against few_rows_kernel and the launch that adds up): everywhere. The fewest weight rows on the busiest CU, and tiles of more
//    than 80 rows only where a CU has two of them (40 rows, 18,560 of 4,096: 48.7 and 35.7; 10,752: 28.4 and 23.0; 51,200 93.7 and 82.8; 28,672 by 7 sixteens 53.4, by 4 48.8,
//    before 53.8).
static int few_whole_tile(const FwArgs& p, int order) {
    const int cus = ka_compute_units();
    auto tiles = [&](int tw) { return (long)ka_cdiv(p.a.N, 16 * tw) + (p.b.W ? ka_cdiv(p.b.N, 16 * tw) : 0); };
    if (order == FW_EIGHTHS) {
        const long N = (long)p.a.N + (p.b.W ? p.b.N : 0);
        if (p.M > 48 ? N < 1024 || (p.K > 1536 && p.K <= 2048 && N > 64L * cus) : N < 3072 || N > (p.K <= 1536 ? 64L : 40L) * cus) return 0;
        for (int tw = 1; tw <= 5; ++tw)
            if (tiles(tw) <= cus) return tw;
        return 0;
    }
    int best = 0;
    long least = 0;
    for (int tw = 7; tw >= 3; --tw) {
        const long rows = (tiles(tw) + cus - 1) / cus * tw;
        if ((tw <= 5 || tiles(tw) > cus) && (!best || rows < least)) { best = tw; least = rows; }
    }
    return best;
}

template <int GX>
static int launch_whole_rows(const FwArgs& p, int tw, int order, hipStream_t stream) {
    switch (order * 10 + tw) {
        case 1: return launch_whole<1, GX, FW_EIGHTHS>(p, stream);
        case 2: return launch_whole<2, GX, FW_EIGHTHS>(p, stream);
        case 3: return launch_whole<3, GX, FW_EIGHTHS>(p, stream);
        case 4: return launch_whole<4, GX, FW_EIGHTHS>(p, stream);
        case 5: return launch_whole<5, GX, FW_EIGHTHS>(p, stream);
        case 13: return launch_whole<3, GX, FW_HALVES>(p, stream);
        case 14: return launch_whole<4, GX, FW_HALVES>(p, stream);
        case 15: return launch_whole<5, GX, FW_HALVES>(p, stream);
        case 16: return launch_whole<6, GX, FW_HALVES>(p, stream);
        case 17: return launch_whole<7, GX, FW_HALVES>(p, stream);
    }
    KA_CHECK(false, "linear of few rows: unknown tile %d", tw);
}

// The tile for one linear (N2 = 0) or two of M rows, in sixteens of weight rows; 0: not by these tiles.
KA_API int ka_few_rows_whole_tile(int M, int N1, int N2, int K, int halves) {
    if (M < 17 || M > 64 || N1 < 1 || N2 < 0 || K < 64 || K % (halves ? 64 : 512)) return 0;
    FwArgs p = {};
    p.M = M; p.K = K; p.a.N = N1; p.b.N = N2;
    p.b.W = N2 ? reinterpret_cast<const bf16_t*>(&p) : nullptr;          // (asked for as "there is one" alone)
    return few_whole_tile(p, halves ? FW_HALVES : FW_EIGHTHS);
}

// `halves`: the sums of the kernel with parts of K, for a K in one part; else those of the persistent kernel. 0: done; 1: not covered, nothing was run; -1: an error.
int ka_few_rows_whole(const SkinnyArgs& args, bool halves, hipStream_t stream) {
    const int K = args.K[0];
    if (args.M < 17 || args.M > 64 || K % (halves ? 64 : 512) || args.A[1] || args.ln_x || !args.A[0]) return 1;
    // (outputs and biases go by fours; others stay with the kernels of before, whose bits these are)
    for (const SkinnyTarget* t : {&args.a, &args.b})
        if (t->W && (t->N % 4 || (uintptr_t)t->bias % 16 || (!ka_act_gated(t->act) && (t->ldo % 4 || (uintptr_t)t->out % 16)))) return 1;
    FwArgs p = {};
    p.A = args.A[0]; p.lda = args.lda[0]; p.M = args.M; p.K = K; p.a = args.a; p.b = args.b;
    const int order = halves ? FW_HALVES : FW_EIGHTHS, tw = few_whole_tile(p, order);
    if (!tw) return 1;
    return (args.M <= 32 ? launch_whole_rows<2>(p, tw, order, stream) : launch_whole_rows<4>(p, tw, order, stream)) ? -1 : 0;
}
