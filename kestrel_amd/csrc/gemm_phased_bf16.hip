// Linears of prompts on the phased tiles (ka_phased_tiles.h): the first linears of a block whose branches read the same rows, in one
// launch, and a block's two last linears with K of both in parts.
#include "ka_common.h"
#include "ka_partials.h"
#include "ka_phased_tiles.h"
#include "ka_quad_tiles.h"

// out[s] = act[s](A W[s]^T + bias[s]), s = 0, 1, in bf16; the tiles of the second linear follow those of the first.
struct KpJoint {
    const bf16_t* A;        // [M, K]
    long lda;
    int M, K, tiles_m, tiles_n[2];
    const bf16_t* W[2];     // [N[s], K]
    const float* bias[2];   // may be null
    bf16_t* out[2];         // [M, N[s]]
    long ldw[2], ldo[2];
    int N[2], act[2];
};

template <int QW0, int QW1, int QX0, int QX1, int GW, int GX>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
joint_tiles_kernel(KpJoint p) {
    using T = KpTile<QW0, QW1, QX0, QX1, GW, GX>;
    extern __shared__ __attribute__((aligned(16))) unsigned char kp_lds[];
    const int total = (p.tiles_n[0] + p.tiles_n[1]) * p.tiles_m, per_xcd = (total + 7) / 8;
    const int logical = blockIdx.x % 8 * per_xcd + blockIdx.x / 8;      // an XCD's tiles: neighbours in N, whose rows of W they share
    if (logical >= total) return;
    const int m0 = logical % p.tiles_m * T::BM, tile = logical / p.tiles_m;
    const bool second = tile >= p.tiles_n[0];
    const int n0 = (second ? tile - p.tiles_n[0] : tile) * T::BN;
    const char* const W = (const char*)(second ? p.W[1] : p.W[0]);
    const long ldw = second ? p.ldw[1] : p.ldw[0], ldo = second ? p.ldo[1] : p.ldo[0];
    const int N = second ? p.N[1] : p.N[0], act = second ? p.act[1] : p.act[0];
    const float* const bias = second ? p.bias[1] : p.bias[0];
    bf16_t* const out = second ? p.out[1] : p.out[0];
    const char* const A = (const char*)p.A;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KA_WAVE), lane = threadIdx.x % KA_WAVE;
    // (bytes from the operand's start, which the host has checked to fit in 32 bits; rows past the end are read from the last row, and never stored)
    unsigned woff[T::LW0 + T::LW1], xoff[T::LX0 + T::LX1];
#pragma unroll
    for (int i = 0; i < T::LW0 + T::LW1; ++i)
        woff[i] = (unsigned)(min(n0 + T::w_row(i, wave, lane), N - 1) * ldw + T::w_channel(i, wave, lane)) * 2u;
#pragma unroll
    for (int i = 0; i < T::LX0 + T::LX1; ++i)
        xoff[i] = (unsigned)(min(m0 + T::x_row(i, wave, lane), p.M - 1) * p.lda + T::x_channel(i, wave, lane)) * 2u;
    floatx4 acc[2][2][T::QW][T::QX];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int a = 0; a < T::QW; ++a)
#pragma unroll
                for (int b = 0; b < T::QX; ++b) acc[h][g][a][b] = floatx4{0.f, 0.f, 0.f, 0.f};
    asm volatile("" ::"s"(bias), "s"(out), "s"(ldo), "s"(act), "s"(p.M), "s"(N));       // (no scalar load later, on the counter of the LDS reads)
    kp_product<QW0, QW1, QX0, QX1, GW, GX>(kp_lds, wave, lane, p.K / 64, [&](int i, int t) { return W + (size_t)t * 128 + woff[i]; },
                                           [&](int i, int t) { return A + (size_t)t * 128 + xoff[i]; }, acc);
    gd_barrier();                                        // the last K-step has been read by everybody
    const int n_wave = n0 + wave / GX * T::WAVE_N, m_wave = m0 + wave % GX * T::WAVE_M, quarter = lane / 16;
    // (N is a multiple of 8: four columns of a tile are inside it or past it together, and so are the eight of a store)
    floatx4 add[2][T::QW];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int a = 0; a < (h ? QW1 : QW0); ++a) {
            const int n = n_wave + (h * QW0 + a) * 16 + quarter * 4;
            add[h][a] = bias && n < N ? *reinterpret_cast<const floatx4*>(bias + n) : floatx4{0.f, 0.f, 0.f, 0.f};
        }
    auto rows_out = [&](auto activate) {
        kp_rows_out<bf16_t, QW0, QW1, QX0, QX1, GW, GX>(
            kp_lds, wave, lane,
            [&](auto h, auto g, auto a, auto b) {
                floatx4 v = acc[h.value][g.value][a.value][b.value] + add[h.value][a.value];
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = activate(v[i]);
                return v;
            },
            [&](int r, int c, const unsigned char* from) {
                const int m = m_wave + r, n = n_wave + c;
                if (m < p.M && n < N) *reinterpret_cast<bf16x8*>(out + (size_t)m * ldo + n) = *reinterpret_cast<const bf16x8*>(from);
            });
    };
    // (the two activations that matter have an epilogue of their own: chosen per value, an activation costs a branch a value)
    if (act == KA_ACT_NONE) rows_out([](float x) { return x; });
    else if (act == KA_ACT_GELU_TANH) rows_out([](float x) { return ka_gelu_tanh_fast(x); });
    else rows_out([&](float x) { return ka_activate_fast(act, x); });
}

template <int QW0, int QW1, int QX0, int QX1, int GW, int GX>
static int launch_joint(KpJoint p, hipStream_t stream) {
    using T = KpTile<QW0, QW1, QX0, QX1, GW, GX>;
    static bool configured = false;
    auto kernel = joint_tiles_kernel<QW0, QW1, QX0, QX1, GW, GX>;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, T::SMEM);
        KA_CHECK(e == hipSuccess, "joint linears: cannot reserve %d bytes of LDS: %s", T::SMEM, hipGetErrorString(e));
        configured = true;
    }
    p.tiles_m = ka_cdiv(p.M, T::BM);
    for (int s = 0; s < 2; ++s) p.tiles_n[s] = ka_cdiv(p.N[s], T::BN);
    const long total = ((long)(p.tiles_n[0] + p.tiles_n[1]) * p.tiles_m + 7) / 8 * 8;
    KA_CHECK(total < (1L << 31), "joint linears: too many tiles");
    hipLaunchKernelGGL(kernel, dim3((unsigned)total), dim3(512), T::SMEM, stream, p);
    KA_LAUNCH_CHECK();
    return 0;
}

// The tile for two linears of the same rows in one launch, 0: not covered, or left to the vendor library one after the other. Of the tiles whose workgroups are one round of the chip
// the smallest wins, since a K-step of it is the shortest: four waves a tile up to 160 x 256 (ka_quad_tiles.h), above that the phased ones.
// Measured, us, the library's two launches, the phased tiles (128 x 128, 128 x 256, 192 x 256) that ran here before, and these; 14,336 from 2,048: 96 rows 31.7, 23.1, 18.6; 256 rows 50,
// 26, 25.8; 384 rows 49, 31.5, 30.0; 512 rows 51, 34, 33.6; 17,920 from 2,560: 96 rows 43, 32.5, 30.4; 256 rows 70, 45, 37.8; 512 rows 71, 54, 47.3. Over widths of 768 to 4,096 and 65 to
// 1,024 rows the tile chosen is the fastest but in three cases of 98 (4 % behind), and one launch 1.2 to 2.6 times as fast as the library's two. That is not so where nearly half of a
// large tile is no rows (22,528 from 4,096, 257 rows: 85 us in one launch, 82 by the library), and where the tiles take more than one round, in which neither
// side is ahead everywhere (library and the best of the tiles 256 x 256, 192 x 256 and 128 x 256; 14,336 from 2,048: 1,100 rows 74 and 84, 1,300 rows 90
// and 86, 1,536 rows 88 and 89, 2,048 rows 104 and 106; 17,920 from 2,560: 1,024 rows 105 and 106, 1,200 rows 128 and 109, 1,536 rows 125 and 127, 1,792 rows
// 162 and 131): a rule for those rows would go by the fill of the last round, and has not been measured at other widths.
static const struct { int code, rows_w, rows_x; } KP_JOINT_TILES[] = {{6, 64, 128}, {7, 96, 128}, {8, 128, 128}, {5, 160, 128}, {3, 128, 192}, {9, 96, 256}, {10, 160, 192},
                                                                      {11, 128, 256}, {12, 160, 256}, {2, 192, 256}, {4, 256, 192}, {1, 256, 256}};
static bool kp_phased(int code) { return code == 1 || code == 2 || code == 4; }

KA_API int ka_linear_joint_tile(int M, int N1, int N2, int K) {
    if (M < 1 || N1 < 8 || N2 < 8 || N1 % 8 || N2 % 8 || K % 64 || K < 128) return 0;
    for (const auto& t : KP_JOINT_TILES)
        if ((long)ka_cdiv(M, t.rows_x) * (ka_cdiv(N1, t.rows_w) + ka_cdiv(N2, t.rows_w)) <= ka_compute_units())
            return !kp_phased(t.code) || M * 20 >= ka_cdiv(M, t.rows_x) * t.rows_x * 11 ? t.code : 0;
    return 0;
}

// The tile for one linear of more rows than the weight-streaming kernels take, 0: left to the vendor library. The smallest whose workgroups are one round, as above, if they are enough:
// with K up to 1,024 a sixth of the CUs (and 1,024 outputs); up to 2,304 five eighths, below which the library cuts K (us, library and tile: 2,048 of 2,048, 448 rows, 112
// workgroups 12.1 and 12.1; 1,024 of 2,048, 768 rows, 96 workgroups 11.3 and 11.9); up to 4,608 seven eighths, or two thirds of the smallest tile, whose stages run furthest ahead (4,096 of
// 4,096, 768 rows, 192 of 128 x 128 33.9 and 38.5; 2,048 of 4,096, 768 rows, 192 of 64 x 128 23.4 and 21.3). Over 976 sizes (512 to 12,416 outputs, K of 512 to 8,192, 80 to 2,048
// rows, bf16 and fp32 out, weights from HBM) what this takes is 19 % faster on the average, up to 1.7 times (5,632 of 704, 256 rows 13.1 and 7.6), and 4 % behind at most (6,144 of 704, 1,024
// rows into fp32, 14.4 and 15.0): 2,048 of 2,048, 2,048 rows 21.4 and 18.8; 4,096 of 2,048 31.5 and 29.7; 5,632 of 2,048, 512 rows 24.3 and 17.6. Longer K and more than a round: the library.
KA_API int ka_linear_quad_tile(int M, int N, int K) {
    if (M < 1 || N < 8 || N % 8 || K < 64 || K % 64) return 0;
    const long cus = ka_compute_units();
    for (const auto& t : KP_JOINT_TILES) {
        if (kp_phased(t.code)) break;
        const long tiles = (long)ka_cdiv(M, t.rows_x) * ka_cdiv(N, t.rows_w);
        if (tiles > cus) continue;
        if (K <= 1024) return tiles * 6 >= cus && N >= 1024 ? t.code : 0;
        if (K <= 2304) return tiles * 8 >= cus * 5 ? t.code : 0;
        return K <= 4608 && (tiles * 8 >= cus * 7 || (t.code == 6 && tiles * 3 >= cus * 2)) ? t.code : 0;
    }
    return 0;
}

// One linear by the tiles of four waves into bf16 or fp32.
KA_API int ka_linear_quad_bf16(const void* A, long lda, const void* W, long ldw, const float* bias, void* out, int out_dtype, long ldo, int M, int N, int K, int act,
                               int accumulate, int code, hipStream_t stream) {
    const char* who = "ka_linear_quad_bf16";
    KA_CHECK(M > 0 && K >= 64 && K % 64 == 0 && N > 0 && N % 8 == 0, "%s: M=%d K=%d N=%d", who, M, K, N);
    KA_CHECK(lda >= K && ldw >= K && lda % 8 == 0 && ldw % 8 == 0 && ldo >= N && ldo % 8 == 0, "%s: strides", who);
    KA_CHECK(((uintptr_t)A | (uintptr_t)W | (uintptr_t)bias | (uintptr_t)out) % 16 == 0, "%s: operands must be 16-byte aligned", who);
    KA_CHECK((M - 1) * lda + K < (1L << 31) && (N - 1) * ldw + K < (1L << 31), "%s: an operand of 4 GB", who);
    KA_CHECK(ka_act_known(act) && !ka_act_gated(act) && (out_dtype == KA_F32 || out_dtype == KA_BF16) && !(accumulate && out_dtype != KA_F32), "%s: activation %d, output %d", who, act, out_dtype);
    KqLinears q = {};
    q.A = (const bf16_t*)A; q.lda = lda; q.M = M; q.K = K; q.accumulate = accumulate;
    q.W[0] = (const bf16_t*)W; q.ldw[0] = ldw; q.bias[0] = bias; q.out[0] = out; q.ldo[0] = ldo; q.N[0] = N; q.act[0] = act;
    return out_dtype == KA_F32 ? ka_quad_f32(q, code, stream) : ka_quad_bf16(q, code, stream);
}

KA_API int ka_linear_joint_bf16(const void* A, long lda, int M, int K, const void* W1, long ldw1, const float* bias1, void* out1, long ldo1, int N1,
                                int act1, const void* W2, long ldw2, const float* bias2, void* out2, long ldo2, int N2, int act2, int config,
                                hipStream_t stream) {
    const char* who = "ka_linear_joint_bf16";
    KA_CHECK(M > 0 && K >= 128 && K % 64 == 0 && N1 > 0 && N1 % 8 == 0 && N2 > 0 && N2 % 8 == 0, "%s: M=%d K=%d N=%d and %d", who, M, K, N1, N2);
    KA_CHECK(lda >= K && ldw1 >= K && lda % 8 == 0 && ldw1 % 8 == 0 && ldo1 >= N1 && ldo1 % 8 == 0, "%s: strides", who);
    KA_CHECK(ldw2 >= K && ldw2 % 8 == 0 && ldo2 >= N2 && ldo2 % 8 == 0, "%s: strides of the second linear", who);
    KA_CHECK(((uintptr_t)A | (uintptr_t)W1 | (uintptr_t)W2 | (uintptr_t)bias1 | (uintptr_t)bias2 | (uintptr_t)out1 | (uintptr_t)out2) % 16 == 0,
             "%s: operands must be 16-byte aligned", who);
    KA_CHECK((M - 1) * lda + K < (1L << 31) && (N1 - 1) * ldw1 + K < (1L << 31) && (N2 - 1) * ldw2 + K < (1L << 31), "%s: an operand of 4 GB", who);
    KA_CHECK(ka_act_known(act1) && ka_act_known(act2) && !ka_act_gated(act1) && !ka_act_gated(act2), "%s: activations %d and %d", who, act1, act2);
    KpJoint p = {};
    p.A = (const bf16_t*)A; p.lda = lda; p.M = M; p.K = K;
    p.W[0] = (const bf16_t*)W1; p.bias[0] = bias1; p.out[0] = (bf16_t*)out1; p.ldw[0] = ldw1; p.ldo[0] = ldo1; p.N[0] = N1; p.act[0] = act1;
    p.W[1] = (const bf16_t*)W2; p.bias[1] = bias2; p.out[1] = (bf16_t*)out2; p.ldw[1] = ldw2; p.ldo[1] = ldo2; p.N[1] = N2; p.act[1] = act2;
    switch (config) {
        case 1: return launch_joint<4, 4, 2, 2, 2, 4>(p, stream);
        case 2: return launch_joint<4, 2, 2, 2, 2, 4>(p, stream);
        case 4: return launch_joint<4, 4, 2, 1, 2, 4>(p, stream);
    }
    KqLinears q = {};
    q.A = p.A; q.lda = p.lda; q.M = p.M; q.K = p.K;
    for (int i = 0; i < 2; ++i) {
        q.W[i] = p.W[i]; q.ldw[i] = p.ldw[i]; q.bias[i] = p.bias[i]; q.out[i] = p.out[i]; q.ldo[i] = p.ldo[i]; q.N[i] = p.N[i]; q.act[i] = p.act[i];
    }
    return ka_quad_bf16(q, config, stream);
}

// A block's two last linears: out += A[0] W[0]^T + A[1] W[1]^T, the K-steps of both one behind the other and cut into parts of `per`,
// whose fp32 sums go out as [M, N] of their own for the kernel that finishes the rows.
template <int QW0, int QW1, int QX0, int QX1, int GW, int GX>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
pair_phased_kernel(KaPairTiles p) {
    using T = KpTile<QW0, QW1, QX0, QX1, GW, GX>;
    extern __shared__ __attribute__((aligned(16))) unsigned char kp_lds[];
    const KaPairPlace at = ka_pair_place(p, blockIdx.x);
    if (at.part < 0) return;
    const int m0 = at.tile_m * T::BM, n0 = at.tile_n * T::BN;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KA_WAVE), lane = threadIdx.x % KA_WAVE;
    const int lo = at.part * p.per, hi = min(lo + p.per, p.steps[0] + p.steps[1]), border = p.steps[0] - lo;
    // this part's first K-step of either linear: address(t) is of linear 0 while t < border
    const char* const A0 = (const char*)p.A[0] + (size_t)lo * 128;
    const char* const W0 = (const char*)p.W[0] + (size_t)lo * 128;
    const char* const A1 = (const char*)p.A[1] - (ptrdiff_t)border * 128;
    const char* const W1 = (const char*)p.W[1] - (ptrdiff_t)border * 128;
    unsigned woff[2][T::LW0 + T::LW1], xoff[2][T::LX0 + T::LX1];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int i = 0; i < T::LW0 + T::LW1; ++i)
            woff[s][i] = (unsigned)(min(n0 + T::w_row(i, wave, lane), p.N - 1) * p.ldw[s] + T::w_channel(i, wave, lane)) * 2u;
#pragma unroll
        for (int i = 0; i < T::LX0 + T::LX1; ++i)
            xoff[s][i] = (unsigned)(min(m0 + T::x_row(i, wave, lane), p.M - 1) * p.lda[s] + T::x_channel(i, wave, lane)) * 2u;
    }
    floatx4 acc[2][2][T::QW][T::QX];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int a = 0; a < T::QW; ++a)
#pragma unroll
                for (int b = 0; b < T::QX; ++b) acc[h][g][a][b] = floatx4{0.f, 0.f, 0.f, 0.f};
    float* const mine = p.partial + (size_t)at.part * p.M * p.N;
    asm volatile("" ::"s"(mine), "s"(p.M), "s"(p.N));
    kp_product<QW0, QW1, QX0, QX1, GW, GX>(
        kp_lds, wave, lane, hi - lo, [&](int i, int t) { return t < border ? W0 + (size_t)t * 128 + woff[0][i] : W1 + (size_t)t * 128 + woff[1][i]; },
        [&](int i, int t) { return t < border ? A0 + (size_t)t * 128 + xoff[0][i] : A1 + (size_t)t * 128 + xoff[1][i]; }, acc);
    gd_barrier();
    const int n_wave = n0 + wave / GX * T::WAVE_N, m_wave = m0 + wave % GX * T::WAVE_M;
    kp_rows_out<float, QW0, QW1, QX0, QX1, GW, GX>(
        kp_lds, wave, lane, [&](auto h, auto g, auto a, auto b) { return acc[h.value][g.value][a.value][b.value]; },
        [&](int r, int c, const unsigned char* from) {
            const int m = m_wave + r, n = n_wave + c;
            if (m < p.M && n < p.N) *reinterpret_cast<floatx4*>(mine + (size_t)m * p.N + n) = *reinterpret_cast<const floatx4*>(from);
        });
}

template <int QW0, int QW1, int QX0, int QX1, int GW, int GX>
static int launch_pair(KaPairTiles p, int parts, hipStream_t stream) {
    using T = KpTile<QW0, QW1, QX0, QX1, GW, GX>;
    static bool configured = false;
    auto kernel = pair_phased_kernel<QW0, QW1, QX0, QX1, GW, GX>;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, T::SMEM);
        KA_CHECK(e == hipSuccess, "pair of linears: cannot reserve %d bytes of LDS: %s", T::SMEM, hipGetErrorString(e));
        configured = true;
    }
    p.tiles_m = ka_cdiv(p.M, T::BM);
    p.tiles_n = ka_cdiv(p.N, T::BN);
    p.parts = parts;
    const long launched = ((long)p.tiles_n * p.tiles_m * parts + 7) / 8 * 8;
    KA_CHECK(launched < (1L << 31), "pair of linears: too many tiles");
    hipLaunchKernelGGL(kernel, dim3((unsigned)launched), dim3(512), T::SMEM, stream, p);
    KA_LAUNCH_CHECK();
    return 0;
}

// tile: 256 x 256 (W x A rows) 1, those of ka_pair_quad. Every part needs two K-steps.
int ka_pair_phased(const KaPairTiles& p, int tile, int parts, hipStream_t stream) {
    const int steps = p.steps[0] + p.steps[1];
    KA_CHECK(parts >= 1 && p.per >= 2 && (parts - 1) * p.per < steps && parts * p.per >= steps && steps - (parts - 1) * p.per >= 2,
             "pair of linears: %d parts of %d K-steps, %d in all", parts, p.per, steps);
    for (int s = 0; s < 2; ++s)
        KA_CHECK((p.M - 1) * p.lda[s] + p.steps[s] * 64L < (1L << 31) && (p.N - 1) * p.ldw[s] + p.steps[s] * 64L < (1L << 31), "pair of linears: an operand of 4 GB");
    return tile == 1 ? launch_pair<4, 4, 2, 2, 2, 4>(p, parts, stream) : ka_pair_quad(p, tile, parts, stream);
}
