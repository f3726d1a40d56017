// Linears of prompts on the phased tiles (ka_phased_tiles.h): a block's two last linears with K of both in parts.
#include "ka_common.h"
#include "ka_partials.h"
#include "ka_phased_tiles.h"

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

// tile: 256 x 256 (W x A rows) 1, 128 x 256 3, 256 x 128 5. Every part needs two K-steps.
int ka_pair_phased(const KaPairTiles& p, int tile, int parts, hipStream_t stream) {
    const int steps = p.steps[0] + p.steps[1];
    KA_CHECK(parts >= 1 && p.per >= 2 && (parts - 1) * p.per < steps && parts * p.per >= steps && steps - (parts - 1) * p.per >= 2,
             "pair of linears: %d parts of %d K-steps, %d in all", parts, p.per, steps);
    for (int s = 0; s < 2; ++s)
        KA_CHECK((p.M - 1) * p.lda[s] + p.steps[s] * 64L < (1L << 31) && (p.N - 1) * p.ldw[s] + p.steps[s] * 64L < (1L << 31), "pair of linears: an operand of 4 GB");
    switch (tile) {
        case 1: return launch_pair<4, 4, 2, 2, 2, 4>(p, parts, stream);
        case 3: return launch_pair<2, 2, 2, 2, 2, 4>(p, parts, stream);
        case 5: return launch_pair<2, 2, 2, 2, 4, 2>(p, parts, stream);
    }
    KA_CHECK(false, "pair of linears: unknown tile %d", tile);
}
