// A block's two last linears by four waves a tile (ka_quad_tiles.h), K of both in parts.
//
// A workgroup's K-steps bound it (0.53 us for 128 x 128 with one on every CU, 0.88 for 128 x 256, 1.07 for 160 x 256: phased 128 x 256 took 1.02), then its sums on their
// way out and back (4 bytes each, 1.3 us a million). Which tile and how many parts: pair_tiles_choice (gemm_bf16.hip), with both sides' times.
#include "ka_quad_tiles.h"
#include "ka_partials.h"

// out += A[0] W[0]^T + A[1] W[1]^T: the K-steps of both one behind the other and cut into parts of `per`, whose fp32 sums go out as [M, N] of their own
// for the kernel that finishes the rows.
template <int TW, int TX, int NS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
pair_quad_kernel(KaPairTiles p) {
    using T = KqTile<TW, TX, NS>;
    extern __shared__ __attribute__((aligned(16))) unsigned char kq_lds[];
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
    unsigned woff[2][T::WL], xoff[2][T::XL];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int i = 0; i < T::WL; ++i) {
            const int r = T::w_row(i, wave, lane);
            woff[s][i] = (unsigned)(min(n0 + r, p.N - 1) * p.ldw[s] + kd_load_channel<8>(r, lane)) * 2u;
        }
#pragma unroll
        for (int i = 0; i < T::XL; ++i) {
            const int r = T::x_row(i, wave, lane);
            xoff[s][i] = (unsigned)(min(m0 + r, p.M - 1) * p.lda[s] + kd_load_channel<8>(r, lane)) * 2u;
        }
    }
    floatx4 acc[TW][TX];
#pragma unroll
    for (int a = 0; a < TW; ++a)
#pragma unroll
        for (int b = 0; b < TX; ++b) acc[a][b] = floatx4{0.f, 0.f, 0.f, 0.f};
    float* const mine = p.partial + (size_t)at.part * p.M * p.N;
    asm volatile("" ::"s"(mine), "s"(p.M), "s"(p.N));                          // (no scalar load later, on the counter of the LDS reads)
    kq_product<TW, TX, NS>(
        kq_lds, wave, lane, hi - lo, [&](int i, int t) { return t < border ? W0 + (size_t)t * 128 + woff[0][i] : W1 + (size_t)t * 128 + woff[1][i]; },
        [&](int i, int t) { return t < border ? A0 + (size_t)t * 128 + xoff[0][i] : A1 + (size_t)t * 128 + xoff[1][i]; }, acc);
    gd_barrier();                                        // the last K-step has been read by everybody
    const int n_wave = n0 + wave / 2 * T::WAVE_N, m_wave = m0 + wave % 2 * T::WAVE_M;
    kq_rows_out<float, TW, TX, NS>(
        kq_lds, wave, lane, [&](auto a, auto b) { return acc[a.value][b.value]; },
        [&](int r, int c, const unsigned char* from) {
            const int m = m_wave + r, n = n_wave + c;
            if (m < p.M && n < p.N) *reinterpret_cast<floatx4*>(mine + (size_t)m * p.N + n) = *reinterpret_cast<const floatx4*>(from);
        });
}

template <int TW, int TX, int NS>
static int launch_pair_quad(KaPairTiles p, int parts, hipStream_t stream) {
    using T = KqTile<TW, TX, NS>;
    static bool configured = false;
    auto kernel = pair_quad_kernel<TW, TX, NS>;
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
    hipLaunchKernelGGL(kernel, dim3((unsigned)launched), dim3(256), T::SMEM, stream, p);
    KA_LAUNCH_CHECK();
    return 0;
}

// tile: 128 x 256 (W x A rows) 3, 160 x 128 5, 128 x 128 8, 160 x 192 10, 160 x 256 12. (The operands have been checked by ka_pair_phased.)
int ka_pair_quad(const KaPairTiles& p, int tile, int parts, hipStream_t stream) {
    switch (tile) {
        case 8: return launch_pair_quad<4, 4, 4>(p, parts, stream);
        case 5: return launch_pair_quad<5, 4, 4>(p, parts, stream);
        case 10: return launch_pair_quad<5, 6, 3>(p, parts, stream);
        case 3: return launch_pair_quad<4, 8, 3>(p, parts, stream);
        case 12: return launch_pair_quad<5, 8, 3>(p, parts, stream);
    }
    KA_CHECK(false, "pair of linears: unknown tile %d", tile);
}
