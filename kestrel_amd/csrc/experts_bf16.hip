// The linears of routed experts on the matrix cores (bf16): the pairs (token, choice) of a step come listed by expert, in
// runs that start on multiples of a tile's rows (ka_experts_sort, ka_experts_gemm_tile), and a workgroup multiplies one
// tile of list rows by 256 rows of its expert's weights: out[row] = act(a[row'] W_e^T).
//
//  * the first linear gathers: list row i holds pair p = sorted[i] (-1: an unused row), whose input is row p / gather_div
//    of `a`; its output goes to row i of `out` (the hidden rows stay in list order);
//  * the second linear scatters: its input is row i of `a`, its output goes to row p of `out`;
//  * gated (KA_ACT_GATED): weight rows 2j and 2j + 1 are gate and value of output j, as in every gated linear here, with or
//    without clamps (KaGateClamp).
//
// The weights are the row operand: a lane ends with outputs of ONE list row, four neighbours at a time, so the pair of a
// gated output meets in a lane's registers.
//
// First the kernel for a K in no steps of 64, tiles of KL_ROWS staged through registers (ka_listed_tiles.h).
#include "ka_common.h"
#include "ka_dma_tiles.h"
#include "ka_listed_tiles.h"

#include <math.h>

#include <utility>

typedef __attribute__((ext_vector_type(2))) __bf16 eb_bf16x2;

constexpr int EF_MAX_PAIRS = 512;          // most pairs of a step of few

__global__ void __launch_bounds__(256)
experts_gemm_kernel(const bf16_t* __restrict__ a, long lda, int gather_div, const bf16_t* __restrict__ W, const int* __restrict__ sorted,
                    const int* __restrict__ tile_expert, int N, int K, int act, KaGateClamp clamp, void* __restrict__ out, long ldo,
                    int scatter, int out_f32) {
    extern __shared__ __attribute__((aligned(16))) bf16_t eb_lds[];
    const int tile = blockIdx.y;
    const int e = tile_expert[tile];
    if (e < 0) return;                                   // (the unused end of the list: the whole workgroup)
    const int wave = threadIdx.x / KA_WAVE, lane = threadIdx.x % KA_WAVE;
    const int col = lane % 32, half = lane / 32;
    const int o0 = blockIdx.x * KL_COLS + wave * 64;
    const int i0 = tile * KL_ROWS;
    int pr[4];
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) pr[rb] = sorted[i0 + rb * 32 + col];
    // rows past the end, and unused rows of the list, are clamped for the loads and not stored
    auto list_row = [&](int r) { return a + (gather_div > 0 ? (long)max(sorted[i0 + r], 0) / gather_div : (long)i0 + r) * lda; };
    auto weight_row = [&](int r) { return W + ((size_t)e * N + min((int)blockIdx.x * KL_COLS + r, N - 1)) * K; };
    kl_floatx16 acc[2][4];
    const bool swap[2] = {false, false};
    kl_tile_product<true, false>(eb_lds, K, o0 < N, swap, list_row, weight_row, acc);
    if (o0 >= N) return;
    const bool gated = ka_act_gated(act);
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
        const int p = pr[rb];
        if (p < 0) continue;
        const long row = scatter ? (long)p : (long)i0 + rb * 32 + col;
#pragma unroll
        for (int wb = 0; wb < 2; ++wb) {
            const kl_floatx16& acc_here = acc[wb][rb];
            // register i: weight row o0 + 32 wb + (i / 4) * 8 + half * 4 + i % 4 of the lane's list row
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const int o = o0 + wb * 32 + g4 * 8 + half * 4;
                if (gated) {
                    if (o + 3 < N) {
                        eb_bf16x2 y;
                        y[0] = (bf16_t)ka_gate_product<true>(act, clamp, acc_here[g4 * 4], acc_here[g4 * 4 + 1]);
                        y[1] = (bf16_t)ka_gate_product<true>(act, clamp, acc_here[g4 * 4 + 2], acc_here[g4 * 4 + 3]);
                        *reinterpret_cast<eb_bf16x2*>(reinterpret_cast<bf16_t*>(out) + row * ldo + o / 2) = y;
                    } else if (o + 1 < N) {
                        reinterpret_cast<bf16_t*>(out)[row * ldo + o / 2] = (bf16_t)ka_gate_product<true>(act, clamp, acc_here[g4 * 4], acc_here[g4 * 4 + 1]);
                    }
                } else if (out_f32) {
                    float* op = reinterpret_cast<float*>(out) + row * ldo + o;
                    if (o + 3 < N) {
                        *reinterpret_cast<float4*>(op) = make_float4(acc_here[g4 * 4], acc_here[g4 * 4 + 1], acc_here[g4 * 4 + 2], acc_here[g4 * 4 + 3]);
                    } else {
#pragma unroll
                        for (int x = 0; x < 4; ++x)
                            if (o + x < N) op[x] = acc_here[g4 * 4 + x];
                    }
                } else {
                    bf16_t* op = reinterpret_cast<bf16_t*>(out) + row * ldo + o;
                    kl_bf16x4 y;
#pragma unroll
                    for (int x = 0; x < 4; ++x) y[x] = (bf16_t)(ka_act_base(act) ? ka_activate_fast(act, acc_here[g4 * 4 + x]) : acc_here[g4 * 4 + x]);
                    if (o + 3 < N && ldo % 4 == 0) {
                        *reinterpret_cast<kl_bf16x4*>(op) = y;
                    } else {
#pragma unroll
                        for (int x = 0; x < 4; ++x)
                            if (o + x < N) op[x] = y[x];
                    }
                }
            }
        }
    }
}

// ----------------------------------------------------------------------------
// The same linears where K is a multiple of 64: operands go from memory straight into LDS (ka_dma_tiles.h), the list's rows
// gathered by the addresses of the loads. Eight waves and 256 weight rows a workgroup; a tile has 64, 128 or 256 list rows, as
// many as the list was made for (32: experts_dma_few_kernel).
//
// What bounds it: an expert sees a few hundred rows of a step, so its weights come from HBM for little more work than they cost
// to read (62 experts of 2 x 896 x 4,096 at 198 rows each: 910 MB and 180 GFLOP, 160 us of either). The tiles that share an
// expert therefore run side by side on one XCD (workgroups go to the XCDs in turn; each XCD gets one stretch of the list, all
// columns of a list tile before the next), so that its L2 passes weights between list tiles and rows between column
// tiles. For that the used part of the list has to be known, or the XCD with its unused end would idle: every workgroup counts
// the tiles that have an expert, in one read of the list of tiles.
//
// A sum's channels meet in the order of the kernel above, so a pair's numbers are the same bits in tiles of any size and in
// either kernel.
//
// Measured, us of the gated first and the fp32 second linear, before (the kernel above, which staged through registers, one wave
// a SIMD, with sums that went through scratch memory) -> now: 62 experts of 4,096 x 896, 2,048 tokens of 6 choices 542 + 372 ->
// 261 + 187; 512 tokens 302 + 175 -> 163 + 114; 30 experts of 2,048 x 704, 2,048 tokens of 4 choices 147 + 119 -> 81 + 60.
// ----------------------------------------------------------------------------
struct ExpertsDmaArgs {
    const bf16_t* a;
    long lda;
    int gather_div;             // as above
    const bf16_t* W;
    const int* sorted;
    const int* tile_expert;
    int n_tiles, tiles_n, N, K, act;
    KaGateClamp clamp;
    void* out;
    long ldo;
    int scatter;
};

// The workgroup's tile of the list and of the columns (of g.tiles_n); false: it has none.
__device__ __forceinline__ bool experts_dma_find(const ExpertsDmaArgs& g, int& tile, int& column) {
    int used = 0;
    for (int t0 = 0; t0 < g.n_tiles; t0 += blockDim.x) {
        const int t = t0 + (int)threadIdx.x;
        used += __syncthreads_count(t < g.n_tiles && g.tile_expert[min(t, g.n_tiles - 1)] >= 0);
    }
    const int total = used * g.tiles_n, per_xcd = (total + 7) / 8;
    const int at = blockIdx.x / 8, logical = blockIdx.x % 8 * per_xcd + at;
    if (at >= per_xcd || logical >= total) return false;
    tile = logical / g.tiles_n;
    column = logical - tile * g.tiles_n;
    return true;
}

// This lane's address of load i of the tile's list rows, and of its weight rows, at K-step 0 (kd_product).
template <typename T>
__device__ __forceinline__ const bf16_t* experts_dma_row(const ExpertsDmaArgs& g, int i0, int wave, int lane, int i) {
    const int r = kd_load_row<T::CPR>(wave * T::X_LOADS + i, lane);
    const long row = g.gather_div > 0 ? (long)(max(g.sorted[i0 + r], 0) / g.gather_div) : (long)i0 + r;
    return g.a + row * g.lda + kd_load_channel<T::CPR>(r, lane);
}
template <typename T>
__device__ __forceinline__ const bf16_t* experts_dma_weight(const ExpertsDmaArgs& g, int e, int n0, int wave, int lane, int i) {
    const int r = kd_load_row<T::CPR>(wave * T::W_LOADS + i, lane);
    return g.W + ((size_t)e * g.N + min(n0 + r, g.N - 1)) * g.K + kd_load_channel<T::CPR>(r, lane);
}

template <int WN, int WM, int GN, int GM, int NS, int SL, bool GATED, bool F32>
__global__ void __launch_bounds__(KA_WAVE * GN * GM)
    __attribute__((amdgpu_waves_per_eu(GN * GM / 4, (WN * WM > 8 ? 1 : 2) * (GN * GM / 4))))
experts_dma_kernel(ExpertsDmaArgs g) {
    using T = KdTile<WN, WM, GN, GM, 64, NS>;
    constexpr int BN = T::BN, BM = T::BM;
    extern __shared__ __attribute__((aligned(16))) unsigned char eb_dma_lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KA_WAVE), lane = threadIdx.x % KA_WAVE;
    int tile, column;
    if (!experts_dma_find(g, tile, column)) return;
    const int e = g.tile_expert[tile], i0 = tile * BM, n0 = column * BN;
    const int wn = wave / GM, wm = wave % GM, li = lane % 32, lg = lane / 32;
    const bf16_t* wsrc[T::W_LOADS];
    const bf16_t* xsrc[T::X_LOADS];
#pragma unroll
    for (int i = 0; i < T::X_LOADS; ++i) xsrc[i] = experts_dma_row<T>(g, i0, wave, lane, i);
#pragma unroll
    for (int i = 0; i < T::W_LOADS; ++i) wsrc[i] = experts_dma_weight<T>(g, e, n0, wave, lane, i);
    floatx16 acc[WN][WM];
#pragma unroll
    for (int a = 0; a < WN; ++a)
#pragma unroll
        for (int b = 0; b < WM; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.f;
    // (the pairs of this wave's list rows, a row a lane: asked for where the rows are stored, each was a trip to memory that the store waited for. F32, us: 30 experts of
    // 2,048 x 704, 2,048 tokens of 4 choices 62.9 -> 57.6)
    int pairs[WM];
#pragma unroll
    for (int b = 0; b < WM; ++b) pairs[b] = g.sorted[i0 + (wm * WM + b) * 32 + li];
    kd_product<WN, WM, GN, GM, 64, NS, SL, true>(eb_dma_lds, wave, lane, g.K, wsrc, xsrc, acc);

    // A lane ends with four neighbouring weight rows of one list row, a store instruction would touch 32 rows with 8 or 16
    // bytes each: a wave passes 32 list rows at a time through its share of LDS and stores its piece of every row whole.
    using E = std::conditional_t<F32, float, bf16_t>;
    constexpr int OUTS = GATED ? 16 * WN : 32 * WN;      // outputs of a row of the wave's tile
    constexpr int RB = OUTS * (int)sizeof(E), RS = RB + (F32 ? 16 : 8), CH = RB / 16, PER = 16 / (int)sizeof(E), RPI = KA_WAVE / CH;
    static_assert(32 * RS <= T::SMEM / T::WAVES, "a wave's share of LDS does not hold 32 rows of its tile");
    const int n_out = GATED ? g.N / 2 : g.N, o_wave = (n0 + wn * 32 * WN) / (GATED ? 2 : 1);
    unsigned char* mine = eb_dma_lds + wave * (T::SMEM / T::WAVES);
    gd_barrier();                                        // the last stage has been read by everybody
    gd_static_for<0, WM>([&](auto bc) {
        constexpr int b = decltype(bc)::value;
        gd_static_for<0, WN>([&](auto ac) {
            constexpr int a = decltype(ac)::value;
            gd_static_for<0, 4>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                const floatx4 v = {acc[a][b][q * 4], acc[a][b][q * 4 + 1], acc[a][b][q * 4 + 2], acc[a][b][q * 4 + 3]};
                const int nl = a * 32 + q * 8 + lg * 4;
                if constexpr (GATED) {
                    eb_bf16x2 y;
                    y[0] = (bf16_t)ka_gate_product<true>(g.act, g.clamp, v[0], v[1]);
                    y[1] = (bf16_t)ka_gate_product<true>(g.act, g.clamp, v[2], v[3]);
                    *reinterpret_cast<eb_bf16x2*>(mine + li * RS + nl) = y;
                } else if constexpr (F32) {
                    *reinterpret_cast<floatx4*>(mine + li * RS + nl * 4) = v;
                } else {
                    bf16x4 y;
#pragma unroll
                    for (int x = 0; x < 4; ++x) y[x] = (bf16_t)ka_activate_fast(g.act, v[x]);
                    *reinterpret_cast<bf16x4*>(mine + li * RS + nl * 2) = y;
                }
            });
        });
        at_epilogue_wave_sync();
#pragma unroll
        for (int r0 = 0; r0 < 32; r0 += RPI) {
            const int rl = r0 + lane / CH, c = lane % CH, i = i0 + wm * 32 * WM + b * 32 + rl, o = o_wave + c * PER;
            const int p = __shfl(pairs[b], rl);
            if (p >= 0 && o < n_out) {
                const unsigned char* from = mine + rl * RS + c * 16;
                E* op = reinterpret_cast<E*>(g.out) + (g.scatter ? (long)p : (long)i) * g.ldo + o;
                if (o + PER <= n_out) {
                    // (the fp32 rows are more than the caches of an XCD hold, and pass by them: 62 experts of 4,096 x 896, 1,204 tokens of 6 choices 149 -> 132 us)
                    if constexpr (F32) __builtin_nontemporal_store(*reinterpret_cast<const floatx4*>(from), reinterpret_cast<floatx4*>(op));
                    else *reinterpret_cast<floatx4*>(op) = *reinterpret_cast<const floatx4*>(from);
                } else {
                    for (int x = 0; x < PER && o + x < n_out; ++x) op[x] = reinterpret_cast<const E*>(from)[x];
                }
            }
        }
        at_epilogue_wave_sync();                         // the next pass writes over what was just read
    });
}

template <int WN, int WM, int GN, int GM, int NS, int SL, bool GATED, bool F32>
static int experts_dma_launch(ExpertsDmaArgs g, hipStream_t stream) {
    using T = KdTile<WN, WM, GN, GM, 64, NS>;
    static bool configured = false;
    auto kernel = experts_dma_kernel<WN, WM, GN, GM, NS, SL, GATED, F32>;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, T::SMEM);
        KA_CHECK(e == hipSuccess, "ka_experts_gemm_bf16: cannot reserve %d bytes of LDS: %s", T::SMEM, hipGetErrorString(e));
        configured = true;
    }
    g.tiles_n = ka_cdiv(g.N, T::BN);
    const long blocks = ((long)g.n_tiles * g.tiles_n + 7) / 8 * 8;
    KA_CHECK(blocks < (1L << 31), "ka_experts_gemm_bf16: too many tiles");
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(KA_WAVE * GN * GM), T::SMEM, stream, g);
    KA_LAUNCH_CHECK();
    return 0;
}

// Lists of as few pairs as the kernel further down takes (ka_experts_few_bf16): its sums, on products of 16 x 16 by 32 channels, every
// fourth K-step into the same of four sums, so that a pair's bits do not depend on which of the two a step goes to. Tiles of EF_TILE list rows
// by 128 weight rows, four waves, two workgroups a CU: four sums of each number are 64 registers, and it is the loads in flight that count
// (the stream of the chosen experts' weights bounds it). Both linears, us, there -> here, weights from HBM: 30 experts of 2,048 x 704, 160
// pairs 69 -> 69, 256 75 -> 70, 512 96 -> 73; 62 of 4,096 x 896, 144 pairs 271 -> 252, 240 295 -> 256, 510 340 -> 261. Tiles of 64 list rows by
// eight waves: 76 to 82 and 271 to 289; by 256 weight rows 106 to 110 and 390; six stages and one workgroup a CU 73 to 80 and 266 to 277.
constexpr int EF_TILE = 32;

template <int WN, int WM, int GN, int GM, int NS>
__global__ void __launch_bounds__(KA_WAVE * GN * GM) __attribute__((amdgpu_waves_per_eu(GN * GM / 4, GN * GM / 2)))
experts_dma_few_kernel(ExpertsDmaArgs g, int out_f32) {
    using T = KdTile<WN, WM, GN, GM, 64, NS, 16>;
    extern __shared__ __attribute__((aligned(16))) unsigned char eb_dma_lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KA_WAVE), lane = threadIdx.x % KA_WAVE;
    int tile, column;
    if (!experts_dma_find(g, tile, column)) return;
    const int e = g.tile_expert[tile], i0 = tile * T::BM, n0 = column * T::BN;
    const bf16_t* wsrc[T::W_LOADS];
    const bf16_t* xsrc[T::X_LOADS];
#pragma unroll
    for (int i = 0; i < T::X_LOADS; ++i) xsrc[i] = experts_dma_row<T>(g, i0, wave, lane, i);
#pragma unroll
    for (int i = 0; i < T::W_LOADS; ++i) wsrc[i] = experts_dma_weight<T>(g, e, n0, wave, lane, i);
    floatx4 acc[KD_FOURTHS][WN][WM];
#pragma unroll
    for (int c = 0; c < KD_FOURTHS; ++c)
#pragma unroll
        for (int a = 0; a < WN; ++a)
#pragma unroll
            for (int b = 0; b < WM; ++b) acc[c][a][b] = floatx4{0.f, 0.f, 0.f, 0.f};
    kd_product_16<WN, WM, GN, GM, NS, KD_FOURTHS>(
        eb_dma_lds, wave, lane, g.K / 64, [&](int i, int st) { return wsrc[i] + st * 64; }, [&](int i, int st) { return xsrc[i] + st * 64; }, acc);
    const int wn = wave / GM, wm = wave % GM, col = lane % 16, quarter = lane / 16;
    const bool gated = ka_act_gated(g.act);
#pragma unroll
    for (int b = 0; b < WM; ++b) {
        const int i = i0 + (wm * WM + b) * 16 + col, p = g.sorted[i];
        if (p < 0) continue;
        const long at = (g.scatter ? (long)p : (long)i) * g.ldo;
#pragma unroll
        for (int a = 0; a < WN; ++a) {
            floatx4 y = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < KD_FOURTHS; ++c) y += acc[c][a][b];
            const int o = n0 + (wn * WN + a) * 16 + quarter * 4;
            if (gated) {
                bf16_t* op = reinterpret_cast<bf16_t*>(g.out) + at + o / 2;
                if (o + 1 < g.N) op[0] = (bf16_t)ka_gate_product<true>(g.act, g.clamp, y[0], y[1]);
                if (o + 3 < g.N) op[1] = (bf16_t)ka_gate_product<true>(g.act, g.clamp, y[2], y[3]);
                continue;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (o + r >= g.N) continue;
                const float v = ka_activate_fast(g.act, y[r]);
                if (out_f32) reinterpret_cast<float*>(g.out)[at + o + r] = v;
                else reinterpret_cast<bf16_t*>(g.out)[at + o + r] = (bf16_t)v;
            }
        }
    }
}

static int experts_dma_few(ExpertsDmaArgs g, int out_f32, hipStream_t stream) {
    using T = KdTile<2, 2, 4, 1, 64, 3, 16>;
    static_assert(T::BM == EF_TILE, "the list is made for it");
    static bool configured = false;
    auto kernel = experts_dma_few_kernel<2, 2, 4, 1, 3>;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, T::SMEM);
        KA_CHECK(e == hipSuccess, "ka_experts_gemm_bf16: cannot reserve %d bytes of LDS: %s", T::SMEM, hipGetErrorString(e));
        configured = true;
    }
    g.tiles_n = ka_cdiv(g.N, T::BN);
    const long blocks = ((long)g.n_tiles * g.tiles_n + 7) / 8 * 8;
    KA_CHECK(blocks < (1L << 31), "ka_experts_gemm_bf16: too many tiles");
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(KA_WAVE * T::WAVES), T::SMEM, stream, g, out_f32);
    KA_LAUNCH_CHECK();
    return 0;
}

template <int WN, int WM, int GN, int GM, int NS, int SL>
static int experts_dma(const ExpertsDmaArgs& g, int out_f32, hipStream_t stream) {
    if (ka_act_gated(g.act)) return experts_dma_launch<WN, WM, GN, GM, NS, SL, true, false>(g, stream);
    if (out_f32) return experts_dma_launch<WN, WM, GN, GM, NS, SL, false, true>(g, stream);
    return experts_dma_launch<WN, WM, GN, GM, NS, SL, false, false>(g, stream);
}

// Whether the kernels cover these sizes and this alignment.
KA_API int ka_experts_gemm_supported(long lda, int N, int K, long ldo, int act, int out_f32) {
    const int n_out = ka_act_outputs(act, N);
    return K > 0 && K % 16 == 0 && lda % 8 == 0 && N > 0 && (!ka_act_gated(act) || (N % 4 == 0 && ldo % 2 == 0 && !out_f32)) &&
           (!out_f32 || ldo % 4 == 0) && ldo >= n_out ? 1 : 0;
}

static bool experts_dma_covers(int N, int K, long ldo, int act, int out_f32) {
    return K % 64 == 0 && ldo * (out_f32 ? 4 : 2) % 16 == 0 && !(out_f32 && act) && (!ka_act_gated(act) || N % 4 == 0);
}

// List rows of a tile for `n_pairs` pairs of `E` experts whose linears have N1 x K1 and N2 x K2 weights (the second K is the
// first's output): the list has to be made for it. The kernel that stages through registers has tiles of KL_ROWS; for the other
// one the choice goes by the rows an expert can expect, with a quarter on top for routers that do not spread evenly:
//  * where these fit 64, a tile holds an expert and there is nothing to gain from a larger one (50 rows: 277 us both linears
//    of 62 x 4,096 x 896, against 300 with 128 and 402 with 256);
//  * else by the rounds that the tiles make on the chip, one workgroup a CU. A row of a tile of 128 costs 1.2 times one of a tile
//    of 256, which asks LDS for less per product (198 rows of the same experts: 525 against 448 us); where an expert's
//    last tile is half empty or the tiles just miss a round, 128 is ahead (256 rows of 30 experts of 2,048 x 704: 141
//    against 183 us; 150 rows: 119 against 105).
KA_API int ka_experts_gemm_tile(int n_pairs, int E, int N1, int K1, int act, int N2) {
    const int ff = ka_act_outputs(act, N1);
    if (n_pairs <= 0 || E <= 0 || !experts_dma_covers(N1, K1, ff, act, 0) || !experts_dma_covers(N2, ff, N2, 0, 1)) return KL_ROWS;
    const double rows = (double)n_pairs / E, most = 1.25 * rows;
    if (most <= 64) return 64;
    const int cus = ka_compute_units();
    auto cost = [&](int tile) {
        const double tiles = E * (most <= tile ? 1.0 : rows / tile + 0.5);
        double sum = 0;
        for (const auto& [n, k] : {std::pair<int, int>{N1, K1}, {N2, ff}})
            sum += ceil(tiles * ka_cdiv(n, 256) / cus) * tile * k;
        return sum;
    };
    return cost(256) < 1.2 * cost(128) ? 256 : 128;
}

// The tile whose sums are those of ka_experts_few_bf16; 0: more pairs than that takes, or sizes that its tiles do not cover.
KA_API int ka_experts_gemm_few_tile(int n_pairs, int N1, int K1, int act, int N2) {
    const int ff = ka_act_outputs(act, N1);
    return n_pairs > 0 && n_pairs <= EF_MAX_PAIRS && experts_dma_covers(N1, K1, ff, act, 0) && experts_dma_covers(N2, ff, N2, 0, 1) ? EF_TILE : 0;
}

KA_API int ka_experts_gemm_bf16(const void* a, long lda, int gather_div, const void* W, const int* sorted, const int* tile_expert,
                                int n_tiles, int tile, int N, int K, int act, int clamped, float limit, float slope, float shift, void* out,
                                long ldo, int scatter, int out_f32, hipStream_t stream) {
    const char* who = "ka_experts_gemm_bf16";
    KA_CHECK(!clamped || ka_act_gated(act), "%s: clamps are a gated linear's", who);
    const KaGateClamp clamp{clamped, limit, slope, shift};
    KA_CHECK(n_tiles >= 0 && n_tiles <= 65535 && gather_div >= 0, "%s: bad sizes (%d tiles)", who, n_tiles);
    KA_CHECK(ka_act_known(act) && ka_experts_gemm_supported(lda, N, K, ldo, act, out_f32), "%s: sizes N=%d K=%d not covered", who, N, K);
    KA_CHECK((uintptr_t)a % 16 == 0 && (uintptr_t)W % 16 == 0 && (uintptr_t)out % 16 == 0, "%s: operands must be 16-byte aligned", who);
    if (n_tiles == 0) return 0;
    if (experts_dma_covers(N, K, ldo, act, out_f32)) {
        const ExpertsDmaArgs g{(const bf16_t*)a, lda, gather_div, (const bf16_t*)W, sorted, tile_expert, n_tiles, 0, N, K, act, clamp, out, ldo, scatter};
        if (tile == EF_TILE) return experts_dma_few(g, out_f32, stream);
        if (tile == 64) return experts_dma<2, 1, 4, 2, 3, 2>(g, out_f32, stream);
        if (tile == 128) return experts_dma<2, 2, 4, 2, 3, 2>(g, out_f32, stream);
        if (tile == 256) return experts_dma<2, 4, 4, 2, 2, 1>(g, out_f32, stream);
    }
    KA_CHECK(tile == KL_ROWS, "%s: no kernel for tiles of %d list rows at these sizes", who, tile);
    const dim3 grid((N + KL_COLS - 1) / KL_COLS, n_tiles);
    static bool sized = false;
    if (!sized) {
        (void)hipFuncSetAttribute((const void*)experts_gemm_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        sized = true;
    }
    hipLaunchKernelGGL(experts_gemm_kernel, grid, dim3(256), KL_LDS_BYTES, stream, (const bf16_t*)a, lda, gather_div, (const bf16_t*)W, sorted,
                       tile_expert, N, K, act, clamp, out, ldo, scatter, out_f32);
    KA_LAUNCH_CHECK();
    return 0;
}

// ----------------------------------------------------------------------------
// The same linears for a step of few pairs (a decode step), where all that matters is to read every chosen expert's
// weights once: no lists are made beforehand. A workgroup owns
// 16 weight rows of one expert; it looks through the choices for its expert's pairs (an expert that nobody chose ends there), its
// four waves take every fourth step of 64 inputs each and their sums meet in LDS. Weights are the row operand and pairs
// the columns: a lane ends with four neighbouring outputs of one pair. Up to eight pairs of an expert go with the weights straight into LDS
// where K is in steps of 64 (ef_stream); 16 or 32 at a time, and any other K, from memory to the matrix cores without LDS.
// ----------------------------------------------------------------------------
constexpr int EF_ROWS = 16;
constexpr int EF_WAVES = 4;
typedef __attribute__((ext_vector_type(8))) __bf16 ef_bf16x8;
typedef __attribute__((ext_vector_type(4))) float ef_floatx4;

struct ExpertsFewArgs {
    const bf16_t* a;
    long lda;
    int gather_div;             // the input of pair p is row p / gather_div of `a`
    const bf16_t* W;            // [E, N, K]
    const int* chosen;
    int n_pairs, N, K, act;
    KaGateClamp clamp;
    void* out;                  // row p: the outputs of pair p
    long ldo;
    int out_f32;
};

// Four neighbouring outputs, o to o + 3, of a pair.
__device__ __forceinline__ void ef_store(const ExpertsFewArgs& g, const ef_floatx4 y, int pair, int o) {
    const size_t row = (size_t)pair * g.ldo;
    if (ka_act_gated(g.act)) {
        bf16_t* op = reinterpret_cast<bf16_t*>(g.out) + row + o / 2;
        if (o + 1 < g.N) op[0] = (bf16_t)ka_gate_product<true>(g.act, g.clamp, y[0], y[1]);
        if (o + 3 < g.N) op[1] = (bf16_t)ka_gate_product<true>(g.act, g.clamp, y[2], y[3]);
        return;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (o + r >= g.N) continue;
        const float v = ka_activate_fast(g.act, y[r]);
        if (g.out_f32) reinterpret_cast<float*>(g.out)[row + o + r] = v;
        else reinterpret_cast<bf16_t*>(g.out)[row + o + r] = (bf16_t)v;
    }
}

// The waves' sums through LDS and the outputs of MB * 16 columns; pair: the pair of this lane's column of a block.
template <int MB>
__device__ __forceinline__ void ef_finish(const ExpertsFewArgs& g, const ef_floatx4 (&acc)[MB], const int (&pair)[MB], int count, int first, int row0,
                                          float* sums) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KA_WAVE), lane = threadIdx.x % KA_WAVE;
    const int col = lane % 16, quarter = lane / 16;
#pragma unroll
    for (int m = 0; m < MB; ++m) *reinterpret_cast<ef_floatx4*>(sums + ((wave * MB + m) * KA_WAVE + lane) * 4) = acc[m];
    __syncthreads();
    if (wave >= MB) return;
    ef_floatx4 y = ef_floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int v = 0; v < EF_WAVES; ++v) y += *reinterpret_cast<const ef_floatx4*>(sums + ((v * MB + wave) * KA_WAVE + lane) * 4);
    if (first + wave * 16 + col >= count) return;
    ef_store(g, y, pair[MB == 1 ? 0 : wave], row0 + quarter * 4);
}

template <int MB, int U>
__device__ __forceinline__ void ef_columns(const ExpertsFewArgs& g, const bf16_t* W, const int* list, int count, int first, int row0,
                                           float* sums) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KA_WAVE), lane = threadIdx.x % KA_WAVE;
    const int col = lane % 16, quarter = lane / 16;
    const bf16_t* w = W + (size_t)min(row0 + col, g.N - 1) * g.K;          // (rows past the end: not stored)
    const bf16_t* x[MB];
    int pair[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) {
        pair[m] = list[min(first + m * 16 + col, count - 1)];              // (columns past the last pair repeat it: not stored)
        x[m] = g.a + (size_t)(pair[m] / g.gather_div) * g.lda;
    }
    ef_floatx4 acc[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) acc[m] = ef_floatx4{0.f, 0.f, 0.f, 0.f};
    // (two products a step of 64 inputs: a lane's 16 are neighbours, a row's 64 a whole line; which of them meet in which
    // product is the same for weights and pairs)
    for (int k0 = wave * 64 + quarter * 16; k0 - quarter * 16 < g.K; k0 += EF_WAVES * 32 * U) {
        ef_bf16x8 wv[U], xv[U][MB];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u / 2 * EF_WAVES * 64 + u % 2 * 8;
            const bool in = k < g.K;
#pragma unroll
            for (int i = 0; i < 8; ++i) wv[u][i] = (bf16_t)0.f;
            if (in) wv[u] = __builtin_nontemporal_load(reinterpret_cast<const ef_bf16x8*>(w + k));
#pragma unroll
            for (int m = 0; m < MB; ++m) {
#pragma unroll
                for (int i = 0; i < 8; ++i) xv[u][m][i] = (bf16_t)0.f;
                if (in) xv[u][m] = *reinterpret_cast<const ef_bf16x8*>(x[m] + k);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int m = 0; m < MB; ++m) acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[u], xv[u][m], acc[m], 0, 0, 0);
    }
    ef_finish<MB>(g, acc, pair, count, first, row0, sums);
}

// Up to eight columns of a K in steps of 64: the same products in the same order, operands straight into LDS. A wave's share of a step is whole lines of
// 16 weight rows and of the pairs' rows, in a ring of NS steps of its own (no barrier): in registers they cost a workgroup a place on the CU for every few
// loads in flight, and an instruction touches a half of each of 16 lines. Both linears, us, registers -> three stages (two, four): 30 experts of 2,048 x 704,
// top 4, 1 row 20.5 -> 15.8 (15.8, 17.2), 8 rows 49.0 -> 43.5 (43.7, 47.6), 32 rows 67 -> 60; 62 of 4,096 x 896, top 6, 8 rows 176 -> 155 (157, 161), 32
// rows 281 -> 238 (5.5 TB/s). What is left at few bytes is a workgroup's way: the choices, its one or two rounds of steps, the waves' sums. A workgroup of
// one wave that keeps the four sums apart (no such end) took 50.0 and 202 at 8 rows: its stream is one chain of steps.
constexpr int ES_PAIRS = 8;
constexpr int ES_STAGES = 3;
constexpr int ES_STAGE = (EF_ROWS + ES_PAIRS) * 128;

template <int NS>
__device__ __forceinline__ void ef_stream(const ExpertsFewArgs& g, const bf16_t* W, const int* list, int count, int first, int row0,
                                          unsigned char* lds) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KA_WAVE), lane = threadIdx.x % KA_WAVE;
    const int col = lane % 16, quarter = lane / 16;
    unsigned char* const mine = lds + wave * NS * ES_STAGE;
    const int steps = (g.K / 64 - wave + EF_WAVES - 1) / EF_WAVES;                 // this wave's: wave, wave + 4, ...
    // what this lane asks for: a piece of the weight rows lane / 8 and lane / 8 + 8, and of the pair lane / 8 (rows and pairs past the end: not stored)
    const bf16_t* wsrc[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = kd_load_row<8>(i, lane);
        wsrc[i] = W + (size_t)min(row0 + r, g.N - 1) * g.K + kd_load_channel<8>(r, lane);
    }
    const int asked = list[min(first + kd_load_row<8>(0, lane), count - 1)];
    const bf16_t* const xsrc = g.a + (size_t)(asked / g.gather_div) * g.lda + kd_load_channel<8>(kd_load_row<8>(0, lane), lane);
    auto fetch = [&](int stage, int s) {
        unsigned char* const base = mine + stage * ES_STAGE;
        const int k = (wave + s * EF_WAVES) * 64;
#pragma unroll
        for (int i = 0; i < 2; ++i)
            __builtin_amdgcn_global_load_lds((const GD_GLOBAL void*)(wsrc[i] + k), (GD_LDS void*)(base + i * 1024), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((const GD_GLOBAL void*)(xsrc + k), (GD_LDS void*)(base + EF_ROWS * 128), 16, 0, 0);
    };
    for (int s = 0; s < NS && s < steps; ++s) fetch(s, s);
    ef_floatx4 acc[1] = {{0.f, 0.f, 0.f, 0.f}};
    const int wplace = col * 128, xplace = EF_ROWS * 128 + col % ES_PAIRS * 128;
    int stage = 0;                                                                 // of step s
    for (int s = 0; s < steps; ++s) {
        gd_wait_younger<3, NS - 1>(steps - 1 - s);                                 // this step has landed
        asm volatile("" ::: "memory");
        const unsigned char* const base = mine + stage * ES_STAGE;
        ef_bf16x8 w[2], x[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            w[h] = *reinterpret_cast<const ef_bf16x8*>(base + wplace + (((quarter * 2 + h) ^ kd_swizzle<8>(col)) * 16));
            x[h] = *reinterpret_cast<const ef_bf16x8*>(base + xplace + (((quarter * 2 + h) ^ kd_swizzle<8>(col % ES_PAIRS)) * 16));
        }
        gd_wait_lds();                                                             // and is in registers: its place is free
        asm volatile("" ::: "memory");
        if (s + NS < steps) fetch(stage, s + NS);
        stage = stage + 1 == NS ? 0 : stage + 1;
#pragma unroll
        for (int h = 0; h < 2; ++h) acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[h], x[h], acc[0], 0, 0, 0);
    }
    __syncthreads();                                                               // (the sums take the place of the stages)
    const int pair[1] = {list[min(first + col, count - 1)]};
    ef_finish<1>(g, acc, pair, count, first, row0, reinterpret_cast<float*>(lds));
}

constexpr int es_room(int NS) { return NS * EF_WAVES * ES_STAGE > EF_WAVES * 2 * KA_WAVE * 16 ? NS * EF_WAVES * ES_STAGE : EF_WAVES * 2 * KA_WAVE * 16; }

// NS: stages of ef_stream (K in steps of 64: the host's check); 0: any K.
template <int NS>
__global__ void __launch_bounds__(EF_WAVES * KA_WAVE) experts_few_kernel(ExpertsFewArgs g) {
    __shared__ int list[EF_MAX_PAIRS];
    __shared__ __attribute__((aligned(16))) unsigned char room[es_room(NS)];
    float* const sums = reinterpret_cast<float*>(room);
    const int e = blockIdx.y, lane = threadIdx.x % KA_WAVE;
    // (every wave makes the list by itself: all write the same numbers)
    int mine[EF_MAX_PAIRS / KA_WAVE];
#pragma unroll
    for (int i = 0; i < EF_MAX_PAIRS / KA_WAVE; ++i) mine[i] = i * KA_WAVE + lane < g.n_pairs ? g.chosen[i * KA_WAVE + lane] : -1;
    int count = 0;
#pragma unroll
    for (int i = 0; i < EF_MAX_PAIRS / KA_WAVE; ++i) {
        const unsigned long long hit = __builtin_amdgcn_ballot_w64(mine[i] == e);
        if (mine[i] == e) list[count + __popcll(hit & ((1ull << lane) - 1))] = i * KA_WAVE + lane;
        count += __popcll(hit);
    }
    if (count == 0) return;
    __syncthreads();
    const bf16_t* W = g.W + (size_t)e * g.N * g.K;
    const int row0 = blockIdx.x * EF_ROWS;
    for (int first = 0; first < count;) {
        if (NS > 0 && count - first <= ES_PAIRS) {
            if constexpr (NS > 0) ef_stream<NS>(g, W, list, count, first, row0, room);
            first += ES_PAIRS;
        } else if (count - first <= 16) {
            ef_columns<1, 8>(g, W, list, count, first, row0, sums);
            first += 16;
        } else {
            ef_columns<2, 4>(g, W, list, count, first, row0, sums);
            first += 32;
        }
        __syncthreads();
    }
}

// Whether the kernel takes the call: inputs in steps of 8, 16-byte rows, gated pairs inside N.
KA_API int ka_experts_few_supported(int n_pairs, long lda, int N, int K, int act) {
    return n_pairs > 0 && n_pairs <= EF_MAX_PAIRS && N > 0 && K > 0 && K % 8 == 0 && lda % 8 == 0 && (!ka_act_gated(act) || N % 2 == 0) ? 1 : 0;
}

KA_API int ka_experts_few_bf16(const void* a, long lda, int gather_div, const void* W, const int* chosen, int n_pairs, int E, int N, int K,
                               int act, int clamped, float limit, float slope, float shift, void* out, long ldo, int out_f32,
                               hipStream_t stream) {
    const char* who = "ka_experts_few_bf16";
    KA_CHECK(!clamped || ka_act_gated(act), "%s: clamps are a gated linear's", who);
    KA_CHECK(ka_act_known(act) && ka_experts_few_supported(n_pairs, lda, N, K, act), "%s: %d pairs, N=%d K=%d not covered", who, n_pairs, N, K);
    KA_CHECK(E > 0 && E <= 65535 && gather_div > 0 && lda >= K && ldo >= (ka_act_gated(act) ? N / 2 : N), "%s: bad sizes", who);
    KA_CHECK(!ka_act_gated(act) || !out_f32, "%s: a gated linear writes bf16", who);
    KA_CHECK((uintptr_t)a % 16 == 0 && (uintptr_t)W % 16 == 0, "%s: operands must be 16-byte aligned", who);
    const ExpertsFewArgs g{(const bf16_t*)a, lda, gather_div, (const bf16_t*)W, chosen, n_pairs, N, K, act, {clamped, limit, slope, shift}, out, ldo, out_f32};
    auto kernel = K % 64 == 0 ? experts_few_kernel<ES_STAGES> : experts_few_kernel<0>;
    hipLaunchKernelGGL(kernel, dim3(ka_cdiv(N, EF_ROWS), E), dim3(EF_WAVES * KA_WAVE), 0, stream, g);
    KA_LAUNCH_CHECK();
    return 0;
}

// ----------------------------------------------------------------------------
// Several linears of a step of few rows in one launch, each with an input of its own: out_g = act_g(a_g W_g^T), all of one K. The work of
// a workgroup is that of the experts' kernel above, 16 weight rows of one linear over all of its inputs. What a linear of its own
// spends beside its stream (the launch, the first trip to memory) is paid once: five linears of 2,048 inputs (four of 2,048 outputs,
// one of 64) at eight rows took 27 us one by one and take 14.5.
// ----------------------------------------------------------------------------
constexpr int LF_MAX_LINEARS = 8;
constexpr int LF_MAX_ROWS = 32;

struct LinearsFewArgs {
    const bf16_t* a[LF_MAX_LINEARS];
    const bf16_t* W[LF_MAX_LINEARS];
    bf16_t* out[LF_MAX_LINEARS];
    long ldo[LF_MAX_LINEARS];
    int N[LF_MAX_LINEARS], act[LF_MAX_LINEARS], first[LF_MAX_LINEARS + 1];       // first: workgroups before linear g
    long lda;
    int count, rows, K;
};

__global__ void __launch_bounds__(EF_WAVES * KA_WAVE) linears_few_kernel(LinearsFewArgs p) {
    __shared__ int list[LF_MAX_ROWS];
    __shared__ __attribute__((aligned(16))) float sums[EF_WAVES * 2 * KA_WAVE * 4];
    int g = 0;
    while (g + 1 < p.count && (int)blockIdx.x >= p.first[g + 1]) ++g;
    if (threadIdx.x < LF_MAX_ROWS) list[threadIdx.x] = threadIdx.x;
    __syncthreads();
    const ExpertsFewArgs one{p.a[g], p.lda, 1, nullptr, nullptr, p.rows, p.N[g], p.K, p.act[g], KaGateClamp{0, 0.f, 0.f, 0.f}, p.out[g], p.ldo[g], 0};
    const int row0 = ((int)blockIdx.x - p.first[g]) * EF_ROWS;
    if (p.rows <= 16) ef_columns<1, 8>(one, p.W[g], list, p.rows, 0, row0, sums);
    else ef_columns<2, 4>(one, p.W[g], list, p.rows, 0, row0, sums);
}

// `a`, `W`, `out`: one pointer a linear; inputs [rows, K] of row stride lda, weights [N, K], bf16 outputs of row stride ldo.
KA_API int ka_linears_few_bf16(int count, const void* const* a, long lda, const void* const* W, const int* N, const int* act, void* const* out,
                               const long* ldo, int rows, int K, hipStream_t stream) {
    const char* who = "ka_linears_few_bf16";
    KA_CHECK(count > 0 && count <= LF_MAX_LINEARS && rows > 0 && rows <= LF_MAX_ROWS, "%s: %d linears of %d rows", who, count, rows);
    KA_CHECK(K > 0 && K % 8 == 0 && lda >= K && lda % 8 == 0, "%s: inputs in steps of 8", who);
    LinearsFewArgs p{};
    p.lda = lda;
    p.count = count;
    p.rows = rows;
    p.K = K;
    for (int g = 0; g < count; ++g) {
        KA_CHECK(N[g] > 0 && N[g] < (1 << 24) && ka_act_known(act[g]) && !ka_act_gated(act[g]) && ldo[g] >= N[g], "%s: linear %d: sizes or activation", who, g);
        KA_CHECK((uintptr_t)a[g] % 16 == 0 && (uintptr_t)W[g] % 16 == 0, "%s: operands must be 16-byte aligned", who);
        p.a[g] = (const bf16_t*)a[g];
        p.W[g] = (const bf16_t*)W[g];
        p.out[g] = (bf16_t*)out[g];
        p.ldo[g] = ldo[g];
        p.N[g] = N[g];
        p.act[g] = act[g];
        p.first[g + 1] = p.first[g] + ka_cdiv(N[g], EF_ROWS);
    }
    hipLaunchKernelGGL(linears_few_kernel, dim3(p.first[count]), dim3(EF_WAVES * KA_WAVE), 0, stream, p);
    KA_LAUNCH_CHECK();
    return 0;
}
