// Tiled bf16 linear layer for prompts: out = act(A W^T + bias) or out += A W^T + bias.
//
// Both operands are K-contiguous (A [M, K], W [N, K]), which is exactly what the MFMA
// operand layout wants: a lane holds 8 consecutive k of one row. A workgroup of four waves
// (2 x 2) computes a tile of 64 NT weight rows x 64 MT activation rows in K-steps of BK through
// double-buffered LDS (rows padded by 16 bytes, which keeps the 16-byte operand reads off each
// other's banks); each wave owns NT x MT v_mfma_f32_32x32x16_bf16 tiles. The weight rows are the
// MFMA's row operand, so a lane ends up with four consecutive output columns of one output row
// and stores them as one vector. Bias, GELU-tanh and the fp32 residual accumulate run in the
// epilogue.
//
// That kernel takes any K (in steps of 8); where K is a multiple of 64 the large-tile kernel
// further down, which loads straight into LDS, is used instead.
#include "ka_common.h"
#include "ka_dma_tiles.h"
#include "ka_partials.h"

#include <stdlib.h>

#include <type_traits>

constexpr int GB_THREADS = 256;
constexpr int GB_PAD = 8;          // bf16 of padding per LDS row

constexpr int gb_smem(int nt, int mt, int bk) { return 2 * 64 * (nt + mt) * (bk + GB_PAD) * 2; }

__device__ __forceinline__ bf16x8 gb_load8(const bf16_t* p) { return *reinterpret_cast<const bf16x8*>(p); }

template <int NT, int MT, int BK>
__global__ void __launch_bounds__(GB_THREADS)
gemm_bf16_kernel(const bf16_t* __restrict__ A, long lda, const bf16_t* __restrict__ W, long ldw,
                 const float* __restrict__ bias, void* __restrict__ out, int out_dtype, long ldo, int M,
                 int N, int K, int act, int accumulate, int tiles_n, int tiles_m) {
    constexpr int BN = 64 * NT, BM = 64 * MT, LD = BK + GB_PAD;
    constexpr int CPR = BK / 8;                          // 16-byte chunks per tile row
    constexpr int WCH = BN * CPR / GB_THREADS;           // chunks of W a thread moves per k-step
    constexpr int XCH = BM * CPR / GB_THREADS;
    static_assert(BN * CPR % GB_THREADS == 0 && BM * CPR % GB_THREADS == 0, "tile does not divide over the threads");
    extern __shared__ __attribute__((aligned(16))) unsigned char gb_lds[];
    bf16_t (*Ws)[BN][LD] = reinterpret_cast<bf16_t (*)[BN][LD]>(gb_lds);
    bf16_t (*Xs)[BM][LD] = reinterpret_cast<bf16_t (*)[BM][LD]>(gb_lds + 2 * BN * LD * sizeof(bf16_t));
    // Tiles are numbered so that the workgroups one XCD gets (every 8th) walk down a column of
    // tiles that share the same weight rows, which then stay in that XCD's L2.
    int pid = blockIdx.x;
    int total = tiles_n * tiles_m;
    int per_xcd = (total + 7) / 8;
    int logical = (pid % 8) * per_xcd + pid / 8;
    if (logical >= total) return;
    int tn = logical / tiles_m, tm = logical % tiles_m;
    const int n0 = tn * BN, m0 = tm * BM;
    const int tid = threadIdx.x, wave = tid / KA_WAVE, lane = tid % KA_WAVE;
    const int wn = wave / 2, wm = wave % 2;
    const int li = lane % 32, lg = lane / 32;

    floatx16 acc[NT][MT];
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int b = 0; b < MT; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.f;

    const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
    bf16x8 wreg[WCH], xreg[XCH];
    // chunk c = tid + i * 256: row c / CPR, k-chunk c % CPR
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < WCH; ++i) {
            int c = tid + i * GB_THREADS;
            int n = n0 + c / CPR, k = k0 + (c % CPR) * 8;
            wreg[i] = (n < N && k < K) ? gb_load8(W + (size_t)n * ldw + k) : zero;
        }
#pragma unroll
        for (int i = 0; i < XCH; ++i) {
            int c = tid + i * GB_THREADS;
            int m = m0 + c / CPR, k = k0 + (c % CPR) * 8;
            xreg[i] = (m < M && k < K) ? gb_load8(A + (size_t)m * lda + k) : zero;
        }
    };
    auto stash = [&](int buf) {
#pragma unroll
        for (int i = 0; i < WCH; ++i) {
            int c = tid + i * GB_THREADS;
            *reinterpret_cast<bf16x8*>(&Ws[buf][c / CPR][(c % CPR) * 8]) = wreg[i];
        }
#pragma unroll
        for (int i = 0; i < XCH; ++i) {
            int c = tid + i * GB_THREADS;
            *reinterpret_cast<bf16x8*>(&Xs[buf][c / CPR][(c % CPR) * 8]) = xreg[i];
        }
    };

    const int steps = (K + BK - 1) / BK;
    fetch(0);
    stash(0);
    __syncthreads();
    for (int s = 0; s < steps; ++s) {
        int buf = s & 1;
        if (s + 1 < steps) fetch((s + 1) * BK);
#pragma unroll
        for (int ks = 0; ks < BK / 16; ++ks) {
            bf16x8 wa[NT], xb[MT];
#pragma unroll
            for (int t = 0; t < NT; ++t)
                wa[t] = *reinterpret_cast<const bf16x8*>(&Ws[buf][wn * 32 * NT + t * 32 + li][ks * 16 + lg * 8]);
#pragma unroll
            for (int t = 0; t < MT; ++t)
                xb[t] = *reinterpret_cast<const bf16x8*>(&Xs[buf][wm * 32 * MT + t * 32 + li][ks * 16 + lg * 8]);
#pragma unroll
            for (int a = 0; a < NT; ++a)
#pragma unroll
                for (int b = 0; b < MT; ++b)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wa[a], xb[b], acc[a][b], 0, 0, 0);
        }
        if (s + 1 < steps) stash(buf ^ 1);
        __syncthreads();
    }

    // epilogue: acc[a][b][v] is out[m][n] with n = n0 + wn*32*NT + a*32 + (v/4)*8 + lg*4 + v%4,
    // m = m0 + wm*32*MT + b*32 + li
    const bool vec_ok = (N % 4 == 0) && (ldo % 4 == 0);
#pragma unroll
    for (int b = 0; b < MT; ++b) {
        int m = m0 + wm * 32 * MT + b * 32 + li;
        if (m >= M) continue;
#pragma unroll
        for (int a = 0; a < NT; ++a) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                int n = n0 + wn * 32 * NT + a * 32 + q * 8 + lg * 4;
                if (n >= N) continue;
                float v[4];
                if (ka_act_gated(act)) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] = acc[a][b][q * 4 + i] + (bias && n + i < N ? bias[n + i] : 0.f);
                    ka_gated_store<true, 4>(out, out_dtype, ldo, m, n, N, v, act);
                    continue;
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float x = acc[a][b][q * 4 + i];
                    if (bias && n + i < N) x += bias[n + i];
                    if (act) x = ka_activate_fast(act, x);
                    v[i] = x;
                }
                size_t o = (size_t)m * ldo + n;
                if (out_dtype == KA_F32) {
                    float* op = reinterpret_cast<float*>(out) + o;
                    if (vec_ok) {
                        floatx4 cur = accumulate ? *reinterpret_cast<floatx4*>(op) : floatx4{0.f, 0.f, 0.f, 0.f};
                        floatx4 res = {cur[0] + v[0], cur[1] + v[1], cur[2] + v[2], cur[3] + v[3]};
                        *reinterpret_cast<floatx4*>(op) = res;
                    } else {
                        for (int i = 0; i < 4 && n + i < N; ++i) op[i] = accumulate ? op[i] + v[i] : v[i];
                    }
                } else {
                    bf16_t* op = reinterpret_cast<bf16_t*>(out) + o;
                    if (vec_ok) {
                        bf16x4 res = {(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
                        *reinterpret_cast<bf16x4*>(op) = res;
                    } else {
                        for (int i = 0; i < 4 && n + i < N; ++i) op[i] = (bf16_t)v[i];
                    }
                }
            }
        }
    }
}

// ----------------------------------------------------------------------------
// The large-tile kernel: four (2 x 2) or eight (4 x 2) waves over the loop of ka_dma_tiles.h. Rows past the end of a matrix are
// read from its last row (and never stored); K must be a multiple of BK.
// ----------------------------------------------------------------------------
template <int WN, int WM, int GN, int GM, int BK, int NS, int SL>
__global__ void __launch_bounds__(KA_WAVE * GN * GM)
    __attribute__((amdgpu_waves_per_eu(GN * GM / 4, (WN * WM > 8 ? 1 : 2) * (GN * GM / 4))))
gemm_dma_kernel(const bf16_t* __restrict__ A, long lda, const bf16_t* __restrict__ W, long ldw,
                const float* __restrict__ bias, void* __restrict__ out, int out_dtype, long ldo, int M,
                int N, int K, int act, int accumulate, int tiles_n, int tiles_m, int k_per) {
    // K cut into parts (grid y): part p multiplies the k_per columns from p * k_per on and writes
    // its sums as fp32 [M, N] of its own (the host passes the partial buffer as `out`, no bias,
    // no activation; a finishing kernel adds the parts up)
    if (k_per > 0) {
        const int part = blockIdx.y;
        A += (size_t)part * k_per;
        W += (size_t)part * k_per;
        K = min(k_per, K - part * k_per);
        out = reinterpret_cast<float*>(out) + (size_t)part * M * ldo;
    }
    using T = KdTile<WN, WM, GN, GM, BK, NS>;
    constexpr int WAVES = T::WAVES, BN = T::BN, BM = T::BM, CPR = T::CPR, W_LOADS = T::W_LOADS, X_LOADS = T::X_LOADS;
    extern __shared__ __attribute__((aligned(16))) unsigned char gb_lds[];
    int pid = blockIdx.x;
    int total = tiles_n * tiles_m;
    int per_xcd = (total + 7) / 8;
    int logical = (pid % 8) * per_xcd + pid / 8;
    if (logical >= total) return;
    int tn = logical / tiles_m, tm = logical % tiles_m;
    const int n0 = tn * BN, m0 = tm * BM;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / KA_WAVE), lane = tid % KA_WAVE;
    const int wn = wave / GM, wm = wave % GM;
    const int li = lane % 32, lg = lane / 32;

    floatx16 acc[WN][WM];
#pragma unroll
    for (int a = 0; a < WN; ++a)
#pragma unroll
        for (int b = 0; b < WM; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.f;

    // What this lane asks for in the wave's loads. Rows past the end of a matrix are read from its last row (and never stored).
    const bf16_t* wsrc[W_LOADS];
    const bf16_t* xsrc[X_LOADS];
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i) {
        const int r = kd_load_row<CPR>(wave * W_LOADS + i, lane);
        wsrc[i] = W + (size_t)min(n0 + r, N - 1) * ldw + kd_load_channel<CPR>(r, lane);
    }
#pragma unroll
    for (int i = 0; i < X_LOADS; ++i) {
        const int r = kd_load_row<CPR>(wave * X_LOADS + i, lane);
        xsrc[i] = A + (size_t)min(m0 + r, M - 1) * lda + kd_load_channel<CPR>(r, lane);
    }
    // (The arguments that only the epilogue uses are asked for here: the compiler otherwise fetches them, with scalar loads, as
    // late as it can, and a scalar load in flight on the counter that LDS reads share makes the loop wait for all of them.)
    asm volatile("" ::"s"(bias), "s"(out), "s"(ldo), "s"(act), "s"(accumulate), "s"(out_dtype), "s"(M), "s"(N));
    kd_product<WN, WM, GN, GM, BK, NS, SL>(gb_lds, wave, lane, K, wsrc, xsrc, acc);

    // Epilogue. acc[a][b][v] is out[m][n] with n = n0 + wn*32*WN + a*32 + (v/4)*8 + lg*4 + v%4 and
    // m = m0 + wm*32*WM + b*32 + li: a lane holds four neighbouring outputs of one row, and one
    // store instruction of the wave would touch 32 rows with 16 (bf16) or 32 bytes each, which the
    // memory system takes at a fraction of its rate (measured: 15 us of 79 for the 33 MB of the
    // first feed-forward linear of a 2,048-token prompt). So a wave passes its outputs through its
    // share of the stages' LDS, 32 rows at a time or more, and stores whole rows of its tile: 128
    // or 256 contiguous bytes per row, 16 bytes per lane. Bias and activation are applied on the
    // way in; an fp32 output that accumulates is read and added on the way out.
    gd_barrier();                                        // the last stage has been read by everybody
    const bool bias_vec = (N % 4 == 0) && (reinterpret_cast<uintptr_t>(bias) % 16 == 0);
    auto staged = [&](auto* typed_out) {
        using E = std::remove_pointer_t<decltype(typed_out)>;
        constexpr int ES = sizeof(E);                    // 2 or 4
        constexpr int PER = 16 / ES;                     // outputs per 16-byte store
        constexpr int RB = 32 * WN * ES;                 // bytes of a row of the wave's tile
        constexpr int RS = RB + (ES == 2 ? 8 : 16);      // its place in LDS: padded so that the lanes' writes spread over the banks
        constexpr int SHARE = gd_smem(BN, BM, BK, NS) / WAVES;
        constexpr int BP = SHARE / (32 * RS) < WM ? SHARE / (32 * RS) : WM;      // blocks of 32 rows per pass
        static_assert(BP >= 1, "a wave's share of LDS does not hold 32 rows of its tile");
        constexpr int CH = RB / 16;                      // 16-byte chunks of a row
        constexpr int RPI = KA_WAVE / CH;                // rows one store instruction covers
        unsigned char* mine = gb_lds + wave * SHARE;
        const int n_wave = n0 + wn * 32 * WN, m_wave = m0 + wm * 32 * WM;
        const bool wide = (ldo * ES) % 16 == 0 && reinterpret_cast<uintptr_t>(typed_out) % 16 == 0 && n0 % PER == 0;
        gd_static_for<0, (WM + BP - 1) / BP>([&](auto pc) {
            constexpr int b0 = decltype(pc)::value * BP;
            constexpr int nb = b0 + BP <= WM ? BP : WM - b0;
            gd_static_for<0, nb>([&](auto bc) {
                constexpr int b = b0 + decltype(bc)::value;
                gd_static_for<0, WN>([&](auto ac) {
                    constexpr int a = decltype(ac)::value;
                    gd_static_for<0, 4>([&](auto qc) {
                        constexpr int q = decltype(qc)::value;
                        const int nl = a * 32 + q * 8 + lg * 4;
                        const int n = n_wave + nl;
                        floatx4 bv = {0.f, 0.f, 0.f, 0.f};
                        if (bias && n < N) {
                            if (bias_vec) bv = *reinterpret_cast<const floatx4*>(bias + n);       // n + 3 < N: N % 4 == 0
                            else
                                for (int i = 0; i < 4 && n + i < N; ++i) bv[i] = bias[n + i];
                        }
                        float v[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            float x = acc[a][b][q * 4 + i] + bv[i];
                            if (act) x = ka_activate_fast(act, x);
                            v[i] = x;
                        }
                        unsigned char* at = mine + ((b - b0) * 32 + li) * RS + nl * ES;
                        if constexpr (ES == 2) *reinterpret_cast<bf16x4*>(at) = bf16x4{(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
                        else *reinterpret_cast<floatx4*>(at) = floatx4{v[0], v[1], v[2], v[3]};
                    });
                });
            });
            at_epilogue_wave_sync();
#pragma unroll
            for (int r0 = 0; r0 < nb * 32; r0 += RPI) {
                const int rl = r0 + lane / CH, c = lane % CH;
                const int m = m_wave + b0 * 32 + rl, n = n_wave + c * PER;
                if (lane < RPI * CH && rl < nb * 32 && m < M && n < N) {      // (a row's chunks need not divide 64 lanes)
                    const unsigned char* from = mine + rl * RS + c * 16;
                    E* op = typed_out + (size_t)m * ldo + n;
                    if (wide && n + PER <= N) {
                        if constexpr (ES == 2) {
                            *reinterpret_cast<bf16x8*>(op) = *reinterpret_cast<const bf16x8*>(from);
                        } else {
                            floatx4 x = *reinterpret_cast<const floatx4*>(from);
                            if (accumulate) {
                                const floatx4 cur = *reinterpret_cast<const floatx4*>(op);
                                x = floatx4{cur[0] + x[0], cur[1] + x[1], cur[2] + x[2], cur[3] + x[3]};
                            }
                            *reinterpret_cast<floatx4*>(op) = x;
                        }
                    } else {
                        const E* src = reinterpret_cast<const E*>(from);
                        for (int i = 0; i < PER && n + i < N; ++i) {
                            if constexpr (ES == 2) op[i] = src[i];
                            else op[i] = accumulate ? op[i] + src[i] : src[i];
                        }
                    }
                }
            }
            at_epilogue_wave_sync();                     // the next pass writes over what was just read
        });
    };
    if (out_dtype == KA_F32) staged(reinterpret_cast<float*>(out));
    else staged(reinterpret_cast<bf16_t*>(out));
}

template <int WN, int WM, int GN, int GM, int BK, int NS, int SL = 1>
static int launch_dma(const bf16_t* A, long lda, const bf16_t* W, long ldw, const float* bias, void* out,
                      int out_dtype, long ldo, int M, int N, int K, int act, int accumulate, hipStream_t stream,
                      int parts = 1, int k_per = 0) {
    static bool configured = false;
    constexpr int BN = 32 * WN * GN, BM = 32 * WM * GM;
    constexpr int smem = gd_smem(BN, BM, BK, NS);
    static_assert(smem <= 160 * 1024, "the stages do not fit in LDS");
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_dma_kernel<WN, WM, GN, GM, BK, NS, SL>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        KA_CHECK(e == hipSuccess, "ka_linear_tiled_bf16: cannot reserve %d bytes of LDS: %s", smem, hipGetErrorString(e));
        configured = true;
    }
    int tiles_n = ka_cdiv(N, BN), tiles_m = ka_cdiv(M, BM);
    long total = (long)tiles_n * tiles_m;
    long launched = ((total + 7) / 8) * 8;
    KA_CHECK(launched < (1L << 31), "ka_linear_tiled_bf16: too many tiles");
    hipLaunchKernelGGL((gemm_dma_kernel<WN, WM, GN, GM, BK, NS, SL>), dim3((unsigned)launched, parts), dim3(KA_WAVE * GN * GM), smem,
                       stream, A, lda, W, ldw, bias, out, out_dtype, ldo, M, N, K, act, accumulate, tiles_n, tiles_m, k_per);
    return 0;
}

// The two last linears of a block whose branches run side by side, out += A1 W1^T + A2 W2^T, for more rows than the
// weight-streaming kernels take and fewer than fill the chip with tiles of the output: K of both, one behind the other, is cut
// into `parts` parts of `per` K-steps, and a part's sums go out as fp32 [M, N] of its own, which the kernel that
// finishes the rows adds up (with both biases, the residual and the next block's norm).
// (KaPairTiles in ka_partials.h.)
//
// The rows of A are the product's first operand here: a lane then holds one column of 16 rows, and a store of the wave covers
// two rows of 128 bytes, whole lines of the memory, without a pass through LDS.
template <int WN, int WM, int GN, int GM, int BK, int NS, int SL>
__global__ void __launch_bounds__(KA_WAVE * GN * GM) __attribute__((amdgpu_waves_per_eu(GN * GM / 4, GN * GM / 4)))
pair_tiles_kernel(KaPairTiles p) {
    using T = KdTile<WN, WM, GN, GM, BK, NS>;
    constexpr int CPR = T::CPR;
    extern __shared__ __attribute__((aligned(16))) unsigned char gb_lds[];
    const KaPairPlace at = ka_pair_place(p, blockIdx.x);
    if (at.part < 0) return;
    const int m0 = at.tile_m * T::BN, n0 = at.tile_n * T::BM;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / KA_WAVE), lane = tid % KA_WAVE;
    const int lo = at.part * p.per, hi = min(lo + p.per, p.steps[0] + p.steps[1]);

    floatx16 acc[WN][WM];
#pragma unroll
    for (int a = 0; a < WN; ++a)
#pragma unroll
        for (int b = 0; b < WM; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.f;
#pragma unroll 1
    for (int s = 0; s < 2; ++s) {
        const int before = s ? p.steps[0] : 0;
        const int first = max(lo - before, 0), last = min(hi - before, p.steps[s]);
        if (first >= last) continue;                     // (the same for the whole workgroup)
        const bf16_t* const A = p.A[s] + (size_t)first * BK;
        const bf16_t* const W = p.W[s] + (size_t)first * BK;
        const bf16_t* asrc[T::W_LOADS];
        const bf16_t* wsrc[T::X_LOADS];
#pragma unroll
        for (int i = 0; i < T::W_LOADS; ++i) {
            const int r = kd_load_row<CPR>(wave * T::W_LOADS + i, lane);
            asrc[i] = A + (size_t)min(m0 + r, p.M - 1) * p.lda[s] + kd_load_channel<CPR>(r, lane);
        }
#pragma unroll
        for (int i = 0; i < T::X_LOADS; ++i) {
            const int r = kd_load_row<CPR>(wave * T::X_LOADS + i, lane);
            wsrc[i] = W + (size_t)min(n0 + r, p.N - 1) * p.ldw[s] + kd_load_channel<CPR>(r, lane);
        }
        // everybody has read the last stage of the segment before
        gd_wait_lds();
        gd_barrier();
        kd_product<WN, WM, GN, GM, BK, NS, SL>(gb_lds, wave, lane, (last - first) * BK, asrc, wsrc, acc);
    }

    float* const mine = p.partial + (size_t)at.part * p.M * p.N;
    const int wn = wave / GM, wm = wave % GM, li = lane % 32, lg = lane / 32;
#pragma unroll
    for (int b = 0; b < WM; ++b) {
        const int n = n0 + wm * 32 * WM + b * 32 + li;
        if (n >= p.N) continue;
#pragma unroll
        for (int a = 0; a < WN; ++a)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int m = m0 + wn * 32 * WN + a * 32 + (v / 4) * 8 + lg * 4 + v % 4;
                if (m < p.M) mine[(size_t)m * p.N + n] = acc[a][b][v];
            }
    }
}

// Bound by the K-steps that follow one another on a CU, 0.5 to 0.6 us each whatever the stages in flight (three to five: 73 to
// 71 us for K = 8,192 alone on 64 CUs): parts of K spread them over all CUs. Measured with the norm that follows, against the
// vendor library's two products and the norm's launch (us; K = 2,560 + 10,240, N = 2,560): 128 rows 31 against 78, 512 rows
// 56.5 (three parts) against 83, 1,024 rows 108 against 117 (where the phased tiles of 256 rows take over: pair_tiles_choice).
constexpr int PT_TILE = 128, PT_BK = 64, PT_STAGES = 5, PT_TILE_CODE = 100;

template <int WN, int WM, int GN, int GM, int NS, int SL>
static int launch_pair_tiles(KaPairTiles& p, int parts, hipStream_t stream) {
    using T = KdTile<WN, WM, GN, GM, PT_BK, NS>;
    static bool configured = false;
    auto kernel = pair_tiles_kernel<WN, WM, GN, GM, PT_BK, NS, SL>;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, T::SMEM);
        KA_CHECK(e == hipSuccess, "linear by tiles: cannot reserve %d bytes of LDS: %s", T::SMEM, hipGetErrorString(e));
        configured = true;
    }
    p.tiles_m = ka_cdiv(p.M, T::BN);
    p.tiles_n = ka_cdiv(p.N, T::BM);
    p.parts = parts;
    const long launched = (((long)p.tiles_n * p.tiles_m * parts + 7) / 8) * 8;
    KA_CHECK(launched < (1L << 31), "linear by tiles: too many tiles");
    hipLaunchKernelGGL(kernel, dim3((unsigned)launched), dim3(KA_WAVE * T::WAVES), T::SMEM, stream, p);
    KA_LAUNCH_CHECK();
    return 0;
}

// Few rows (at most 64), for the weight-streaming launcher: the sums of one linear, or of two added up, in parts in `partial`. Parts and
// order of a sum are those of skinny_wide_kernel, whose bits these are: part p has the p-th range of K of either linear, and a part's sum is
// that of the first halves of its K-steps plus that of the second.
//
// Bound by the weights' way from HBM: what counts is that every CU has 64 KB of loads in flight, which the stages in LDS hold without
// registers. Tiles of 64 weight rows by all rows, five stages in half of a CU's LDS, four waves; an XCD's tiles are neighbours. At 40
// rows, us, weights from HBM, the launch that adds up included, against that kernel: N = 2,048, K = 2,048 + 8,192: 15.2 and 18.6; 2,560, 2,560 +
// 10,240: 20.1 and 24.8; N = K = 4,096: 13.0 and 16.3; 4,096 by 12,288: 26.4 and 31.0; at 17 and 64 rows likewise. (One linear whose K would be in one part goes by
// gemm_few_bf16.hip, but for outputs in no fours.)
template <int WN, int WM, int GN, int GM, int NS>
__global__ void __launch_bounds__(KA_WAVE * GN * GM) __attribute__((amdgpu_waves_per_eu(2, 2)))
few_rows_kernel(KaFewRows p) {
    using T = KdTile<WN, WM, GN, GM, 64, NS, 16>;
    constexpr int CPR = T::CPR;
    extern __shared__ __attribute__((aligned(16))) unsigned char gb_lds[];
    const int tiles = (p.N + T::BN - 1) / T::BN, per_xcd = (tiles + 7) / 8;
    const int tile = blockIdx.x % 8 * per_xcd + blockIdx.x / 8;        // an XCD's tiles: neighbours
    if (tile >= tiles) return;
    const int n0 = tile * T::BN, part = blockIdx.y;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KA_WAVE), lane = threadIdx.x % KA_WAVE;
    int first[2], count[2];                              // this part's K-steps of either linear
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const int all = p.K[s] / 64, per = (all + p.parts - 1) / p.parts;
        first[s] = min(part * per, all);
        count[s] = min(per, all - first[s]);
    }
    const bf16_t* w[2][T::W_LOADS];
    const bf16_t* x[2][T::X_LOADS];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const bool has = p.K[s] > 0;
#pragma unroll
        for (int i = 0; i < T::W_LOADS; ++i) {
            const int r = kd_load_row<CPR>(wave * T::W_LOADS + i, lane);
            w[s][i] = has ? (const bf16_t*)p.W[s] + (size_t)min(n0 + r, p.N - 1) * p.ldw[s] + first[s] * 64 + kd_load_channel<CPR>(r, lane) : nullptr;
        }
#pragma unroll
        for (int i = 0; i < T::X_LOADS; ++i) {
            const int r = kd_load_row<CPR>(wave * T::X_LOADS + i, lane);
            x[s][i] = has ? (const bf16_t*)p.A[s] + (size_t)min(r, p.M - 1) * p.lda[s] + first[s] * 64 + kd_load_channel<CPR>(r, lane) : nullptr;
        }
    }
    floatx4 acc[KD_HALVES][WN][WM];
#pragma unroll
    for (int h = 0; h < KD_HALVES; ++h)
#pragma unroll
        for (int a = 0; a < WN; ++a)
#pragma unroll
            for (int b = 0; b < WM; ++b) acc[h][a][b] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int steps = count[0] + count[1];
    if (steps > 0)                                       // (the same for the whole workgroup)
        kd_product_16<WN, WM, GN, GM, NS, KD_HALVES>(
            gb_lds, wave, lane, steps, [&](int i, int st) { return st < count[0] ? w[0][i] + st * 64 : w[1][i] + (st - count[0]) * 64; },
            [&](int i, int st) { return st < count[0] ? x[0][i] + st * 64 : x[1][i] + (st - count[0]) * 64; }, acc);
    float* const mine = p.partial + (size_t)part * p.M * p.N;
    const int wn = wave / GM, wm = wave % GM, col = lane % 16, quarter = lane / 16;
#pragma unroll
    for (int b = 0; b < WM; ++b) {
        const int m = (wm * WM + b) * 16 + col;
        if (m >= p.M) continue;
#pragma unroll
        for (int a = 0; a < WN; ++a) {
            const int n = n0 + (wn * WN + a) * 16 + quarter * 4;
            const floatx4 v = acc[0][a][b] + acc[1][a][b];
            float* dst = mine + (size_t)m * p.N + n;
            if (n + 3 < p.N && p.N % 4 == 0) *reinterpret_cast<floatx4*>(dst) = v;
            else
                for (int i = 0; i < 4 && n + i < p.N; ++i) dst[i] = v[i];
        }
    }
}

template <int WN, int WM, int GN, int GM, int NS>
static int launch_few_rows(const KaFewRows& f, hipStream_t stream) {
    using T = KdTile<WN, WM, GN, GM, 64, NS, 16>;
    static bool configured = false;
    auto kernel = few_rows_kernel<WN, WM, GN, GM, NS>;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, T::SMEM);
        KA_CHECK(e == hipSuccess, "linear of few rows: cannot reserve %d bytes of LDS: %s", T::SMEM, hipGetErrorString(e));
        configured = true;
    }
    hipLaunchKernelGGL(kernel, dim3(ka_cdiv(ka_cdiv(f.N, T::BN), 8) * 8, f.parts), dim3(KA_WAVE * T::WAVES), T::SMEM, stream, f);
    KA_LAUNCH_CHECK();
    return 0;
}

// 1: done; 0: the operands are not covered (K in steps of 64); -1: an error.
int ka_few_rows_by_tiles(const KaFewRows& f, hipStream_t stream) {
    if (f.M < 1 || f.M > 64 || f.K[0] % 64 || f.K[1] % 64 || f.K[0] < 64 || f.parts < 1 || !f.partial) return 0;
    // Up to 32 rows tiles of 32, which ask for half the activations, six stages in the same LDS (us, 64 rows a tile and 32, at 24 rows: 2,560 by 2,560 + 10,240
    // 19.3 and 18.2, 2,048 by 2,048 + 8,192 14.6 and 14.1). Eight or twelve stages where a CU has one workgroup: 2 to 8 % slower at any number of rows.
    return (f.M <= 32 ? launch_few_rows<2, 1, 2, 2, 6>(f, stream) : launch_few_rows<2, 2, 2, 2, 5>(f, stream)) ? -1 : 1;
}

// The tile and the parts of K for `ka_linear_pair_tiles_bf16`.
//  * Tiles of 128 x 128: as many parts as leave the fewest K-steps to a CU, a part more than another costing the finishing kernel one more read
//    of the output (a K-step 0.55 us, eight of them a tile's start and end, 4 TB/s for the sums; 1.08 of that is measured on the average).
//  * The phased tiles of 256 x 256, and those of four waves (gemm_quad_pair_bf16.hip), where their estimate says so and their workgroups are one round of the
//    chip: a K-step takes `step` us with few workgroups and `full` more with one on every CU (the clock gives way under load), a workgroup's start and
//    end `edge` and `edge_full` more, a million sums `sums`. Fitted to timings of 65 to 2,048 rows, widths of 512 to 4,096, K of 1,536 to 20,480 in all:
//    off by 5 % on the average. The phased tiles give way only to an estimate 5 % below theirs: from some 1,300 rows on both take the same time, and theirs
//    is the shorter chain of sums (2,048, K = 10,240: 1,536 rows 75.3 and 74.6 us, 2,048 rows 88.6 and 90.2; 2,560, 12,800, 1,536 rows 100.8 and 105.5). Not
//    tiles of more than 128 rows where more than four tenths of them are none.
// Measured with the norm behind, what was chosen without the tiles of four waves and with them (us): N = 2,048, K = 10,240: 96 rows 21.3 and 19.5, 282 rows 29.3 and 27.5,
// 512 rows 38.1 and 34.0, 743 rows 48.8 and 44.4, 1,024 rows 58.2 and 51.9; 2,560, 12,800: 256 rows 36.0 and 35.0, 384 rows 47.2 and 45.4, 512 rows 52.2 and
// 47.6; 1,024, 5,120, 1,940 rows 37.9 and 33.9; 4,096, 14,336, 199 rows 43.5 and 40.9; 3,072, 13,312, 540 rows 67.8 and 59.0. Of 45 sizes drawn over that range
// 28 are faster, 17 go as before.
struct PairChoice {
    int tile, parts;        // tile 0: 128 x 128 (pair_tiles_kernel); else a tile of ka_pair_phased or ka_pair_quad; parts 0: none fits
    double us;
};

// How far ahead of the small tiles' the estimate of phased tiles of 256 x 256 that take `us` has to be (those of four waves: not at all) (0.99: 1 % behind will do). Both sides measured at 336 sizes where the estimates meet
// (512 to 4,096 wide, K of 2,560 to 20,480, their ratio 0.93 to 1.03):
//  * Short ones are up to 20 % slower, their start and end being more than the estimate has (1,024, 5,120, 769 rows 22.4 and 26.1 us; 2,048, 4,096, 771 rows 28.6 and
//    30.3; 1,024, 8,192, 769 rows 28.7 and 31.1).
//  * Longer ones that this takes are 5 % faster on the average, up to 16 % (2,560, 12,800: 480 rows 55.4 and 48.2, 512 rows 57.3 and 50.0; 2,048, 12,800, 512
//    rows 47.6 and 41.0), and 3 % slower at most (768, 10,240, 1,049 rows 32.2 and 33.2; 3,072, 20,480, 309 rows 72.5 and 74.3).
//  * Rows that fill the last tile count for the phased ones (2,048, 10,240, 490 rows 36.4 and 35.1 at a ratio of 0.998; 1,536, 12,800, 513 rows 43.1 and 46.9 at 1.005).
static double pair_lead(int M, double us) {
    if (us < 33.0) return 1.05;
    return M * 10L >= ka_cdiv(M, 256) * 256 * 8L ? 0.99 : 1.01;
}

// large_only: the small tiles are not among what the caller can take; the phased ones then have to be well ahead of them.
static PairChoice pair_tiles_choice(int M, int N, int steps, long partial_floats, bool phased, bool large_only) {
    const int cus = ka_compute_units();
    PairChoice best = {0, 0, 0.0};
    const long small = (long)ka_cdiv(N, PT_TILE) * ka_cdiv(M, PT_TILE);
    for (int parts = 1; parts <= 8 && (long)parts * M * N <= partial_floats; ++parts) {
        const int per = ka_cdiv(steps, parts);
        if ((parts > 1 && per < 4) || ka_cdiv(steps, per) != parts) continue;
        const double rounds = (double)((small * parts + cus - 1) / cus);
        const double us = 1.08 * (rounds * (per + 8) * 0.55 + parts * (double)M * N * 8.0 / 4.0e6);
        if (best.parts == 0 || us < best.us) best = {0, parts, us};
    }
    static const struct { int tile, rows_w, rows_x; double step, full, edge, edge_full, sums; } tiles[] = {
        {1, 256, 256, 1.05, 0.51, 11.9, -8.6, 1.43}, {8, 128, 128, 0.47, 0.10, 6.0, 0.0, 1.3},  {5, 160, 128, 0.50, 0.20, 8.0, 0.0, 1.3},
        {10, 160, 192, 0.62, 0.24, 8.0, 0.0, 1.3},   {3, 128, 256, 0.66, 0.22, 8.0, 0.0, 1.3}, {12, 160, 256, 0.74, 0.33, 8.0, 0.0, 1.3}};
    PairChoice large = {0, 0, 0.0};
    for (const auto& t : tiles) {
        if (!phased || (t.rows_x > PT_TILE && M * 10L < ka_cdiv(M, t.rows_x) * t.rows_x * 6L)) continue;
        const long each = (long)ka_cdiv(N, t.rows_w) * ka_cdiv(M, t.rows_x);
        for (int parts = 1; parts <= 8 && each * parts <= cus && (long)parts * M * N <= partial_floats; ++parts) {
            const int per = ka_cdiv(steps, parts), last = steps - (parts - 1) * per;
            if (per < 4 || ka_cdiv(steps, per) != parts || last < 2 || (large_only && parts == 1 && t.tile != 1)) continue;
            const double load = (double)(each * parts) / cus * (each * parts) / cus;
            const double us = per * (t.step + t.full * load) + t.edge + t.edge_full * load + parts * (double)M * N * t.sums * 1e-6;
            if (large.parts == 0 || us < (large.tile == 1 && t.tile != 1 ? 0.95 : 1.0) * large.us) large = {t.tile, parts, us};
        }
    }
    if (large.parts && (best.parts == 0 || (large_only ? 1.05 : large.tile == 1 ? pair_lead(M, large.us) : 1.0) * large.us < best.us)) {
        best = large;
        best.us *= 1.05;               // (what the vendor library is compared with)
    }
    return best;
}

static bool pair_tiles_fit(int M, int N, int K1, int K2) {
    return M >= 1 && N >= 1 && N % 4 == 0 && K1 % PT_BK == 0 && K2 % PT_BK == 0 && K1 >= PT_BK && K2 >= PT_BK;
}

// Parts and tile (parts + PT_TILE_CODE * tile), 0: not covered. phased 0: without the phased tiles and those of four waves, whose offsets have to fit in 32 bits.
KA_API int ka_linear_pair_tiles_parts(int M, int N, int K1, int K2, long partial_floats, int phased) {
    if (!pair_tiles_fit(M, N, K1, K2)) return 0;
    const PairChoice c = pair_tiles_choice(M, N, (K1 + K2) / PT_BK, partial_floats, phased, false);
    return c.parts ? c.parts + PT_TILE_CODE * c.tile : 0;
}

// The same for outputs of more small tiles than a CU's worth: large tiles with K in parts where they are faster than two products of the vendor
// library and the norm behind them (its operations at 0.85 PFLOP/s, 8 us for two launches' starts and ends, 10 bytes an output at 4 TB/s). Measured,
// us, library and tiles: N = 2,048, K = 10,240: 1,536 rows 91.5 and 74, 2,048 rows 105.5 and 88.5; 2,560, 12,800: 1,280 rows 131 and 89.5, 2,048 rows
// 158 and 131; 2,560, 5,120: 2,048 rows 83 and 72; 4,096, 8,192: 2,048 rows 140 and 133; in one part 4,096 rows of the last 249 against 243.
KA_API int ka_linear_pair_large_parts(int M, int N, int K1, int K2, long partial_floats) {
    if (!pair_tiles_fit(M, N, K1, K2)) return 0;
    const PairChoice c = pair_tiles_choice(M, N, (K1 + K2) / PT_BK, partial_floats, true, true);
    const double library = 2.0 * M * N * (double)(K1 + K2) / 0.85e9 + 8.0 + (double)M * N * 10.0 / 4.0e6;
    return c.tile && c.parts > 1 && c.us < library ? c.parts + PT_TILE_CODE * c.tile : 0;
}

KA_API int ka_linear_pair_tiles_bf16(const void* A1, long lda1, int K1, const void* A2, long lda2, int K2, const void* W1, long ldw1,
                                     const float* bias1, const void* W2, long ldw2, const float* bias2, float* out, long ldo, int N,
                                     int accumulate, int M, int parts, float* partials, long partial_floats, const float* gamma,
                                     const float* beta, float eps, void* normed, int normed_dtype, long ldn, hipStream_t stream) {
    const char* who = "ka_linear_pair_tiles_bf16";
    KA_CHECK(M > 0 && N > 0 && N % 4 == 0, "%s: M=%d N=%d (N must be a multiple of 4)", who, M, N);
    KA_CHECK(K1 >= PT_BK && K2 >= PT_BK && K1 % PT_BK == 0 && K2 % PT_BK == 0, "%s: K must be multiples of %d, got %d and %d", who, PT_BK, K1, K2);
    KA_CHECK(lda1 % 8 == 0 && ldw1 % 8 == 0 && lda2 % 8 == 0 && ldw2 % 8 == 0 && lda1 >= K1 && ldw1 >= K1 && lda2 >= K2 && ldw2 >= K2,
             "%s: row strides must be multiples of 8 and >= K", who);
    KA_CHECK(((uintptr_t)A1 | (uintptr_t)A2 | (uintptr_t)W1 | (uintptr_t)W2 | (uintptr_t)out | (uintptr_t)partials) % 16 == 0,
             "%s: operands must be 16-byte aligned", who);
    KA_CHECK(((uintptr_t)bias1 | (uintptr_t)bias2) % 16 == 0 || !gamma, "%s: biases must be 16-byte aligned beside a norm", who);
    KA_CHECK(ldo >= N && ldo % 4 == 0, "%s: output stride %ld for N=%d", who, ldo, N);
    const int steps = (K1 + K2) / PT_BK, tile = parts / PT_TILE_CODE;
    parts %= PT_TILE_CODE;
    KA_CHECK(parts >= 1 && parts <= steps && partials && (long)parts * M * N <= partial_floats, "%s: %d parts of %d steps, %ld floats", who, parts, steps,
             partial_floats);
    KaPairTiles p;
    p.A[0] = (const bf16_t*)A1; p.lda[0] = lda1; p.W[0] = (const bf16_t*)W1; p.ldw[0] = ldw1; p.steps[0] = K1 / PT_BK;
    p.A[1] = (const bf16_t*)A2; p.lda[1] = lda2; p.W[1] = (const bf16_t*)W2; p.ldw[1] = ldw2; p.steps[1] = K2 / PT_BK;
    p.M = M; p.N = N;
    p.per = ka_cdiv(steps, parts);
    parts = ka_cdiv(steps, p.per);
    p.partial = partials;
    if (tile ? ka_pair_phased(p, tile, parts, stream) : launch_pair_tiles<1, 2, 4, 2, PT_STAGES, 2>(p, parts, stream)) return -1;
    if (gamma) {
        const KaThenNorm then = {gamma, beta, eps, normed, normed_dtype, ldn};
        KA_CHECK(ka_then_norm_fits(N) && normed && ldn >= N && ldn % 4 == 0, "%s: cannot normalise rows of %d", who, N);
        ka_launch_finish_norm(M, N, stream, partials, parts, bias1, bias2, out, ldo, accumulate, then);
    } else {
        hipLaunchKernelGGL(ka_partials_finish_kernel, dim3(ka_cdiv((long)M * (N / 4), 256)), dim3(256), 0, stream, partials, parts, bias1, bias2,
                           out, KA_F32, ldo, M, N, KA_ACT_NONE, accumulate);
    }
    KA_LAUNCH_CHECK();
    return 0;
}

template <int NT, int MT, int BK>
static int launch_config(const bf16_t* A, long lda, const bf16_t* W, long ldw, const float* bias, void* out,
                         int out_dtype, long ldo, int M, int N, int K, int act, int accumulate,
                         hipStream_t stream) {
    static bool configured = false;
    constexpr int smem = gb_smem(NT, MT, BK);
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_bf16_kernel<NT, MT, BK>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        KA_CHECK(e == hipSuccess, "ka_linear_tiled_bf16: cannot reserve %d bytes of LDS: %s", smem, hipGetErrorString(e));
        configured = true;
    }
    int tiles_n = ka_cdiv(N, 64 * NT), tiles_m = ka_cdiv(M, 64 * MT);
    long total = (long)tiles_n * tiles_m;
    long launched = ((total + 7) / 8) * 8;
    KA_CHECK(launched < (1L << 31), "ka_linear_tiled_bf16: too many tiles");
    hipLaunchKernelGGL((gemm_bf16_kernel<NT, MT, BK>), dim3((unsigned)launched), dim3(GB_THREADS), smem, stream, A, lda,
                       W, ldw, bias, out, out_dtype, ldo, M, N, K, act, accumulate, tiles_n, tiles_m);
    return 0;
}

// `config`: 0 chooses by size; other values force a tile (for measurements and tests), with
// 1000000 * parts added to force K to be cut into that many parts as well. `partials`: scratch
// memory for the sums of such parts (null: K is never cut).
KA_API int ka_linear_tiled_bf16(const void* A, long lda, const void* W, long ldw, const float* bias,
                                void* out, int out_dtype, long ldo, int M, int N, int K, int act,
                                int accumulate, int config, float* partials, long partial_floats,
                                hipStream_t stream) {
    KA_CHECK(M > 0 && N > 0 && K > 0 && K % 8 == 0, "ka_linear_tiled_bf16: M=%d N=%d K=%d (K must be a multiple of 8)", M, N, K);
    KA_CHECK(lda % 8 == 0 && ldw % 8 == 0 && lda >= K && ldw >= K, "ka_linear_tiled_bf16: row strides must be multiples of 8 and >= K");
    KA_CHECK(((uintptr_t)A % 16 == 0) && ((uintptr_t)W % 16 == 0), "ka_linear_tiled_bf16: operands must be 16-byte aligned");
    KA_CHECK(ka_act_known(act), "ka_linear_tiled_bf16: unknown activation %d", act);
    KA_CHECK(ldo >= ka_act_outputs(act, N), "ka_linear_tiled_bf16: output stride too small");
    KA_CHECK(!ka_act_gated(act) || (N % 2 == 0 && !accumulate), "ka_linear_tiled_bf16: a gated linear needs an even N and no accumulation");
    KA_CHECK(out_dtype == KA_F32 || out_dtype == KA_BF16, "ka_linear_tiled_bf16: bad output type");
    KA_CHECK(!(accumulate && out_dtype != KA_F32), "ka_linear_tiled_bf16: accumulate needs an fp32 output");
    KA_CHECK((uintptr_t)out % 16 == 0, "ka_linear_tiled_bf16: output must be 16-byte aligned");
    int parts = config >= 1000000 ? config / 1000000 : 0;      // 0: chosen below
    config %= 1000000;
    if (ka_act_gated(act) && config != 211 && config != 221) {
        // the pairs of a gated linear meet in the epilogue of the tiles that are staged through registers (the
        // large tiles write their outputs as whole rows through LDS, laid out for N columns)
        config = (long)ka_cdiv(N, 128) * ka_cdiv(M, 128) >= 512 ? 221 : 211;
        parts = 0;
    }
    if (config == 0) {
        if (K % 64 == 0) {
            // Tiles of 128 x 128 read 64 flops' worth of operands per byte from L2, which is what
            // bounds them (measured: 11 TB/s of L2 traffic at 800 TFLOP/s); 256 x 256 halves that
            // and wins where its tiles fill most of the CUs in every round (measured inside the
            // model at 2048 rows: N = 6144 and 8192). Where 128 x 128 tiles leave a CU with one
            // workgroup only, eight waves and three stages hide the trip to HBM that two
            // workgroups would otherwise hide for each other (N = 2048: 35 us of 120 at K = 8192).
            const int cus = ka_compute_units();
            long t256 = (long)ka_cdiv(N, 256) * ka_cdiv(M, 256);
            long t128 = (long)ka_cdiv(N, 128) * ka_cdiv(M, 128);
            long rounds = (t256 + cus - 1) / cus;
            // (192 x 256 where its tiles fill the CUs and those of 256 x 256 do not: N = 6144 at
            // 2048 rows is 192 tiles of the one, 256 of the other; measured 7 us of 74 faster)
            long t192 = (long)ka_cdiv(N, 192) * ka_cdiv(M, 256);
            long rounds192 = (t192 + cus - 1) / cus;
            if (t192 * 10 >= rounds192 * cus * 7 && t192 * rounds * 10 > t256 * rounds192 * 11) config = 22232;
            else if (t256 * 10 >= rounds * cus * 7) config = 22224;
            else if (t128 <= cus) {
                config = 23212;
                // Few tiles (a few hundred rows of a narrow output): K is cut into parts so that
                // about every CU gets a workgroup; a second kernel adds the parts up.
                if (parts == 0 && partials && t128 * 2 <= cus && K >= 1024) {
                    parts = (int)(cus / t128);
                    if (parts > K / 512) parts = K / 512;
                    if (parts > 8) parts = 8;
                }
            } else config = 12222;
        } else {
            long t22 = (long)ka_cdiv(N, 128) * ka_cdiv(M, 128);
            config = t22 >= 512 ? 221 : 211;
        }
    }
    const bf16_t* a = (const bf16_t*)A;
    const bf16_t* w = (const bf16_t*)W;
    int rc;
    if (parts >= 2 && config == 23212 && K % 64 == 0) {
        int k_per = ka_cdiv(ka_cdiv(K, parts), 64) * 64;
        parts = ka_cdiv(K, k_per);
        if (parts >= 2 && partials && (long)parts * M * N <= partial_floats) {
            rc = launch_dma<1, 2, 4, 2, 64, 3, 4>(a, lda, w, ldw, nullptr, partials, KA_F32, N, M, N, K, 0, 0, stream, parts, k_per);
            if (rc) return rc;
            KA_LAUNCH_CHECK();
            const int quads = M * ka_cdiv(N, 4);
            hipLaunchKernelGGL(ka_partials_finish_kernel, dim3(ka_cdiv(quads, 256)), dim3(256), 0, stream, partials, parts,
                               bias, (const float*)nullptr, out, out_dtype, ldo, M, N, act, accumulate);
            KA_LAUNCH_CHECK();
            return 0;
        }
    }
    switch (config) {
        case 221: rc = launch_config<2, 2, 64>(a, lda, w, ldw, bias, out, out_dtype, ldo, M, N, K, act, accumulate, stream); break;
        case 211: rc = launch_config<2, 1, 64>(a, lda, w, ldw, bias, out, out_dtype, ldo, M, N, K, act, accumulate, stream); break;
#define KA_DMA(CODE, WNV, WMV, GNV, GMV, BKV, NSV, SLV)                                                               \
        case CODE:                                                                                                \
            KA_CHECK(K % BKV == 0, "ka_linear_tiled_bf16: this tile needs K to be a multiple of %d", BKV);        \
            rc = launch_dma<WNV, WMV, GNV, GMV, BKV, NSV, SLV>(a, lda, w, ldw, bias, out, out_dtype, ldo, M, N, K, act, accumulate, stream); \
            break;
        // 10000 (four waves, 2 x 2) or 20000 (eight waves, 4 x 2) + stages * 1000 + (K-step / 32) * 100 + wave tile
        KA_DMA(12222, 2, 2, 2, 2, 64, 2, 2)      // 128 x 128, two workgroups per CU
        KA_DMA(23212, 1, 2, 4, 2, 64, 3, 4)      // 128 x 128 by eight waves, three stages: for one workgroup per CU
        KA_DMA(22224, 2, 4, 4, 2, 64, 2, 1)      // 256 x 256, one workgroup of eight waves per CU
        KA_DMA(22232, 3, 2, 2, 4, 64, 2, 1)      // 192 x 256 (N x M), eight waves: for an N that 256 leaves CUs idle with
        KA_DMA(13122, 2, 2, 2, 2, 32, 3, 2)      // (slower everywhere; kept as the test of K-steps of 32)
#undef KA_DMA
        default: KA_CHECK(false, "ka_linear_tiled_bf16: unknown tile configuration %d", config);
    }
    if (rc) return rc;
    KA_LAUNCH_CHECK();
    return 0;
}
