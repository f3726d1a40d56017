// Generic linear layer: out = act(A W^T + bias) or out += A W^T + bias.
//
// Four kernels, each with an order of a sum that K alone fixes:
//  * any M, N, K, any mix of fp32 and bf16 operands: plain FMA in fp32 with an LDS-tiled 64x64x16 block, k = 0..K-1 in that
//    order; the fallback of the bf16 path;
// and, of aligned fp32 operands, the true 32-bit path,
//  * up to 16 rows of a linear without a gate: a stream of weights (gemv_f32_kernel);
//  * else K in steps of 32: the matrix pipes, every number as three of bf16 (gemm_f32_split_kernel);
//  * else wider FMA tiles, k in ascending order as the first (gemm_f32_kernel).
// So a row's result does not depend on what else is in the batch, but for the step from 16 to 17 rows without a gate.
#include "ka_common.h"
#include "ka_dma_tiles.h"

constexpr int GT = 64;   // tile edge in M and N
constexpr int GK = 16;   // tile depth

template <typename TA, typename TW, typename TOut>
__global__ void __launch_bounds__(256)
gemm_generic_kernel(const TA* __restrict__ A, long lda, const TW* __restrict__ W, long ldw,
                    const float* __restrict__ bias, TOut* __restrict__ out, long ldo, int M, int N,
                    int K, int act, int accumulate) {
    __shared__ float As[GK][GT + 4];
    __shared__ float Ws[GK][GT + 4];
    int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    int m0 = blockIdx.y * GT, n0 = blockIdx.x * GT;
    float acc[4][4] = {};
    // Each thread loads 4 elements of each operand tile: row = tid / 4, k = (tid % 4) * 4 .. +4.
    int lr = threadIdx.x / 4, lk = (threadIdx.x % 4) * 4;
    for (int k0 = 0; k0 < K; k0 += GK) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            int k = k0 + lk + j;
            int m = m0 + lr, n = n0 + lr;
            As[lk + j][lr] = (m < M && k < K) ? ka_to_float(A[(size_t)m * lda + k]) : 0.f;
            Ws[lk + j][lr] = (n < N && k < K) ? ka_to_float(W[(size_t)n * ldw + k]) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < GK; ++k) {
            float a[4], w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[k][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] = Ws[k][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], w[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        int m = m0 + ty * 4 + i;
        if (m >= M) continue;
        if (ka_act_gated(act)) {           // pairs of neighbouring columns make one output
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = acc[i][j] + (bias && n0 + tx * 4 + j < N ? bias[n0 + tx * 4 + j] : 0.f);
            ka_gated_store<false, 4>(out, sizeof(TOut) == 4 ? KA_F32 : KA_BF16, ldo, m, n0 + tx * 4, N, v, act);
            continue;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            int n = n0 + tx * 4 + j;
            if (n >= N) continue;
            float v = acc[i][j] + (bias ? bias[n] : 0.f);
            if (act) v = ka_activate(act, v);
            size_t o = (size_t)m * ldo + n;
            if (accumulate) v += ka_to_float(out[o]);
            out[o] = ka_from_float<TOut>(v);
        }
    }
}

// Many rows in fp32 where K is a multiple of 32: products on the bf16 matrix pipes, which have sixteen times the rate of the fp32 ones. A number of 32 bits is
// the sum of three bf16 numbers to its last bit (24 bits of mantissa, eight in each: what rounding to the nearest leaves is representable, so
// both subtractions are exact), and w x = w1 x1 + (w1 x2 + w2 x1) + (w2 x2 + w1 x3 + w3 x1) + what is below 2^-25 of it: six products, each exact in the
// pipe, summed in fp32.
//
// Operands go straight from memory into swizzled LDS as in ka_dma_tiles.h, two steps of 16 numbers at a time (whole lines), and are split by the wave that
// multiplies them: 44 instructions per eight numbers a lane, laid between the products of the step before, which the compiler does only where each step is a
// region of its own with an end that names the parts (157 rows of 2,048 x 8,192 by tiles of 64 x 64: 96 us without, 83 with). At one wave a SIMD an instruction
// takes five cycles, so a step of 64 x 64 x 16 (24 products, some 225 other instructions) takes 1,400 where its products are 768: that is what bounds it. The
// activations' parts by a launch of their own, in front, were no faster: 10 KB a step instead of 8.
//
// The order of a sum is fixed by K alone. K is cut into F32_PARTS parts, each summed by a wave of its own (so no wave waits for another before the
// end): w1 x1 of 128 of K from zero, these sums in order, the five smaller products, whose roundings weigh 2^-8, in an accumulator beside them; the
// parts' sums meet in LDS and are added in their order. All tiles give the same bits.
//
// Weights that are bf16 numbers, as checkpoints hold them, have one part, and three of the six products are zeros: a wave begins its part with the other three, looks
// at the lower halves of the weights as it goes, and where it meets one that is not zero begins again with all six, to the same bits (282 rows as below:
// 51, 26, 75 and 75 us; weights that need all six pay for the first steps, 67, 31, 95 and 93).
//
// What three bf16 numbers cannot say (infinities, numbers beyond bf16's largest) leaves an infinity or NaN in the sum: such an output is summed again by
// plain FMA from memory. (Numbers below 2^-109 lose what is below 2^-133 of them.)
//
// Measured, us, fp32 products on the matrix pipes (v_mfma_f32_32x32x2_f32) -> here, 64 rows through 2,048 x 6,144, 2,048 x 2,048, 2,048 x
// 8,192 and 8,192 x 2,048 28.6, 16.4, 27.8 and 52.2 -> 25.0, 15.8, 27.4 and 47.3; 282 rows 85, 38, 105 and 131 -> 66, 30, 90 and 92; 2,048 rows 446, 162, 591 and 611
// -> 385, 134, 511 and 432. Error against 64 bits of such sums 1.35e-7 -> 8.7e-8, of K = 8,192 2.2e-7 -> 1.1e-7.
constexpr int F32_PARTS = 4;
constexpr int F32_STEP = 32;
constexpr int F32_BLOCK = 8;       // steps of 16 that are summed from zero

typedef __attribute__((ext_vector_type(2))) float gs_float2;
typedef __attribute__((ext_vector_type(2))) __bf16 gs_bf16x2;

// part[0] + part[1] + part[2] is the eight numbers of lo and hi to the last bit
__device__ __forceinline__ void gs_split(const floatx4& lo, const floatx4& hi, bf16x8 (&part)[3]) {
    uint4 out[3];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float a = i < 2 ? lo[2 * i] : hi[2 * i - 4], b = i < 2 ? lo[2 * i + 1] : hi[2 * i - 3];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            const unsigned pair = __builtin_bit_cast(unsigned, __builtin_convertvector(gs_float2{a, b}, gs_bf16x2));
            (i == 0 ? out[p].x : i == 1 ? out[p].y : i == 2 ? out[p].z : out[p].w) = pair;
            if (p == 2) break;
            a -= __uint_as_float(pair << 16);
            b -= __uint_as_float(pair & 0xffff0000u);
        }
    }
#pragma unroll
    for (int p = 0; p < 3; ++p) part[p] = __builtin_bit_cast(bf16x8, out[p]);
}

template <int WN, int WM, int NS>
__global__ void __launch_bounds__(KA_WAVE * F32_PARTS, WN * WM > 1 ? 1 : 2)
gemm_f32_split_kernel(const float* __restrict__ A, long lda, const float* __restrict__ W, long ldw, const float* __restrict__ bias,
                      float* __restrict__ out, long ldo, int M, int N, int K, int act, int accumulate, int tiles_n, int tiles_m) {
    constexpr int BN = 32 * WN, BM = 32 * WM, STEP = 16;
    constexpr int ROW = STEP * 4, CPR = ROW / 16, RPL = KA_WAVE / CPR, STAGE = (BN + BM) * ROW;
    constexpr int W_LOADS = BN / RPL, X_LOADS = BM / RPL, LPW = W_LOADS + X_LOADS;
    extern __shared__ __attribute__((aligned(16))) unsigned char gf_lds[];
    const int total = tiles_n * tiles_m, per_xcd = (total + 7) / 8;
    const int logical = blockIdx.x % 8 * per_xcd + blockIdx.x / 8;
    if (logical >= total || (int)blockIdx.x / 8 >= per_xcd) return;
    const int n0 = logical / tiles_m * BN, m0 = logical % tiles_m * BM;
    const int part = __builtin_amdgcn_readfirstlane(threadIdx.x / KA_WAVE), lane = threadIdx.x % KA_WAVE;
    const int li = lane % 32, lg = lane / 32;
    const float* wsrc[W_LOADS];
    const float* xsrc[X_LOADS];
    const int part_steps = ((K + F32_PARTS - 1) / F32_PARTS + F32_STEP - 1) / F32_STEP * (F32_STEP / STEP), k_steps = K / STEP;
    const int first = part * part_steps, steps = max(0, min(part_steps, k_steps - first));
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i) {
        const int r = kd_load_row<CPR>(i, lane);
        wsrc[i] = W + (size_t)min(n0 + r, N - 1) * ldw + kd_load_channel<CPR>(r, lane) / 2 + first * STEP;      // (four numbers a piece)
    }
#pragma unroll
    for (int i = 0; i < X_LOADS; ++i) {
        const int r = kd_load_row<CPR>(i, lane);
        xsrc[i] = A + (size_t)min(m0 + r, M - 1) * lda + kd_load_channel<CPR>(r, lane) / 2 + first * STEP;
    }
    unsigned char* mine = gf_lds + part * NS * STAGE;
    auto fetch = [&](int step) {
        unsigned char* base = mine + step % NS * STAGE;
#pragma unroll
        for (int i = 0; i < W_LOADS; ++i)
            __builtin_amdgcn_global_load_lds((const GD_GLOBAL void*)(wsrc[i] + step * STEP), (GD_LDS void*)(base + i * RPL * ROW), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < X_LOADS; ++i)
            __builtin_amdgcn_global_load_lds((const GD_GLOBAL void*)(xsrc[i] + step * STEP), (GD_LDS void*)(base + BN * ROW + i * RPL * ROW), 16, 0, 0);
    };
    const int swz = kd_swizzle<CPR>(li);
    floatx16 acc[WN][WM], few[WN][WM], low[WN][WM];
    auto clear = [&] {
#pragma unroll
        for (int a = 0; a < WN; ++a)
#pragma unroll
            for (int b = 0; b < WM; ++b)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[a][b][v] = few[a][b][v] = low[a][b][v] = 0.f;
    };
    clear();
    bf16x8 op[2][WN + WM][3];
    // the operands of a step from LDS, split (the step's loads have landed; a wave reads what it asked for itself: no barrier)
    unsigned seen = 0;                                                         // bits of the weights that were read
    auto operands = [&](auto slot_c, auto whole_c, int step) __attribute__((always_inline)) {
        constexpr int slot = decltype(slot_c)::value;
        constexpr bool WHOLE = decltype(whole_c)::value;
        const unsigned char* base = mine + step % NS * STAGE;
        floatx4 raw[WN + WM][2];
#pragma unroll
        for (int r = 0; r < WN + WM; ++r)
#pragma unroll
            for (int h = 0; h < 2; ++h) raw[r][h] = *reinterpret_cast<const floatx4*>(base + (r * 32 + li) * ROW + ((h * 2 + lg) ^ swz) * 16);
#pragma unroll
        for (int r = 0; r < WN + WM; ++r) {
            if (WHOLE || r >= WN) {
                gs_split(raw[r][0], raw[r][1], op[slot][r]);
                continue;
            }
            uint4 upper;
            const uint4 lo = __builtin_bit_cast(uint4, raw[r][0]), hi = __builtin_bit_cast(uint4, raw[r][1]);
            upper.x = __builtin_amdgcn_perm(lo.y, lo.x, 0x07060302);
            upper.y = __builtin_amdgcn_perm(lo.w, lo.z, 0x07060302);
            upper.z = __builtin_amdgcn_perm(hi.y, hi.x, 0x07060302);
            upper.w = __builtin_amdgcn_perm(hi.w, hi.z, 0x07060302);
            op[slot][r][0] = __builtin_bit_cast(bf16x8, upper);
            seen |= lo.x | lo.y | lo.z | lo.w | hi.x | hi.y | hi.z | hi.w;
        }
    };
    // Step s, the place-th of four: its products, and between them the split of the next one's operands, which the matrix pipe does not need.
    // STEADY: a step that has NS behind it.
    auto step = [&](auto place_c, auto steady_c, auto whole_c, int s) __attribute__((always_inline)) {
        constexpr bool WHOLE = decltype(whole_c)::value;
        constexpr int place = decltype(place_c)::value, slot = place & 1;
        constexpr bool STEADY = decltype(steady_c)::value;
        if constexpr (slot == 1) {                                             // the last step of a pair
            if constexpr (STEADY) gd_wait_loads<2 * LPW * (NS / 2 - 2)>();
            else if (s + 1 < steps) gd_wait_younger<2 * LPW, NS / 2 - 2>(min(NS / 2 - 2, (steps - 1 - s) / 2 - 1));
            gd_wait_lds();                                                     // own reads of the pair are in registers: its stages may be written
            if (STEADY || s + NS < steps) {
                fetch(s + NS - 1);
                fetch(s + NS);
            }
        }
        operands(std::integral_constant<int, slot ^ 1>{}, whole_c, s + 1);              // (behind the last step: memory that nobody uses)
        auto add = [&](floatx16 (&sum)[WN][WM], int i, int j) {
#pragma unroll
            for (int a = 0; a < WN; ++a)
#pragma unroll
                for (int b = 0; b < WM; ++b) sum[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op[slot][a][i], op[slot][WN + b][j], sum[a][b], 0, 0, 0);
        };
        add(low, 0, 2);
        if constexpr (WHOLE) add(low, 2, 0);
        add(few, 0, 0);
        if constexpr (WHOLE) add(low, 1, 1);
        add(low, 0, 1);
        if constexpr (WHOLE) add(low, 1, 0);
        constexpr int PRODUCTS = (WHOLE ? 6 : 3) * WN * WM, EACH = ((WHOLE ? 44 : 8) * WN + 44 * WM + PRODUCTS - 1) / PRODUCTS;
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * (WN + WM), 0);
        gd_static_for<0, PRODUCTS>([&](auto) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, EACH, 0);
        });
        // (the split belongs here: the compiler would put it off to the step that uses it, in front of that step's products)
#pragma unroll
        for (int r = 0; r < WN + WM; ++r)
#pragma unroll
            for (int i = 0; i < (WHOLE || r >= WN ? 3 : 1); ++i) asm volatile("" : "+v"(op[slot ^ 1][r][i]));
        __builtin_amdgcn_sched_barrier(0);
    };
    auto settle = [&] {
#pragma unroll
        for (int a = 0; a < WN; ++a)
#pragma unroll
            for (int b = 0; b < WM; ++b) {
                acc[a][b] += few[a][b];
#pragma unroll
                for (int v = 0; v < 16; ++v) few[a][b][v] = 0.f;
            }
    };
    // Whether every weight of the part was a bf16 number; a part that meets another ends early and is begun again with all six products.
    auto multiply = [&](auto whole_c) __attribute__((always_inline)) {
        constexpr bool WHOLE = decltype(whole_c)::value;
#pragma unroll
        for (int st = 0; st < NS; ++st)
            if (st < steps) fetch(st);
        gd_wait_younger<2 * LPW, NS / 2 - 1>(min(NS / 2, steps / 2) - 1);
        operands(std::integral_constant<int, 0>{}, whole_c, 0);
        int s = 0;
        auto block = [&](auto steady_c) __attribute__((always_inline)) {
            step(std::integral_constant<int, 0>{}, steady_c, whole_c, s);
            step(std::integral_constant<int, 1>{}, steady_c, whole_c, s + 1);
            step(std::integral_constant<int, 2>{}, steady_c, whole_c, s + 2);
            step(std::integral_constant<int, 3>{}, steady_c, whole_c, s + 3);
            s += 4;
            if (s % F32_BLOCK == 0) settle();
        };
        auto narrow = [&] { return WHOLE || __builtin_amdgcn_ballot_w64((seen & 0xffff) != 0) == 0; };
        while (s + 3 + NS < steps && narrow()) block(std::true_type{});
        while (s + 3 < steps && narrow()) block(std::false_type{});
        if (s < steps && narrow()) {                                           // (an even number of steps)
            step(std::integral_constant<int, 0>{}, std::false_type{}, whole_c, s);
            step(std::integral_constant<int, 1>{}, std::false_type{}, whole_c, s + 1);
        }
        settle();
        return narrow();
    };
    if (steps > 0 && !multiply(std::false_type{})) {
        gd_wait_loads<0>();                                                    // (what was asked for ahead lands in stages that are written again)
        gd_wait_lds();
        clear();
        multiply(std::true_type{});
    }
    // acc[a][b][v] is out[m][n] with n = n0 + a 32 + (v / 4) 8 + lg 4 + v % 4 and m = m0 + b 32 + li
    const bool vectors = N % 4 == 0 && ldo % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
    auto store = [&](int a, int b, int q, const floatx4& y) {
        const int m = m0 + b * 32 + li, n = n0 + a * 32 + q * 8 + lg * 4;
        if (m >= M || n >= N) return;
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[j] = y[j];
            if (!(fabsf(v[j]) < INFINITY) && n + j < N) {                      // (see above)
                v[j] = 0.f;
                for (int k = 0; k < K; ++k) v[j] = fmaf(A[(size_t)m * lda + k], W[(size_t)(n + j) * ldw + k], v[j]);
            }
            v[j] += bias && n + j < N ? bias[n + j] : 0.f;
        }
        if (ka_act_gated(act)) {
            ka_gated_store<false, 4>(out, KA_F32, ldo, m, n, N, v, act);
            return;
        }
        if (act)
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = ka_activate(act, v[j]);
        float* op = out + (size_t)m * ldo + n;
        if (vectors) {
            floatx4 r = {v[0], v[1], v[2], v[3]};
            if (accumulate) r = *reinterpret_cast<const floatx4*>(op) + r;
            *reinterpret_cast<floatx4*>(op) = r;
        } else {
            for (int j = 0; j < 4 && n + j < N; ++j) op[j] = accumulate ? op[j] + v[j] : v[j];
        }
    };
    // the parts' sums through LDS; every wave finishes a quarter of the tile's numbers
    gd_wait_lds();
    gd_barrier();
    floatx4* sums = reinterpret_cast<floatx4*>(gf_lds);
    gd_static_for<0, WN * WM * 4>([&](auto ic) {
        constexpr int i = decltype(ic)::value, a = i / (4 * WM), b = i / 4 % WM, q = i % 4;
        floatx4 y;
#pragma unroll
        for (int j = 0; j < 4; ++j) y[j] = acc[a][b][q * 4 + j] + low[a][b][q * 4 + j];
        sums[(part * WN * WM * 4 + i) * KA_WAVE + lane] = y;
    });
    gd_wait_lds();
    gd_barrier();
    const int parts = (k_steps + part_steps - 1) / part_steps;                 // (those that hold anything)
    for (int i = 0; i < WN * WM; ++i) {
        const int at = i * 4 + part;
        floatx4 y = sums[at * KA_WAVE + lane];
        for (int p = 1; p < parts; ++p) y += sums[(p * WN * WM * 4 + at) * KA_WAVE + lane];
        store(i / WM, i % WM, part, y);
    }
}

template <int WN, int WM, int NS>
static int launch_f32_split(const float* A, long lda, const float* W, long ldw, const float* bias, float* out, long ldo, int M, int N, int K,
                            int act, int accumulate, hipStream_t stream) {
    constexpr int BN = 32 * WN, BM = 32 * WM, smem = F32_PARTS * NS * (BN + BM) * 64;
    static_assert(smem >= F32_PARTS * WN * WM * 4 * KA_WAVE * 16, "the parts' sums fit");
    static bool configured = false;
    auto kernel = gemm_f32_split_kernel<WN, WM, NS>;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        KA_CHECK(e == hipSuccess, "ka_linear_generic: cannot reserve %d bytes of LDS: %s", smem, hipGetErrorString(e));
        configured = true;
    }
    const int tiles_n = ka_cdiv(N, BN), tiles_m = ka_cdiv(M, BM);
    const long blocks = ((long)tiles_n * tiles_m + 7) / 8 * 8;
    KA_CHECK(blocks < (1L << 31), "ka_linear_generic: too many tiles");
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(KA_WAVE * F32_PARTS), smem, stream, A, lda, W, ldw, bias, out, ldo, M, N, K, act,
                       accumulate, tiles_n, tiles_m);
    KA_LAUNCH_CHECK();
    return 0;
}

// The tile: the one that is done first by what was measured (us per 2,048 of K: a first part, and as much again for every round of one tile a CU); all give the
// same bits. Tiles of 32 x 32 leave room for two workgroups a CU, or for eight stages instead of four where no CU has two and K is long (2,048 of 8,192, 17
// and 96 rows: 49.2 and 48.7 us with four, 43.1 and 46.4 with eight; K of 2,048 the same). Measured, us per 2,048 of K, tiles a CU rounded up (17 to 2,048 rows
// of 2,048 x 2,048, 6,144 x 2,048 and 8,192 x 2,048):
//              1      2      3     4     7     8    12    16
//   64 x 64    30     60     90   122         254   387   509
//   64 x 32    22     38           78         161
//   32 x 32    16     25     34    43    73    88
static int launch_f32_best(const float* A, long lda, const float* W, long ldw, const float* bias, float* out, long ldo, int M, int N, int K,
                           int act, int accumulate, hipStream_t stream) {
    const int cus = ka_compute_units();
    auto rounds = [&](int bn, int bm) { return (float)((((long)ka_cdiv(N, bn) * ka_cdiv(M, bm)) + cus - 1) / cus); };
    const float t64 = 30.5f * rounds(64, 64), t32 = 1.f + 20.f * rounds(64, 32), t1 = 6.f + 9.6f * rounds(32, 32);
#define KA_F32(...) return launch_f32_split<__VA_ARGS__>(A, lda, W, ldw, bias, out, ldo, M, N, K, act, accumulate, stream)
    if (t64 <= t32 && t64 <= t1) KA_F32(2, 2, 4);
    if (t32 <= t1) KA_F32(2, 1, 4);
    if (rounds(32, 32) <= 1.f && K >= 4096) KA_F32(1, 1, 8);
    KA_F32(1, 1, 4);
#undef KA_F32
}

// Many rows in fp32 (prompts on the 32-bit path): the same sums, k in ascending order for every
// output, from a tile of 128 x 128 x 8 with 8 x 8 outputs a thread, 16-byte loads (rows and K
// must allow them: the host sends everything else to the kernel above) and two LDS stages.
constexpr int GF = 128;   // tile edge in M and N
constexpr int GFK = 8;    // tile depth

// (RM: output rows a thread holds, 8 or 4: tiles of 128 or 64 rows; the lower tile doubles the
// workgroups of a narrow output that would otherwise leave CUs with one or none)
template <int RM>
__global__ void __launch_bounds__(256)
gemm_f32_kernel(const float* __restrict__ A, long lda, const float* __restrict__ W, long ldw,
                const float* __restrict__ bias, float* __restrict__ out, long ldo, int M, int N, int K, int act,
                int accumulate) {
    typedef __attribute__((ext_vector_type(4))) float f4;
    constexpr int TM = 16 * RM;
    __shared__ __attribute__((aligned(16))) float As[2][GFK][TM + 4];
    __shared__ __attribute__((aligned(16))) float Ws[2][GFK][GF + 4];
    const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    const int m0 = blockIdx.y * TM, n0 = blockIdx.x * GF;
    // each thread brings four consecutive k of one row of each operand tile (rows past the end
    // are the last row again: their outputs are never stored)
    const int lr = threadIdx.x / 2, lk = (threadIdx.x % 2) * 4;
    const bool brings_a = lr < TM;
    const float* arow = A + (size_t)min(m0 + min(lr, TM - 1), M - 1) * lda + lk;
    const float* wrow = W + (size_t)min(n0 + lr, N - 1) * ldw + lk;
    const f4 zero = {0.f, 0.f, 0.f, 0.f};
    auto fetch = [&](int k0, f4& ra, f4& rw) {
        const bool ok = k0 + lk < K;             // K is a multiple of 4
        ra = ok ? *reinterpret_cast<const f4*>(arow + k0) : zero;
        rw = ok ? *reinterpret_cast<const f4*>(wrow + k0) : zero;
    };
    auto stash = [&](int buf, const f4& ra, const f4& rw) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (brings_a) As[buf][lk + j][lr] = ra[j];
            Ws[buf][lk + j][lr] = rw[j];
        }
    };
    float acc[RM][8] = {};
    f4 ra, rw;
    fetch(0, ra, rw);
    stash(0, ra, rw);
    __syncthreads();
    const int steps = (K + GFK - 1) / GFK;
    for (int s = 0; s < steps; ++s) {
        const int buf = s & 1;
        if (s + 1 < steps) fetch((s + 1) * GFK, ra, rw);
#pragma unroll
        for (int k = 0; k < GFK; ++k) {
            float a[RM];
#pragma unroll
            for (int i = 0; i < RM; i += 4) {
                const f4 v = *reinterpret_cast<const f4*>(&As[buf][k][ty * RM + i]);
#pragma unroll
                for (int u = 0; u < 4; ++u) a[i + u] = v[u];
            }
            const f4 w0 = *reinterpret_cast<const f4*>(&Ws[buf][k][tx * 8]), w1 = *reinterpret_cast<const f4*>(&Ws[buf][k][tx * 8 + 4]);
#pragma unroll
            for (int i = 0; i < RM; ++i)
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[i][j] = fmaf(a[i], j < 4 ? w0[j] : w1[j - 4], acc[i][j]);
        }
        if (s + 1 < steps) stash(buf ^ 1, ra, rw);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < RM; ++i) {
        const int m = m0 + ty * RM + i;
        if (m >= M) continue;
        if (ka_act_gated(act)) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = acc[i][j] + (bias && n0 + tx * 8 + j < N ? bias[n0 + tx * 8 + j] : 0.f);
            ka_gated_store<false, 8>(out, KA_F32, ldo, m, n0 + tx * 8, N, v, act);
            continue;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int n = n0 + tx * 8 + j;
            if (n >= N) continue;
            float v = acc[i][j] + (bias ? bias[n] : 0.f);
            if (act) v = ka_activate(act, v);
            const size_t o = (size_t)m * ldo + n;
            out[o] = accumulate ? out[o] + v : v;
        }
    }
}

// Few rows in fp32 (decoding on the 32-bit path): the tiles above would put a sixteenth of their threads to work and read every
// weight through LDS. Here a wave owns C output columns: its lanes walk over K with 16-byte loads of the weight rows and of each
// activation row, every lane adds up its own k in their order, and the lanes' sums meet in a fixed tree. The order of a sum
// is the same for every M and N.
//
// What bounds it is the stream of weights. Four steps of it are asked for at once (without a branch between them: the loads of a
// loop over the rows that are there are not hoisted over each other), and a step's activations, which come from the CU's cache,
// serve all C columns. Measured, us, before -> now, three rows through 2,048 x 6,144, 2,048 x 2,048, 2,048 x 8,192, 8,192 x 2,048 and the
// head of 2,048 x 51,200: 14.3, 11.0, 23.5, 35.8 and 124 -> 12.7, 6.7, 16.5, 19.6 and 79; one row 11.1, 8.9, 15.7, 22.4 and 78 -> 10.1,
// 4.6, 12.6, 12.5 (5.4 TB/s) and 64. Forms for exactly three and for six rows (instead of four and eight, one or two of them read for nothing): three rows
// of 8,192 x 2,048 19.3 -> 16.7, 2,048 x 8,192 16.3 -> 15.8; six 22.6 -> 21.8, 19.3 -> 18.2.
constexpr int GV_ROWS = 16;      // most rows
constexpr int GV_WAVES = 4;      // waves per workgroup

typedef __attribute__((ext_vector_type(4))) float gv_float4;

template <int MB, int C>
__global__ void __launch_bounds__(GV_WAVES * KA_WAVE)
gemv_f32_kernel(const float* __restrict__ A, long lda, const float* __restrict__ W, long ldw,
                const float* __restrict__ bias, float* __restrict__ out, long ldo, int M, int N, int K, int act,
                int accumulate) {
    constexpr int STEP = KA_WAVE * 4, U = 4;
    constexpr int UA = MB <= 4 ? U : MB <= 8 ? 2 : 1;        // steps whose activations are asked for at once
    const int wave = threadIdx.x / KA_WAVE, lane = threadIdx.x % KA_WAVE;
    const int n0 = (blockIdx.x * GV_WAVES + wave) * C;
    if (n0 >= N) return;
    const float* w[C];
#pragma unroll
    for (int c = 0; c < C; ++c) w[c] = W + (size_t)min(n0 + c, N - 1) * ldw + lane * 4;       // (columns past the end: not stored)
    const float* a[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) a[m] = A + (size_t)min(m, M - 1) * lda + lane * 4;           // (rows past the end: not stored)
    float acc[C][MB];
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int m = 0; m < MB; ++m) acc[c][m] = 0.f;
    auto add = [&](const gv_float4 (&x)[C], const gv_float4 (&y)[MB]) {
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int c = 0; c < C; ++c)
                acc[c][m] = fmaf(y[m][3], x[c][3], fmaf(y[m][2], x[c][2], fmaf(y[m][1], x[c][1], fmaf(y[m][0], x[c][0], acc[c][m]))));
    };
    int k = 0;
    for (; k + U * STEP <= K; k += U * STEP) {
        gv_float4 x[U][C];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int c = 0; c < C; ++c) x[u][c] = __builtin_nontemporal_load(reinterpret_cast<const gv_float4*>(w[c] + k + u * STEP));
#pragma unroll
        for (int u0 = 0; u0 < U; u0 += UA) {
            gv_float4 y[UA][MB];
#pragma unroll
            for (int u = 0; u < UA; ++u)
#pragma unroll
                for (int m = 0; m < MB; ++m) y[u][m] = *reinterpret_cast<const gv_float4*>(a[m] + k + (u0 + u) * STEP);
#pragma unroll
            for (int u = 0; u < UA; ++u) add(x[u0 + u], y[u]);
        }
    }
    for (; k + lane * 4 < K; k += STEP) {
        gv_float4 x[C];
#pragma unroll
        for (int c = 0; c < C; ++c) x[c] = *reinterpret_cast<const gv_float4*>(w[c] + k);
        gv_float4 y[MB];
#pragma unroll
        for (int m = 0; m < MB; ++m) y[m] = *reinterpret_cast<const gv_float4*>(a[m] + k);
        add(x, y);
    }
#pragma unroll
    for (int c = 0; c < C; ++c) {
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            float v = ka_wave_sum(acc[c][m]);
            if (lane == 0 && m < M && n0 + c < N) {
                v += bias ? bias[n0 + c] : 0.f;
                if (act) v = ka_activate(act, v);
                const size_t o = (size_t)m * ldo + n0 + c;
                out[o] = accumulate ? out[o] + v : v;
            }
        }
    }
}

template <int MB, int C>
static void launch_gemv_form(const float* A, long lda, const float* W, long ldw, const float* bias, float* out, long ldo, int M, int N, int K,
                             int act, int accumulate, hipStream_t stream) {
    hipLaunchKernelGGL((gemv_f32_kernel<MB, C>), dim3(ka_cdiv(N, C * GV_WAVES)), dim3(GV_WAVES * KA_WAVE), 0, stream, A, lda, W, ldw, bias, out,
                       ldo, M, N, K, act, accumulate);
}

// Columns a wave: more of them ask the cache for fewer activations, fewer of them leave more waves to wait for memory. Two are
// best over most of the range; one where there are less than 16 waves a CU and at most four rows (2,048 columns of 8,192 at three
// rows: 19.6 us, 22.5 with two, 22.8 with four), four from five rows and 32 waves a CU on (51,200 x 2,048 at sixteen rows:
// 210, 228 with two, 306 with one).
template <int MB>
static void launch_gemv(const float* A, long lda, const float* W, long ldw, const float* bias, float* out, long ldo, int M, int N, int K, int act,
                        int accumulate, hipStream_t stream) {
    const int cus = ka_compute_units();
    if (MB <= 4 && N < 16 * cus) launch_gemv_form<MB, 1>(A, lda, W, ldw, bias, out, ldo, M, N, K, act, accumulate, stream);
    else if (MB >= 6 && N >= 32 * cus) launch_gemv_form<MB, 4>(A, lda, W, ldw, bias, out, ldo, M, N, K, act, accumulate, stream);
    else launch_gemv_form<MB, 2>(A, lda, W, ldw, bias, out, ldo, M, N, K, act, accumulate, stream);
}

template <typename TA, typename TW, typename TOut>
static void launch(const void* A, long lda, const void* W, long ldw, const float* bias, void* out,
                   long ldo, int M, int N, int K, int act, int accumulate, hipStream_t stream) {
    dim3 grid(ka_cdiv(N, GT), ka_cdiv(M, GT)), block(256);
    hipLaunchKernelGGL((gemm_generic_kernel<TA, TW, TOut>), grid, block, 0, stream, (const TA*)A, lda,
                       (const TW*)W, ldw, bias, (TOut*)out, ldo, M, N, K, act, accumulate);
}

// A: [M, K] rows lda apart; W: [N, K] rows ldw apart; bias: fp32 [N] or null;
// out: [M, N] rows ldo apart. act: 0 none, 1 GELU-tanh. accumulate: out += result
// (only into fp32 out).
KA_API int ka_linear_generic(const void* A, int a_dtype, long lda, const void* W, int w_dtype,
                             long ldw, const float* bias, void* out, int out_dtype, long ldo,
                             int M, int N, int K, int act, int accumulate, hipStream_t stream) {
    KA_CHECK(M >= 0 && N > 0 && K > 0, "ka_linear_generic: bad sizes M=%d N=%d K=%d", M, N, K);
    KA_CHECK(ka_act_known(act), "ka_linear_generic: unknown activation %d", act);
    KA_CHECK(lda >= K && ldw >= K && ldo >= ka_act_outputs(act, N), "ka_linear_generic: strides too small");
    KA_CHECK(!ka_act_gated(act) || (N % 2 == 0 && !accumulate), "ka_linear_generic: a gated linear needs an even N and no accumulation");
    KA_CHECK(!(accumulate && out_dtype != KA_F32), "ka_linear_generic: accumulate needs an fp32 output");
    KA_CHECK(ka_cdiv(M, GT) <= 65535, "ka_linear_generic: M=%d too large for one launch", M);
    if (M == 0) return 0;
    int key = a_dtype * 4 + w_dtype * 2 + out_dtype;
    const bool vectors = key == 0 && K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && (uintptr_t)A % 16 == 0 &&
                         (uintptr_t)W % 16 == 0;
    // (a gated linear at any number of rows, since the weight-streaming kernel has no pairs: its sums then never depend on the rows
    // beside a row. 1 to 16 rows of 2,048 inputs, 16,384 outputs: 199 to 212 us by vector tiles, 28 here; 1,408: 180 to 188 and 16.5)
    if (vectors && (M > GV_ROWS || ka_act_gated(act)) && K % F32_STEP == 0) {
        return launch_f32_best((const float*)A, lda, (const float*)W, ldw, bias, (float*)out, ldo, M, N, K, act, accumulate, stream);
    }
    if (vectors && M > GV_ROWS && ka_cdiv(M, 64) <= 65535) {
        if ((long)ka_cdiv(N, GF) * ka_cdiv(M, GF) >= 512)
            hipLaunchKernelGGL(gemm_f32_kernel<8>, dim3(ka_cdiv(N, GF), ka_cdiv(M, GF)), dim3(256), 0, stream, (const float*)A, lda,
                               (const float*)W, ldw, bias, (float*)out, ldo, M, N, K, act, accumulate);
        else
            hipLaunchKernelGGL(gemm_f32_kernel<4>, dim3(ka_cdiv(N, GF), ka_cdiv(M, 64)), dim3(256), 0, stream, (const float*)A, lda,
                               (const float*)W, ldw, bias, (float*)out, ldo, M, N, K, act, accumulate);
        KA_LAUNCH_CHECK();
        return 0;
    }
    if (vectors && M <= GV_ROWS && !ka_act_gated(act)) {      // (a wave per column there: the pair of a gate would meet nowhere)
#define KA_GEMV(MB) launch_gemv<MB>((const float*)A, lda, (const float*)W, ldw, bias, (float*)out, ldo, M, N, K, act, accumulate, stream)
        if (M <= 1) KA_GEMV(1);
        else if (M <= 2) KA_GEMV(2);
        else if (M <= 3) KA_GEMV(3);
        else if (M <= 4) KA_GEMV(4);
        else if (M <= 6) KA_GEMV(6);
        else if (M <= 8) KA_GEMV(8);
        else KA_GEMV(16);
#undef KA_GEMV
        KA_LAUNCH_CHECK();
        return 0;
    }
#define KA_CASE(k, TA, TW, TO) \
    case k: launch<TA, TW, TO>(A, lda, W, ldw, bias, out, ldo, M, N, K, act, accumulate, stream); break;
    switch (key) {
        KA_CASE(0, float, float, float)
        KA_CASE(1, float, float, bf16_t)
        KA_CASE(2, float, bf16_t, float)
        KA_CASE(3, float, bf16_t, bf16_t)
        KA_CASE(4, bf16_t, float, float)
        KA_CASE(5, bf16_t, float, bf16_t)
        KA_CASE(6, bf16_t, bf16_t, float)
        KA_CASE(7, bf16_t, bf16_t, bf16_t)
        default: KA_CHECK(false, "ka_linear_generic: unsupported dtypes a=%d w=%d out=%d", a_dtype, w_dtype, out_dtype);
    }
#undef KA_CASE
    KA_LAUNCH_CHECK();
    return 0;
}
