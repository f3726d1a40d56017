// Generic linear layer: out = act(A W^T + bias) or out += A W^T + bias.
//
// Four kernels, each with an order of a sum that K alone fixes:
//  * any M, N, K, any mix of fp32 and bf16 operands: plain FMA in fp32 with an LDS-tiled 64x64x16 block, k = 0..K-1 in that
//    order; the fallback of the bf16 path;
// and, of aligned fp32 operands, the true 32-bit path,
//  * up to 16 rows of a linear without a gate: a stream of weights (gemv_f32_kernel);
//  * else K in steps of 32: the matrix pipes, in 32 bits, or the activations as three of bf16 where weights are bf16 numbers (gemm_f32_tiles_kernel);
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

// Many rows in fp32 where K is a multiple of 32, on the matrix pipes: products of 32 bits (v_mfma_f32_32x32x2_f32), and for weights that are bf16 numbers, as checkpoints hold
// them, products of the activations' three bf16 parts (v_mfma_f32_32x32x16_bf16, sixteen times the rate). A number of 32 bits is the sum of three bf16 numbers to its last bit:
// 24 bits of mantissa, eight in each; what rounding to the nearest leaves is representable, so both subtractions are exact. Then w x = w x1 + w x2 + w x3, each exact in the
// pipe: nothing is left out, and the sums are fp32 either way.
//
// Which of the two a sum takes is decided per weight row, row of A and part of K, by those rows alone, so that every tile gives the same bits:
//  * A weight whose lower half is not zero has no single bf16 part. Where every row of the tile shows one among its first sixteen numbers (weights of 32 bits do),
//    nothing but products of 32 bits is run.
//  * A number of A below 2^-109 may have bits below bf16's smallest: what is left for the third part then has a lower half.
//  * Infinities, NaN and what lies beyond bf16's largest leave a sum that is not finite.
// Where a tile meets one of these, the wave that does multiplies its part once more in 32 bits, and the sums that need it take that result (us, inputs x outputs here and below, 282 rows, usual numbers, a
// NaN in every row, numbers of 1e-36, and one weight row in 50 of 32 bits: 2,048 x 6,144 64, 108, 133 and 121; 8,192 x 2,048 87, 169, 203 and 160).
//
// Operands go straight from memory into swizzled LDS as in ka_dma_tiles.h, whole lines of 32 numbers, and are split by the wave that multiplies them, between the products of
// the half step before, which the compiler does only where each half is a region of its own with an end that names the parts. Tiles of 32 x 32 alone, two workgroups a
// CU: waves with 64 x 64 split half as often, but are one a SIMD, and the vector unit, which fetches their sums from the matrix pipe's registers, is what multiplies 32-bit
// numbers (us, tiles of 32 and of 64, bf16 weights and those of 32 bits: 282 rows of 2,048 x 6,144 61 and 55, 80 and 94; 2,048 rows 347 and 307, 515 and 558; 2,048 rows of
// 8,192 x 2,048 422 and 306, 644 and 661; 2,560 x 7,680, 64 rows 31 and 51, 33 and 61).
//
// The order of a sum is fixed by K alone. K is cut into F32_PARTS parts, each summed by a wave of its own (so no wave waits for another before the end); the parts' sums meet in LDS
// and are added in their order.
//  * Products of 32 bits: every sixteen k are summed from zero (of every eight in the order 0 4 1 5 2 6 3 7: a lane holds four neighbours), these sums added in order. The short
//    chains take the error of a sum from that of a chain of K / 4 terms to that of one of K / 64 (of every 32 from zero: 6 % faster, an error up to 9 % larger).
//  * Three parts: w x1 of 128 of K from zero, these sums in order; w x2 and w x3, whose roundings weigh 2^-8, in an accumulator beside them.
//
// Measured, us; all products in 32 bits by tiles of 32 x 32 to 64 x 128 -> here with weights of 32 bits and with bf16 numbers: 2,048 x 6,144, 17 rows 19.3 -> 17.6, 15.4; 64
// rows 27.1 -> 28.0, 23.3; 282 rows 81.8 -> 80.3, 59.1; 2,048 rows 445 -> 521, 329. 8,192 x 2,048: 51.1 -> 46.7, 34.8; 51.7 -> 47.8, 38.5; 130 -> 128, 84.8; 614 -> 659, 425. Over 14
// shapes (1,024 to 10,240 outputs, K of 1,024 to 10,240): 17 to 32 rows 0.96 and 0.85 of the time, 48 to 64 0.98 and 0.85, 80 to 160 0.98 and 0.80, 282 1.01 and 0.74, 512 1.05 and 0.77,
// 2,048 1.12 and 0.77. Error against 64 bits of sums of 2,048 1.35e-7, with bf16 weights 8.7e-8; of 8,192 2.2e-7 and 1.1e-7.
constexpr int F32_PARTS = 4;
constexpr int F32_STEP = 32;
constexpr int F32_TILE = 32;
constexpr int F32_BLOCK = 4;       // steps whose main products are summed from zero

typedef __attribute__((ext_vector_type(2))) float gs_float2;
typedef __attribute__((ext_vector_type(2))) __bf16 gs_bf16x2;

// part[0] + part[1] + part[2] is the eight numbers of lo and hi to the last bit, or the lower half of what is returned is not zero: what is left for the third part is a bf16
// number exactly where its lower half is zero.
__device__ __forceinline__ unsigned gs_split(const floatx4& lo, const floatx4& hi, bf16x8 (&part)[3]) {
    uint4 out[3];
    unsigned left = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float a = i < 2 ? lo[2 * i] : hi[2 * i - 4], b = i < 2 ? lo[2 * i + 1] : hi[2 * i - 3];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            const unsigned pair = __builtin_bit_cast(unsigned, __builtin_convertvector(gs_float2{a, b}, gs_bf16x2));
            (i == 0 ? out[p].x : i == 1 ? out[p].y : i == 2 ? out[p].z : out[p].w) = pair;
            if (p == 2) {
                left |= __float_as_uint(a) | __float_as_uint(b);
                break;
            }
            a -= __uint_as_float(pair << 16);
            b -= __uint_as_float(pair & 0xffff0000u);
        }
    }
#pragma unroll
    for (int p = 0; p < 3; ++p) part[p] = __builtin_bit_cast(bf16x8, out[p]);
    return left;
}

// NS: steps in LDS
template <int NS>
__global__ void __launch_bounds__(KA_WAVE * F32_PARTS, 2)
gemm_f32_tiles_kernel(const float* __restrict__ A, long lda, const float* __restrict__ W, long ldw, const float* __restrict__ bias,
                      float* __restrict__ out, long ldo, int M, int N, int K, int act, int accumulate, int tiles_n, int tiles_m) {
    constexpr int ROW = F32_STEP * 4, CPR = ROW / 16, RPL = KA_WAVE / CPR, STAGE = 2 * F32_TILE * ROW;      // a step: the rows of W, then of A
    constexpr int LOADS = F32_TILE / RPL, LPW = 2 * LOADS;
    extern __shared__ __attribute__((aligned(16))) unsigned char gf_lds[];
    const int total = tiles_n * tiles_m, per_xcd = (total + 7) / 8;
    const int logical = blockIdx.x % 8 * per_xcd + blockIdx.x / 8;
    if (logical >= total || (int)blockIdx.x / 8 >= per_xcd) return;
    // Up to ten tiles of A's rows at a time, through all of W: what an XCD's 64 workgroups read at once is nearly a square (2,048 rows of 2,048 x 6,144, bf16 weights, 433 -> 329 us).
    const int groups = (tiles_m + 9) / 10, height = (tiles_m + groups - 1) / groups, group = logical / (height * tiles_n);
    const int here = min(height, tiles_m - group * height), within = logical - group * height * tiles_n;
    const int n0 = within / here * F32_TILE, m0 = (group * height + within % here) * F32_TILE;
    const int part = __builtin_amdgcn_readfirstlane(threadIdx.x / KA_WAVE), lane = threadIdx.x % KA_WAVE;
    const int li = lane % 32, lg = lane / 32;
    const int part_steps = ((K + F32_PARTS - 1) / F32_PARTS + F32_STEP - 1) / F32_STEP, k_steps = K / F32_STEP;
    const int first = part * part_steps, steps = max(0, min(part_steps, k_steps - first));
    const float* wsrc[LOADS];
    const float* xsrc[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {                                          // (four numbers a piece; rows past the end: the last one again, not stored)
        const int r = kd_load_row<CPR>(i, lane), c = kd_load_channel<CPR>(r, lane) / 2 + first * F32_STEP;
        wsrc[i] = W + (size_t)min(n0 + r, N - 1) * ldw + c;
        xsrc[i] = A + (size_t)min(m0 + r, M - 1) * lda + c;
    }
    unsigned char* mine = gf_lds + part * NS * STAGE;
    auto fetch = [&](int step) {
        unsigned char* base = mine + step % NS * STAGE;
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            __builtin_amdgcn_global_load_lds((const GD_GLOBAL void*)(wsrc[i] + step * F32_STEP), (GD_LDS void*)(base + i * RPL * ROW), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            __builtin_amdgcn_global_load_lds((const GD_GLOBAL void*)(xsrc[i] + step * F32_STEP), (GD_LDS void*)(base + (LOADS + i) * RPL * ROW), 16, 0, 0);
    };
    // the first stages, and the first step's loads landed
    auto begin = [&] {
#pragma unroll
        for (int st = 0; st < NS; ++st)
            if (st < steps) fetch(st);
        gd_wait_younger<LPW, NS - 1>(min(NS, steps) - 1);
    };
    const int swz = kd_swizzle<CPR>(li);
    // four numbers of half a step of this lane's row of W (0) or of A (1); h = 0, 1: the eight of its products
    auto four = [&](int step, int half, int operand, int h) {
        return *reinterpret_cast<const floatx4*>(mine + step % NS * STAGE + (operand * F32_TILE + li) * ROW + ((half * 4 + h * 2 + lg) ^ swz) * 16);
    };
    const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    floatx16 acc = zero;
    unsigned odd[2] = {0, 0};        // this lane's row of W, of A: the lower half is not zero where it has a number that the parts do not say
    unsigned rows[2] = {0, 0};       // the same, a bit a row
    auto gather = [&] {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const unsigned long long hit = __builtin_amdgcn_ballot_w64((odd[i] & 0xffff) != 0);
            rows[i] = (unsigned)hit | (unsigned)(hit >> 32);
        }
    };
    bool again = false;              // products of 32 bits
    if (steps > 0) {
        begin();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint4 w = __builtin_bit_cast(uint4, four(0, 0, 0, h));
            odd[0] |= w.x | w.y | w.z | w.w;
        }
        gather();
        again = rows[0] == 0xffffffffu;
    }
    if (steps > 0 && !again) {
        floatx16 few = zero, low = zero;
        bf16x8 w[2], x[2][3];
        // The operands of half a step from LDS (its loads have landed; a wave reads what it asked for itself: no barrier). counts: the half step is one of the part's.
        auto operands = [&](auto half_c, int step, unsigned counts) __attribute__((always_inline)) {
            constexpr int half = decltype(half_c)::value;
            const floatx4 w_lo = four(step, half, 0, 0), w_hi = four(step, half, 0, 1), x_lo = four(step, half, 1, 0), x_hi = four(step, half, 1, 1);
            const uint4 lo = __builtin_bit_cast(uint4, w_lo), hi = __builtin_bit_cast(uint4, w_hi);
            uint4 upper;
            upper.x = __builtin_amdgcn_perm(lo.y, lo.x, 0x07060302);
            upper.y = __builtin_amdgcn_perm(lo.w, lo.z, 0x07060302);
            upper.z = __builtin_amdgcn_perm(hi.y, hi.x, 0x07060302);
            upper.w = __builtin_amdgcn_perm(hi.w, hi.z, 0x07060302);
            w[half] = __builtin_bit_cast(bf16x8, upper);
            odd[0] |= (lo.x | lo.y | lo.z | lo.w | hi.x | hi.y | hi.z | hi.w) & counts;
            odd[1] |= gs_split(x_lo, x_hi, x[half]) & counts;
        };
        // Half a step: its products, and between them the split of the next one's operands, which the matrix pipe does not need. STEADY: a step that has NS behind it.
        auto half_step = [&](auto half_c, auto steady_c, int s) __attribute__((always_inline)) {
            constexpr int half = decltype(half_c)::value;
            constexpr bool STEADY = decltype(steady_c)::value;
            if constexpr (half == 1) {
                if constexpr (STEADY) gd_wait_loads<LPW * (NS - 2)>();
                else if (s + 1 < steps) gd_wait_younger<LPW, NS - 2>(min(NS - 2, steps - 2 - s));
                gd_wait_lds();                                                 // own reads of the step are in registers: its stage may be written
                if (STEADY || s + NS < steps) fetch(s + NS);
                operands(std::integral_constant<int, 0>{}, s + 1, STEADY || s + 1 < steps ? ~0u : 0u);      // (behind the last step: memory that nobody uses)
            } else {
                operands(std::integral_constant<int, 1>{}, s, ~0u);
            }
            low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[half], x[half][2], low, 0, 0, 0);
            few = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[half], x[half][0], few, 0, 0, 0);
            low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[half], x[half][1], low, 0, 0, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
            gd_static_for<0, 3>([&](auto) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 20, 0);
            });
            // (the split belongs here: the compiler would put it off to the half step that uses it, in front of that one's products)
            asm volatile("" : "+v"(w[half ^ 1]), "+v"(x[half ^ 1][0]), "+v"(x[half ^ 1][1]), "+v"(x[half ^ 1][2]));
            __builtin_amdgcn_sched_barrier(0);
        };
        auto settle = [&] {
            acc += few;
            few = zero;
        };
        operands(std::integral_constant<int, 0>{}, 0, ~0u);
        int s = 0;
        auto two_steps = [&](auto steady_c) __attribute__((always_inline)) {
            half_step(std::integral_constant<int, 0>{}, steady_c, s);
            half_step(std::integral_constant<int, 1>{}, steady_c, s);
            half_step(std::integral_constant<int, 0>{}, steady_c, s + 1);
            half_step(std::integral_constant<int, 1>{}, steady_c, s + 1);
            s += 2;
            if (s % F32_BLOCK == 0) settle();
        };
        while (s + 1 + NS < steps) two_steps(std::true_type{});
        while (s + 1 < steps) two_steps(std::false_type{});
        if (s < steps) {
            half_step(std::integral_constant<int, 0>{}, std::false_type{}, s);
            half_step(std::integral_constant<int, 1>{}, std::false_type{}, s);
        }
        settle();
        acc += low;
        gather();
        bool beyond = false;
#pragma unroll
        for (int v = 0; v < 16; ++v) beyond |= !(fabsf(acc[v]) < INFINITY);
        again = rows[0] != 0 || rows[1] != 0 || __builtin_amdgcn_ballot_w64(beyond) != 0;
        if (again) {
            gd_wait_lds();
            begin();
        }
    }
    if (again) {
        floatx16 sum = zero;
        for (int s = 0; s < steps; ++s) {
            if (s > 0) gd_wait_younger<LPW, NS - 1>(min(NS, steps - s) - 1);
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const floatx4 w[2] = {four(s, half, 0, 0), four(s, half, 0, 1)}, x[2] = {four(s, half, 1, 0), four(s, half, 1, 1)};
                floatx16 y = zero;
#pragma unroll
                for (int j = 0; j < 8; ++j) y = __builtin_amdgcn_mfma_f32_32x32x2f32(w[j / 4][j % 4], x[j / 4][j % 4], y, 0, 0, 0);
                sum += y;
            }
            gd_wait_lds();                                                     // own reads of the step are in registers: its stage may be written
            if (s + NS < steps) fetch(s + NS);
        }
#pragma unroll
        for (int v = 0; v < 16; ++v)
            if ((rows[0] >> (v / 4 * 8 + lg * 4 + v % 4) | rows[1] >> li) & 1 || !(fabsf(acc[v]) < INFINITY)) acc[v] = sum[v];
    }
    // acc[v] is out[m][n] with n = n0 + (v / 4) 8 + lg 4 + v % 4 and m = m0 + li. The parts' sums through LDS; every wave finishes a quarter of the tile's numbers.
    gd_wait_lds();
    gd_barrier();
    floatx4* sums = reinterpret_cast<floatx4*>(gf_lds);
#pragma unroll
    for (int q = 0; q < 4; ++q) sums[(part * 4 + q) * KA_WAVE + lane] = floatx4{acc[q * 4], acc[q * 4 + 1], acc[q * 4 + 2], acc[q * 4 + 3]};
    gd_wait_lds();
    gd_barrier();
    const int parts = (k_steps + part_steps - 1) / part_steps;                 // (those that hold anything)
    floatx4 y = sums[part * KA_WAVE + lane];
    for (int p = 1; p < parts; ++p) y += sums[(p * 4 + part) * KA_WAVE + lane];
    const int m = m0 + li, n = n0 + part * 8 + lg * 4;
    if (m >= M || n >= N) return;
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = y[j] + (bias && n + j < N ? bias[n + j] : 0.f);
    if (ka_act_gated(act)) {
        ka_gated_store<false, 4>(out, KA_F32, ldo, m, n, N, v, act);
        return;
    }
    if (act)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = ka_activate(act, v[j]);
    float* op = out + (size_t)m * ldo + n;
    if (N % 4 == 0 && ldo % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0) {
        floatx4 r = {v[0], v[1], v[2], v[3]};
        if (accumulate) r = *reinterpret_cast<const floatx4*>(op) + r;
        *reinterpret_cast<floatx4*>(op) = r;
    } else {
        for (int j = 0; j < 4 && n + j < N; ++j) op[j] = accumulate ? op[j] + v[j] : v[j];
    }
}

template <int NS>
static int launch_f32_tiles(const float* A, long lda, const float* W, long ldw, const float* bias, float* out, long ldo, int M, int N, int K,
                            int act, int accumulate, hipStream_t stream) {
    constexpr int smem = F32_PARTS * NS * 2 * F32_TILE * F32_STEP * 4;
    static_assert(smem >= F32_PARTS * 4 * KA_WAVE * 16, "the parts' sums fit");
    static bool configured = false;
    auto kernel = gemm_f32_tiles_kernel<NS>;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        KA_CHECK(e == hipSuccess, "ka_linear_generic: cannot reserve %d bytes of LDS: %s", smem, hipGetErrorString(e));
        configured = true;
    }
    const int tiles_n = ka_cdiv(N, F32_TILE), tiles_m = ka_cdiv(M, F32_TILE);
    const long blocks = ((long)tiles_n * tiles_m + 7) / 8 * 8;
    KA_CHECK(blocks < (1L << 31), "ka_linear_generic: too many tiles");
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(KA_WAVE * F32_PARTS), smem, stream, A, lda, W, ldw, bias, out, ldo, M, N, K, act,
                       accumulate, tiles_n, tiles_m);
    KA_LAUNCH_CHECK();
    return 0;
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
        // (a third step in LDS where no CU has two workgroups, which have room for two each: 17 rows of 2,048 x 6,144, bf16 weights, 17.3 and 13.9 us; 2,560 x 10,240 of 32 bits, 320 workgroups, 33.6 and 36.0)
        const bool alone = (long)ka_cdiv(M, F32_TILE) * ka_cdiv(N, F32_TILE) <= ka_compute_units();
        return (alone ? launch_f32_tiles<3> : launch_f32_tiles<2>)((const float*)A, lda, (const float*)W, ldw, bias, (float*)out, ldo, M, N, K, act, accumulate, stream);
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
