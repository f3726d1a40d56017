// The linears of a block of two branches for few rows in 32 bits: the two that read the normalised rows in one launch, the norm in its prologue, and the two
// whose results go into the rows in another. Every sum has the order that gemv_f32_kernel and the norm's own launch (gemm_generic.hip, elementwise.hip) give it, to the
// bit: a lane adds up its own k of every 256, ascending, and the lanes' sums meet in a tree.
//
// Both are bound by the stream of weights, 117 and 84 MB a block of 2,048 with 8,192 between the feed-forward's linears. What they save over a launch each is a start and an
// end of some 3 us, and the trips of the activations through the CUs' caches: those lie in LDS here, in the first launch for as long as a workgroup lives, in the
// second a chunk at a time.
// Us, weights from HBM, the launches in turn (norm, linear, linear; linear, linear) and these; width 2,048: one row 23.8 and 20.3, 16.9 and 16.3; three 30.7 and 21.1 (5.6 TB/s),
// 22.2 and 17.4; six 41.7 and 25.6, 34.3 and 20.6; eight 47.4 and 30.1, 38.1 and 22.8; 2,560 wide, three rows 42.4 and 32.2, 40.2 and 29.6; 1,024 wide, three rows 14.0 and 9.5, 12.1
// and 8.2.
#include "ka_common.h"
#include "ka_dma_tiles.h"

typedef __attribute__((ext_vector_type(4))) float gp_float4;

constexpr int GP_WAVES = 4, GP_THREADS = GP_WAVES * KA_WAVE, GP_STEP = KA_WAVE * 4;
constexpr int GP_ROWS = 8;           // most rows

__device__ __forceinline__ void gp_add(float& acc, const gp_float4& y, const gp_float4& x) {
    acc = fmaf(y[3], x[3], fmaf(y[2], x[2], fmaf(y[1], x[1], fmaf(y[0], x[0], acc))));
}

struct GpFirst {
    const float* x;             // [M, K]
    long ldx;
    const float *gamma, *beta;  // null gamma: the rows as they are; beta may be null
    float eps;
    const float* W[2];          // [N[s], K]
    const float* bias[2];       // may be null
    float* out[2];
    long ldw[2], ldo[2];
    int N[2], act[2], M, K;
};

// out[s] = act[s](norm(x) W[s]^T + bias[s]). ITEMS: fours of a row that a thread holds while it is normalised. A wave takes C neighbouring outputs, then those as many further
// on as there are waves, and asks for a unit of U steps of their weights while it multiplies the one before. (One output a wave and eight steps, twice the reads of LDS: three
// rows of 2,048 22.6 us instead of 21.1, six 35.0 instead of 25.6.)
template <int MB, int ITEMS>
__global__ void __launch_bounds__(GP_THREADS)
gp_first_kernel(GpFirst p) {
    constexpr int C = 2, U = 4;
    extern __shared__ __attribute__((aligned(16))) float gp_rows[];
    __shared__ float part[2][MB][GP_WAVES];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KA_WAVE), lane = threadIdx.x % KA_WAVE, K = p.K;
    const int groups0 = (p.N[0] + C - 1) / C, groups = groups0 + (p.N[1] + C - 1) / C, waves = gridDim.x * GP_WAVES;
    const int units = (K + U * GP_STEP - 1) / (U * GP_STEP);
    gp_float4 w[2][U][C];
    auto fetch = [&](gp_float4 (&to)[U][C], int group, int unit) {
        const int s = group >= groups0, n0 = (group - (s ? groups0 : 0)) * C;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int c = 0; c < C; ++c)          // (outputs and steps past the end: the last again, not used)
                to[u][c] = __builtin_nontemporal_load(reinterpret_cast<const gp_float4*>(p.W[s] + (size_t)min(n0 + c, p.N[s] - 1) * p.ldw[s] +
                                                                                         min((unit * U + u) * GP_STEP, K - GP_STEP) + lane * 4));
    };
    int group = __builtin_amdgcn_readfirstlane(blockIdx.x * GP_WAVES + wave), unit = 0;
    if (group < groups) fetch(w[0], group, 0);
    {
        gp_float4 v[MB][ITEMS], g[ITEMS], b[ITEMS];
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            const int d = min((j * GP_THREADS + (int)threadIdx.x) * 4, K - 4);
#pragma unroll
            for (int m = 0; m < MB; ++m) v[m][j] = *reinterpret_cast<const gp_float4*>(p.x + (size_t)min(m, p.M - 1) * p.ldx + d);
            if (p.gamma) {
                g[j] = *reinterpret_cast<const gp_float4*>(p.gamma + d);
                b[j] = p.beta ? *reinterpret_cast<const gp_float4*>(p.beta + d) : gp_float4{0.f, 0.f, 0.f, 0.f};
            }
        }
        if (p.gamma) {
            float mean[MB], rstd[MB];
            auto total = [&](int which, int m) {
                float t = 0.f;
#pragma unroll
                for (int i = 0; i < GP_WAVES; ++i) t += part[which][m][i];
                return t;
            };
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                float s = 0.f;
#pragma unroll
                for (int j = 0; j < ITEMS; ++j) {
                    if ((j * GP_THREADS + (int)threadIdx.x) * 4 >= K) v[m][j] = gp_float4{0.f, 0.f, 0.f, 0.f};
                    s += (v[m][j][0] + v[m][j][1]) + (v[m][j][2] + v[m][j][3]);
                }
                s = ka_wave_sum(s);
                if (lane == 0) part[0][m][wave] = s;
            }
            gd_wait_lds();
            gd_barrier();
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                mean[m] = total(0, m) / (float)K;
                float q = 0.f;
#pragma unroll
                for (int j = 0; j < ITEMS; ++j)
                    if ((j * GP_THREADS + (int)threadIdx.x) * 4 < K) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) q += (v[m][j][e] - mean[m]) * (v[m][j][e] - mean[m]);
                    }
                q = ka_wave_sum(q);
                if (lane == 0) part[1][m][wave] = q;
            }
            gd_wait_lds();
            gd_barrier();
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                rstd[m] = 1.0f / sqrtf(total(1, m) / (float)K + p.eps);
#pragma unroll
                for (int j = 0; j < ITEMS; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[m][j][e] = (v[m][j][e] - mean[m]) * rstd[m] * g[j][e] + b[j][e];
            }
        }
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            const int d = (j * GP_THREADS + (int)threadIdx.x) * 4;
            if (d < K)
#pragma unroll
                for (int m = 0; m < MB; ++m) *reinterpret_cast<gp_float4*>(gp_rows + m * K + d) = v[m][j];
        }
        gd_wait_lds();
        gd_barrier();
    }
    float acc[C][MB];
    auto clear = [&] {
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int m = 0; m < MB; ++m) acc[c][m] = 0.f;
    };
    clear();
    auto turn = [&](gp_float4 (&now)[U][C], gp_float4 (&next)[U][C]) {
        const bool last = unit + 1 == units;
        const int then = last ? group + waves : group;
        if (then < groups) fetch(next, then, last ? 0 : unit + 1);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = (unit * U + u) * GP_STEP;
            if (k < K) {
                gp_float4 y[MB];
#pragma unroll
                for (int m = 0; m < MB; ++m) y[m] = *reinterpret_cast<const gp_float4*>(gp_rows + m * K + k + lane * 4);
#pragma unroll
                for (int m = 0; m < MB; ++m)
#pragma unroll
                    for (int c = 0; c < C; ++c) gp_add(acc[c][m], y[m], now[u][c]);
            }
        }
        if (last) {
            // lane c MB + m finishes output n0 + c of row m
            const int s = group >= groups0, n0 = (group - (s ? groups0 : 0)) * C, n = n0 + lane / MB, m = lane % MB;
            float mine = 0.f;
#pragma unroll
            for (int i = 0; i < C * MB; ++i) {
                const float t = ka_wave_sum(acc[i / MB][i % MB]);
                mine = lane == i ? t : mine;
            }
            if (lane < C * MB && m < p.M && n < p.N[s]) {
                mine += p.bias[s] ? p.bias[s][n] : 0.f;
                if (p.act[s]) mine = ka_activate(p.act[s], mine);
                p.out[s][(size_t)m * p.ldo[s] + n] = mine;
            }
            clear();
        }
        unit = last ? 0 : unit + 1;
        group = then;
    };
    while (group < groups) {
        turn(w[0], w[1]);
        if (group >= groups) break;
        turn(w[1], w[0]);
    }
}

struct GpLast {
    const float* A[2];          // [M, K[s]]
    const float* W[2];          // [N, K[s]]
    const float* bias[2];       // may be null
    long lda[2], ldw[2];
    int K[2], M, N;
    float* out;                 // [M, N]
    long ldo;
};

// out += A[0] W[0]^T + bias[0], then += A[1] W[1]^T + bias[1]. A wave has one output; chunks of four steps, of the first linear and then of the second. The weights are asked for
// two chunks ahead into registers, the activations one chunk ahead, by all of the workgroup into LDS.
template <int MB>
__global__ void __launch_bounds__(GP_THREADS)
gp_last_kernel(GpLast p) {
    constexpr int U = 4, CHUNK = U * GP_STEP;
    static_assert(CHUNK == GP_THREADS * 4, "a thread brings one four of a row");
    __shared__ __attribute__((aligned(16))) float rows[2][MB][CHUNK];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KA_WAVE), lane = threadIdx.x % KA_WAVE;
    const int n = blockIdx.x * GP_WAVES + wave, border = (p.K[0] + CHUNK - 1) / CHUNK, chunks = border + (p.K[1] + CHUNK - 1) / CHUNK;
    const size_t row = (size_t)min(n, p.N - 1);
    gp_float4 w[3][U], a[MB];
    // (a chunk past the last: the last again; places past a linear's K: its last ones again, not used)
    auto weights = [&](gp_float4 (&to)[U], int c) {
        c = min(c, chunks - 1);
        const int s = c >= border, k = (c - (s ? border : 0)) * CHUNK;
        const float* from = p.W[s] + row * p.ldw[s] + lane * 4;
#pragma unroll
        for (int u = 0; u < U; ++u) to[u] = __builtin_nontemporal_load(reinterpret_cast<const gp_float4*>(from + min(k + u * GP_STEP, p.K[s] - GP_STEP)));
    };
    auto activations = [&](int c) {
        c = min(c, chunks - 1);
        const int s = c >= border, k = min((c - (s ? border : 0)) * CHUNK + (int)threadIdx.x * 4, p.K[s] - 4);
#pragma unroll
        for (int m = 0; m < MB; ++m) a[m] = *reinterpret_cast<const gp_float4*>(p.A[s] + (size_t)min(m, p.M - 1) * p.lda[s] + k);
    };
    auto stage = [&](int c) {
#pragma unroll
        for (int m = 0; m < MB; ++m) *reinterpret_cast<gp_float4*>(&rows[c & 1][m][threadIdx.x * 4]) = a[m];
        gd_wait_lds();
        gd_barrier();
    };
    float acc[MB], first[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) acc[m] = 0.f;
    activations(0);
    weights(w[0], 0);
    weights(w[1], 1);
    stage(0);
    auto turn = [&](int c, gp_float4 (&now)[U], gp_float4 (&ahead)[U]) {
        if (c >= chunks) return;                 // (the same for the whole workgroup)
        activations(c + 1);
        weights(ahead, c + 2);
        if (c == border)
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                first[m] = acc[m];
                acc[m] = 0.f;
            }
        const int s = c >= border, k = (c - (s ? border : 0)) * CHUNK;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k + u * GP_STEP < p.K[s])
#pragma unroll
                for (int m = 0; m < MB; ++m) gp_add(acc[m], *reinterpret_cast<const gp_float4*>(&rows[c & 1][m][u * GP_STEP + lane * 4]), now[u]);
        }
        stage(c + 1);                            // (its half of LDS was last read for chunk c - 1, in front of a barrier)
    };
    for (int c = 0; c < chunks; c += 3) {
        turn(c, w[0], w[2]);
        turn(c + 1, w[1], w[0]);
        turn(c + 2, w[2], w[1]);
    }
    float mine = 0.f, more = 0.f;
#pragma unroll
    for (int m = 0; m < MB; ++m) {
        const float t = ka_wave_sum(first[m]), u = ka_wave_sum(acc[m]);
        mine = lane == m ? t : mine;
        more = lane == m ? u : more;
    }
    if (lane < p.M && lane < MB && n < p.N) {
        float* const at = p.out + (size_t)lane * p.ldo + n;
        const float y = *at + (mine + (p.bias[0] ? p.bias[0][n] : 0.f));
        *at = y + (more + (p.bias[1] ? p.bias[1][n] : 0.f));
    }
}

static bool gp_vectors(const void* p, long ld) { return (uintptr_t)p % 16 == 0 && ld % 4 == 0; }

// 1: done; 0: not covered, nothing was run; -1: an error.
KA_API int ka_linears_first_f32(const float* x, long ldx, const float* gamma, const float* beta, float eps, const float* W1, long ldw1, const float* bias1, float* out1, long ldo1,
                                int N1, int act1, const float* W2, long ldw2, const float* bias2, float* out2, long ldo2, int N2, int act2, int M, int K, hipStream_t stream) {
    const char* who = "ka_linears_first_f32";
    KA_CHECK(M > 0 && N1 > 0 && N2 > 0 && K > 0 && ldx >= K && ldw1 >= K && ldw2 >= K && ldo1 >= N1 && ldo2 >= N2, "%s: M=%d N=%d, %d K=%d", who, M, N1, N2, K);
    KA_CHECK(ka_act_known(act1) && ka_act_known(act2), "%s: unknown activation %d or %d", who, act1, act2);
    // (a workgroup normalises ITEMS fours a thread of a row, which has to be all of it: three up to six rows, two for seven and eight)
    if (M > GP_ROWS || K % GP_STEP || K > (M <= 6 ? 3072 : 2048) || M * K > 16384 || ka_act_gated(act1) || ka_act_gated(act2)) return 0;
    if (!gp_vectors(x, ldx) || !gp_vectors(W1, ldw1) || !gp_vectors(W2, ldw2) || !gp_vectors(gamma, 0) || !gp_vectors(beta, 0)) return 0;
    if ((long)N1 + N2 >= (1L << 30)) return 0;
    GpFirst p = {x, ldx, gamma, beta, eps, {W1, W2}, {bias1, bias2}, {out1, out2}, {ldw1, ldw2}, {ldo1, ldo2}, {N1, N2}, {act1, act2}, M, K};
    // Workgroups a CU: three where their rows leave room, which hides the norm of one behind the weights of the others (three rows of 2,048 21.1 us, with two 21.9, with four
    // 21.7; one row 20.3 each; six 25.6 and 26.1, eight 42.4 and 30.1, 1,024 wide 10.2 and 9.5).
    const int per_cu = M <= 3 && K > 1024 ? 3 : 2;
#define KA_FIRST(MB, ITEMS)                                                                                                                                                       \
    {                                                                                                                                                                             \
        KA_CHECK(M <= MB && K <= ITEMS * GP_THREADS * 4, "%s: %d rows of %d by a kernel of %d rows of %d", who, M, K, MB, ITEMS * GP_THREADS * 4);                                \
        static bool configured = false;                                                                                                                                           \
        if (!configured) {                                                                                                                                                        \
            hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gp_first_kernel<MB, ITEMS>), hipFuncAttributeMaxDynamicSharedMemorySize,              \
                                               MB * ITEMS * GP_THREADS * 16);      /* the form's longest rows: 73,728 bytes of six */                                        \
            KA_CHECK(e == hipSuccess, "%s: cannot reserve LDS: %s", who, hipGetErrorString(e));                                                                                    \
            configured = true;                                                                                                                                                    \
        }                                                                                                                                                                         \
        hipLaunchKernelGGL((gp_first_kernel<MB, ITEMS>), dim3(per_cu * ka_compute_units()), dim3(GP_THREADS), MB * K * 4, stream, p);                                               \
    }
#define KA_FIRST_ITEMS(MB)                                                                                                                                                        \
    if (K <= 2048) KA_FIRST(MB, 2) else KA_FIRST(MB, 3)
    if (M == 1) { KA_FIRST_ITEMS(1) }
    else if (M == 2) { KA_FIRST_ITEMS(2) }
    else if (M == 3) { KA_FIRST_ITEMS(3) }
    else if (M == 4) { KA_FIRST_ITEMS(4) }
    else if (M <= 6) { KA_FIRST_ITEMS(6) }
    else KA_FIRST(8, 2)
#undef KA_FIRST_ITEMS
#undef KA_FIRST
    KA_LAUNCH_CHECK();
    return 1;
}

// 1: done; 0: not covered, nothing was run; -1: an error.
KA_API int ka_linears_last_f32(const float* A1, long lda1, int K1, const float* W1, long ldw1, const float* bias1, const float* A2, long lda2, int K2, const float* W2, long ldw2,
                               const float* bias2, float* out, long ldo, int M, int N, hipStream_t stream) {
    const char* who = "ka_linears_last_f32";
    KA_CHECK(M > 0 && N > 0 && K1 > 0 && K2 > 0 && lda1 >= K1 && ldw1 >= K1 && lda2 >= K2 && ldw2 >= K2 && ldo >= N, "%s: M=%d N=%d K=%d, %d", who, M, N, K1, K2);
    if (M > GP_ROWS || K1 % GP_STEP || K2 % GP_STEP || !gp_vectors(A1, lda1) || !gp_vectors(W1, ldw1) || !gp_vectors(A2, lda2) || !gp_vectors(W2, ldw2)) return 0;
    GpLast p = {{A1, A2}, {W1, W2}, {bias1, bias2}, {lda1, lda2}, {ldw1, ldw2}, {K1, K2}, M, N, out, ldo};
#define KA_LAST(MB) hipLaunchKernelGGL(gp_last_kernel<MB>, dim3(ka_cdiv(N, GP_WAVES)), dim3(GP_THREADS), 0, stream, p)
    if (M == 1) KA_LAST(1);
    else if (M == 2) KA_LAST(2);
    else if (M == 3) KA_LAST(3);
    else if (M == 4) KA_LAST(4);
    else if (M <= 6) KA_LAST(6);
    else KA_LAST(8);
#undef KA_LAST
    KA_LAUNCH_CHECK();
    return 1;
}
