// Kernels of a routed mixture of gated feed-forwards: the router's choice, the experts' linears for every (token,
// choice) pair by itself (any sizes, fp32 or bf16 storage, fp32 sums in a fixed order), the list of pairs by expert
// that the matrix-core kernel of the bf16 path walks over, and the weighted sum of what the experts returned.
//
// A pair is p = token * top + choice. chosen[p] names the router's output that the token chose there: a number below
// n_experts is an expert with weights, a number from n_experts on an identity expert whose output is the token's input.
#include "ka_common.h"
#include "ka_route.h"
#include "ka_rows.h"

// (a launch of its own, a workgroup a token)
template <int PER_LANE>
__global__ void __launch_bounds__(KA_WAVE) route_kernel(RouteArgs job) {
    __shared__ RouteRoom<PER_LANE> room;
    ka_route_token<PER_LANE>(job, blockIdx.x, threadIdx.x, room);
}

KA_API int ka_route(const float* logits, long stride, const float* correction, int n, int R, int top, int n_groups, int keep,
                    int group_best, float scale, int mode, int always, int* chosen, float* weights, hipStream_t stream) {
    const RouteArgs job{logits, stride, correction, R, top, n_groups, keep, group_best, mode, always, scale, chosen, weights};
    if (ka_route_check("ka_route", job, n)) return -1;
    if (n == 0) return 0;
    if (R <= KA_WAVE) hipLaunchKernelGGL(route_kernel<1>, dim3(n), dim3(KA_WAVE), 0, stream, job);
    else if (R <= 2 * KA_WAVE) hipLaunchKernelGGL(route_kernel<2>, dim3(n), dim3(KA_WAVE), 0, stream, job);
    else hipLaunchKernelGGL((route_kernel<EX_MAX_OUTPUTS / KA_WAVE>), dim3(n), dim3(KA_WAVE), 0, stream, job);
    KA_LAUNCH_CHECK();
    return 0;
}

// ----------------------------------------------------------------------------
// The linear of every pair's expert, pair by pair: out[p] = act(a[p / a_div] W_e^T) with e = chosen[p] and W [E, N, K].
// Gated (KA_ACT_GATED): rows 2j and 2j + 1 of W_e are gate and value of output j. A pair whose choice is no expert with
// weights (>= E) is passed over. A workgroup takes EX_COLS outputs of one pair; the input row lies in LDS as fp32; a wave
// computes an output as lanes' partial sums over K met in a fixed tree.
// ----------------------------------------------------------------------------
constexpr int EX_COLS = 16;

// R rows of weights against one row of inputs: the rows' loads are in flight together and share the input's. A row's sum is
// made in the order it would be made in alone.
template <typename T, int R>
__device__ __forceinline__ void ex_dots(const T* const (&w)[R], const float* __restrict__ a, int K, int lane, bool vectors, float (&y)[R]) {
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.f;
    if (vectors) {
        constexpr int V = 16 / sizeof(T);
        typedef __attribute__((ext_vector_type(V))) T vec;
#pragma unroll 2
        for (int c = lane * V; c < K; c += KA_WAVE * V) {
            vec x[R];
#pragma unroll
            for (int r = 0; r < R; ++r) x[r] = *reinterpret_cast<const vec*>(w[r] + c);
#pragma unroll
            for (int e = 0; e < V; ++e) {
                const float h = a[c + e];
#pragma unroll
                for (int r = 0; r < R; ++r) acc[r] = fmaf(ka_to_float(x[r][e]), h, acc[r]);
            }
        }
    } else {
        for (int c = lane; c < K; c += KA_WAVE)
#pragma unroll
            for (int r = 0; r < R; ++r) acc[r] = fmaf(ka_to_float(w[r][c]), a[c], acc[r]);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) y[r] = ka_wave_sum(acc[r]);
}

// The same for bf16 rows of at most AHEAD times 512: all that a wave reads of R rows is on its way at once and before the input row has been staged, one
// trip to memory in place of up to eight. Which lane adds what in which order is as above. First and second linear, us, the loop above and this:
// experts of 4,096 x 896, 6 pairs 24.9 + 12.2 and 21.6 + 9.6, 18 pairs 51.8 + 29.7 and 47.8 + 21.4; 2,048 x 704, 5 pairs 9.3 + 5.3 and 9.4 + 5.4,
// 10 pairs 14.6 + 8.6 and 12.4 + 7.2, 20 pairs 24.3 + 14.7 and 21.5 + 11.8. R: four rows of up to 4,096 are 128 registers; eight rows of 2,048, as many
// registers, are behind four of them twice (10 pairs 14.3 against 12.4).
typedef __attribute__((ext_vector_type(8))) bf16_t ex_bf16x8;
template <int R, int AHEAD>
struct ExRows {
    ex_bf16x8 x[AHEAD][R];
    __device__ __forceinline__ void fetch(const bf16_t* const (&w)[R], int K, int lane) {
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
#pragma unroll
            for (int r = 0; r < R; ++r) x[i][r] = __builtin_nontemporal_load(reinterpret_cast<const ex_bf16x8*>(w[r] + min((i * KA_WAVE + lane) * 8, K - 8)));
    }
    __device__ __forceinline__ void dots(const float* __restrict__ a, int K, int lane, float (&y)[R]) const {
        float acc[R];
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] = 0.f;
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            const int c = (i * KA_WAVE + lane) * 8;
            if (c >= K) continue;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float h = a[c + e];
#pragma unroll
                for (int r = 0; r < R; ++r) acc[r] = fmaf(ka_to_float(x[i][r][e]), h, acc[r]);
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) y[r] = ka_wave_sum(acc[r]);
    }
};

// AHEAD 0: any K, alignment and type; else bf16 rows in whole pieces of eight, at most 512 AHEAD of them.
template <typename T, int AHEAD>
__global__ void __launch_bounds__(256)
experts_linear_kernel(const T* __restrict__ a, long a_stride, int a_div, const T* __restrict__ W, const int* __restrict__ chosen,
                      int E, int N, int K, int act, KaGateClamp clamp, void* __restrict__ out, long out_stride, int out_f32) {
    extern __shared__ float row[];
    const int p = blockIdx.y;
    const int e = chosen[p];
    if (e < 0 || e >= E) return;
    const T* ap = a + (size_t)(p / a_div) * a_stride;
    const int wave = threadIdx.x / KA_WAVE, lane = threadIdx.x % KA_WAVE;
    const bool gated = ka_act_gated(act);
    const int n_out = gated ? N / 2 : N;
    const T* We = W + (size_t)e * N * K;
    const bool vectors = K % (16 / sizeof(T)) == 0 && reinterpret_cast<uintptr_t>(W) % 16 == 0;
    constexpr int ROWS = EX_COLS / 4;           // outputs of a wave: four neighbours, or (gated) two pairs at a time
    const int j0 = blockIdx.x * EX_COLS + wave * ROWS;
    float y[ROWS];
    if constexpr (AHEAD > 0) {
        // (rows past the end: not stored)
        constexpr int R = AHEAD <= 2 ? 2 * ROWS : ROWS;
        auto stage = [&]() {
            for (int c = threadIdx.x * 8; c < K; c += blockDim.x * 8) {
                const ex_bf16x8 v = *reinterpret_cast<const ex_bf16x8*>(ap + c);
#pragma unroll
                for (int i = 0; i < 8; ++i) row[c + i] = ka_to_float(v[i]);
            }
            __syncthreads();
        };
        if (gated) {
#pragma unroll
            for (int q = 0; q < ROWS; q += R / 2) {
                const T* w[R];
#pragma unroll
                for (int r = 0; r < R; ++r) w[r] = We + (size_t)min(2 * (j0 + q) + r, N - 1) * K;
                ExRows<R, AHEAD> rows;
                rows.fetch(w, K, lane);
                if (q == 0) stage();
                float s[R];
                rows.dots(row, K, lane, s);
#pragma unroll
                for (int r = 0; r < R; r += 2) y[q + r / 2] = ka_gate_product<false>(act, clamp, s[r], s[r + 1]);
            }
        } else {
            const T* w[ROWS];
#pragma unroll
            for (int r = 0; r < ROWS; ++r) w[r] = We + (size_t)min(j0 + r, N - 1) * K;
            ExRows<ROWS, AHEAD> rows;
            rows.fetch(w, K, lane);
            stage();
            rows.dots(row, K, lane, y);
        }
    } else {
        for (int c = threadIdx.x; c < K; c += blockDim.x) row[c] = ka_to_float(ap[c]);
        __syncthreads();
        if (j0 >= n_out) return;
        if (gated) {
#pragma unroll
            for (int q = 0; q < ROWS; q += 2) {
                const T* w[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) w[r] = We + (size_t)min(2 * (j0 + q) + r, N - 1) * K;     // (rows past the end: not stored)
                float s[4];
                ex_dots<T, 4>(w, row, K, lane, vectors, s);
                y[q] = ka_gate_product<false>(act, clamp, s[0], s[1]);
                y[q + 1] = ka_gate_product<false>(act, clamp, s[2], s[3]);
            }
        } else {
            const T* w[ROWS];
#pragma unroll
            for (int r = 0; r < ROWS; ++r) w[r] = We + (size_t)min(j0 + r, N - 1) * K;
            ex_dots<T, ROWS>(w, row, K, lane, vectors, y);
        }
    }
    if (!gated && ka_act_base(act))
#pragma unroll
        for (int r = 0; r < ROWS; ++r) y[r] = ka_activate(act, y[r]);
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            if (j0 + r >= n_out) break;
            if (out_f32) reinterpret_cast<float*>(out)[(size_t)p * out_stride + j0 + r] = y[r];
            else reinterpret_cast<T*>(out)[(size_t)p * out_stride + j0 + r] = ka_from_float<T>(y[r]);
        }
    }
}

KA_API int ka_experts_linear(const void* a, long a_stride, int a_div, const void* W, int dtype, const int* chosen, int n_pairs,
                             int E, int N, int K, int act, int clamped, float limit, float slope, float shift, void* out,
                             long out_stride, int out_f32, hipStream_t stream) {
    const char* who = "ka_experts_linear";
    KA_CHECK(!clamped || ka_act_gated(act), "%s: clamps are a gated linear's", who);
    const KaGateClamp clamp{clamped, limit, slope, shift};
    KA_CHECK(n_pairs >= 0 && E > 0 && N > 0 && K > 0 && a_div > 0, "%s: bad sizes", who);
    KA_CHECK(ka_act_known(act) && (!ka_act_gated(act) || N % 2 == 0), "%s: unknown activation %d, or a gated linear of %d rows", who, act, N);
    KA_CHECK(dtype == KA_F32 || dtype == KA_BF16, "%s: unsupported dtype %d", who, dtype);
    KA_CHECK(a_stride >= K && out_stride >= ka_act_outputs(act, N), "%s: a row stride is smaller than its row", who);
    KA_CHECK((size_t)K * sizeof(float) <= 64 * 1024, "%s: rows of %d numbers do not fit in LDS", who, K);
    KA_CHECK(n_pairs <= 65535, "%s: too many pairs %d", who, n_pairs);
    if (n_pairs == 0) return 0;
    dim3 grid((ka_act_outputs(act, N) + EX_COLS - 1) / EX_COLS, n_pairs);
    const size_t lds = (size_t)K * sizeof(float);
    const bool pieces = K % 8 == 0 && a_stride % 8 == 0 && ((uintptr_t)a | (uintptr_t)W) % 16 == 0;
#define EX_LINEAR(T, AHEAD)                                                                                                                    \
    hipLaunchKernelGGL((experts_linear_kernel<T, AHEAD>), grid, dim3(256), lds, stream, (const T*)a, a_stride, a_div, (const T*)W, chosen, E, N, K, act, clamp, \
                       out, out_stride, out_f32)
    // As few pieces ahead as the rows have (one past the end is a load for nothing). Rows of up to 512 are one trip either way, and the plain loop is
    // ahead (8 pairs' second linear of 512 to 1,024: 2.9 and 3.7 us).
    if (dtype == KA_F32) EX_LINEAR(float, 0);
    else if (pieces && K > 512 && K <= 1024) EX_LINEAR(bf16_t, 2);
    else if (pieces && K > 1024 && K <= 2048) EX_LINEAR(bf16_t, 4);
    else if (pieces && K > 2048 && K <= 4096) EX_LINEAR(bf16_t, 8);
    else EX_LINEAR(bf16_t, 0);
#undef EX_LINEAR
    KA_LAUNCH_CHECK();
    return 0;
}

// ----------------------------------------------------------------------------
// The weighted sum: out[t] (=, or += if accumulate) sum_k weights[t, k] * (chosen[t, k] < E ? y[t * top + k] : h[t])
//     + sigmoid(shared_gate[t]) * shared[t]       (shared optional; without a gate its weight is 1).
// y fp32 [n top, dim], h of type T (the experts' input), shared fp32 [n, dim], out fp32 [n, dim].
// ----------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256)
experts_combine_kernel(const float* __restrict__ y, const T* __restrict__ h, long h_stride, const int* __restrict__ chosen,
                       const float* __restrict__ weights, int top, int E, const float* __restrict__ shared,
                       const float* __restrict__ shared_gate, long gate_stride, float* __restrict__ out, int dim, int accumulate) {
    const int t = blockIdx.x;
    const float sg = shared ? (shared_gate ? 1.0f / (1.0f + expf(-shared_gate[(size_t)t * gate_stride])) : 1.f) : 0.f;
    for (int c = threadIdx.x; c < dim; c += blockDim.x) {
        float acc = 0.f;
        for (int k = 0; k < top; ++k) {
            const int e = chosen[(size_t)t * top + k];
            const float v = e < E ? y[((size_t)t * top + k) * dim + c] : ka_to_float(h[(size_t)t * h_stride + c]);
            acc = fmaf(weights[(size_t)t * top + k], v, acc);
        }
        if (shared) acc = fmaf(sg, shared[(size_t)t * dim + c], acc);
        float* o = out + (size_t)t * dim + c;
        *o = accumulate ? *o + acc : acc;
    }
}

KA_API int ka_experts_combine(const float* y, const void* h, long h_stride, int dtype, const int* chosen, const float* weights, int n,
                              int top, int E, const float* shared, const float* shared_gate, long gate_stride, float* out, int dim,
                              int accumulate, hipStream_t stream) {
    KA_CHECK(n >= 0 && top > 0 && dim > 0 && h_stride >= dim, "ka_experts_combine: bad sizes");
    KA_CHECK(dtype == KA_F32 || dtype == KA_BF16, "ka_experts_combine: unsupported dtype %d", dtype);
    if (n == 0) return 0;
    if (dtype == KA_F32)
        hipLaunchKernelGGL(experts_combine_kernel<float>, dim3(n), dim3(256), 0, stream, y, (const float*)h, h_stride, chosen, weights, top,
                           E, shared, shared_gate, gate_stride, out, dim, accumulate);
    else
        hipLaunchKernelGGL(experts_combine_kernel<bf16_t>, dim3(n), dim3(256), 0, stream, y, (const bf16_t*)h, h_stride, chosen, weights,
                           top, E, shared, shared_gate, gate_stride, out, dim, accumulate);
    KA_LAUNCH_CHECK();
    return 0;
}

// ----------------------------------------------------------------------------
// The weighted sum of ka_experts_combine as the output of a sublayer whose norm stands behind it: it is normalised and
// added into the fp32 stream x, and the norm of the new rows is computed, in the same launch (ka_rows.h). A workgroup
// per token; the sums are those of ka_experts_combine, in its order. In fp32 h_in may be x itself (a thread reads its channels of a row before it
// writes them), so neither is __restrict__.
// ----------------------------------------------------------------------------
template <typename T, int PIECES, int THREADS>
__global__ void __launch_bounds__(THREADS)
experts_combine_normed_kernel(const float* __restrict__ y, const T* h_in, long h_stride, const int* __restrict__ chosen,
                              const float* __restrict__ weights, int top, int E, const float* __restrict__ shared,
                              const float* __restrict__ shared_gate, long gate_stride, float* x, int dim, KaRowNorms a) {
    __shared__ float smem[THREADS / KA_WAVE];
    const int t = blockIdx.x;
    const float sg = shared ? (shared_gate ? 1.0f / (1.0f + expf(-shared_gate[(size_t)t * gate_stride])) : 1.f) : 0.f;
    auto one = [&](int c) {
        float acc = 0.f;
        for (int k = 0; k < top; ++k) {
            const int e = chosen[(size_t)t * top + k];
            const float v = e < E ? y[((size_t)t * top + k) * dim + c] : ka_to_float(h_in[(size_t)t * h_stride + c]);
            acc = fmaf(weights[(size_t)t * top + k], v, acc);
        }
        return shared ? fmaf(sg, shared[(size_t)t * dim + c], acc) : acc;
    };
    // (everything a piece needs is asked for at once, eight choices at a time and nothing behind a branch; an identity expert has a
    // row in `y` too, which is not used)
    auto piece = [&](int c) {
        const T* hp = h_in + (size_t)t * h_stride + c;
        const float4 own = make_float4(ka_to_float(hp[0]), ka_to_float(hp[1]), ka_to_float(hp[2]), ka_to_float(hp[3]));
        const float4 common = shared ? *reinterpret_cast<const float4*>(shared + (size_t)t * dim + c) : make_float4(0.f, 0.f, 0.f, 0.f);
        constexpr int AHEAD = PIECES == 1 ? 8 : 4;
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int k0 = 0; k0 < top; k0 += AHEAD) {
            float4 v[AHEAD];
            float w[AHEAD];
            bool has[AHEAD];
#pragma unroll
            for (int k = 0; k < AHEAD; ++k) {
                const size_t at = (size_t)t * top + min(k0 + k, top - 1);
                w[k] = weights[at];
                has[k] = chosen[at] < E;
                v[k] = *reinterpret_cast<const float4*>(y + at * dim + c);
            }
#pragma unroll
            for (int k = 0; k < AHEAD; ++k) {
                if (k0 + k >= top) continue;
                const float4 z = has[k] ? v[k] : own;
                acc.x = fmaf(w[k], z.x, acc.x);
                acc.y = fmaf(w[k], z.y, acc.y);
                acc.z = fmaf(w[k], z.z, acc.z);
                acc.w = fmaf(w[k], z.w, acc.w);
            }
        }
        if (shared) {
            acc.x = fmaf(sg, common.x, acc.x);
            acc.y = fmaf(sg, common.y, acc.y);
            acc.z = fmaf(sg, common.z, acc.z);
            acc.w = fmaf(sg, common.w, acc.w);
        }
        return acc;
    };
    ka_finish_row<PIECES, THREADS>(x, t, dim, a, piece, one, smem);
}

KA_API int ka_experts_combine_normed(const float* y, const void* h_in, long h_stride, int dtype, const int* chosen, const float* weights,
                                     int n, int top, int E, const float* shared, const float* shared_gate, long gate_stride, float* x,
                                     int dim, const float* gain, float eps, const float* gain2, float eps2, void* h, hipStream_t stream) {
    const char* who = "ka_experts_combine_normed";
    KA_CHECK(n >= 0 && top > 0 && dim > 0 && h_stride >= dim && eps >= 0.f && eps2 >= 0.f && gain != nullptr, "%s: bad sizes", who);
    KA_CHECK(dtype == KA_F32 || dtype == KA_BF16, "%s: unsupported dtype %d", who, dtype);
    KA_CHECK(gain2 == nullptr || h != nullptr, "%s: the second norm needs its rows", who);
    if (n == 0) return 0;
    const KaRowNorms a{gain, eps, gain2, eps2, h, dtype == KA_BF16};
    const int pieces = (uintptr_t)shared % 16 == 0 ? ka_row_pieces(n, dim, x, y, a) : 0;
#define EX_COMBINE(T, P, THREADS)                                                                                                  \
    hipLaunchKernelGGL((experts_combine_normed_kernel<T, P, THREADS>), dim3(n), dim3(THREADS), 0, stream, y, (const T*)h_in, h_stride, chosen, \
                       weights, top, E, shared, shared_gate, gate_stride, x, dim, a)
#define EX_COMBINE_F32(P, THREADS) EX_COMBINE(float, P, THREADS)
#define EX_COMBINE_BF16(P, THREADS) EX_COMBINE(bf16_t, P, THREADS)
    if (dtype == KA_F32) { KA_ROW_CASES(pieces, EX_COMBINE_F32) } else { KA_ROW_CASES(pieces, EX_COMBINE_BF16) }
#undef EX_COMBINE_F32
#undef EX_COMBINE_BF16
#undef EX_COMBINE
    KA_LAUNCH_CHECK();
    return 0;
}

// ----------------------------------------------------------------------------
// The pairs listed by expert, for kernels that take an expert's pairs together: one workgroup counts the pairs of
// every expert, lays the experts' runs one behind the other, each run starting on a multiple of `tile` rows of the
// list, and fills them. sorted [capacity] holds pair numbers (-1 in the unused rows of a run's last tile);
// tile_expert [capacity / tile] the expert of every tile of the list (-1 behind the last run). Pairs of identity experts
// are in no run. Which row of its run a pair gets depends on the order the threads arrive in; nothing computed from the
// list depends on it (every pair's result is computed from its own row alone).
// capacity >= n_pairs rounded up to tiles + E tiles.
// ----------------------------------------------------------------------------
__global__ void __launch_bounds__(1024)
experts_sort_kernel(const int* __restrict__ chosen, int n_pairs, int E, int tile, int capacity, int* __restrict__ sorted,
                    int* __restrict__ tile_expert) {
    __shared__ int count[EX_MAX_OUTPUTS];
    __shared__ int start[EX_MAX_OUTPUTS + 1];
    const int tid = threadIdx.x;
    for (int e = tid; e < E; e += blockDim.x) count[e] = 0;
    for (int i = tid; i < capacity; i += blockDim.x) sorted[i] = -1;
    __syncthreads();
    for (int p = tid; p < n_pairs; p += blockDim.x) {
        const int e = chosen[p];
        if (e >= 0 && e < E) atomicAdd(&count[e], 1);
    }
    __syncthreads();
    if (tid == 0) {
        int at = 0;
        for (int e = 0; e < E; ++e) {
            start[e] = at;
            at += (count[e] + tile - 1) / tile * tile;
        }
        start[E] = at;
    }
    __syncthreads();
    const int tiles = capacity / tile;
    for (int i = tid; i < tiles; i += blockDim.x) {
        // the expert whose run holds row i * tile: the last one that starts at or before it and is not empty there
        int e_of = -1;
        const int at = i * tile;
        if (at < start[E]) {
            int lo = 0, hi = E - 1;
            while (lo < hi) {
                const int mid = (lo + hi + 1) / 2;
                if (start[mid] <= at) lo = mid; else hi = mid - 1;
            }
            e_of = lo;
        }
        tile_expert[i] = e_of;
    }
    for (int e = tid; e < E; e += blockDim.x) count[e] = 0;
    __syncthreads();
    for (int p = tid; p < n_pairs; p += blockDim.x) {
        const int e = chosen[p];
        if (e >= 0 && e < E) sorted[start[e] + atomicAdd(&count[e], 1)] = p;
    }
}

KA_API int ka_experts_sort(const int* chosen, int n_pairs, int E, int tile, int capacity, int* sorted, int* tile_expert,
                           hipStream_t stream) {
    KA_CHECK(n_pairs >= 0 && E > 0 && E <= EX_MAX_OUTPUTS && tile > 0 && capacity % tile == 0, "ka_experts_sort: bad sizes");
    // (every expert's run may end in a tile that is not full)
    KA_CHECK((long)capacity >= (long)n_pairs + (long)E * (tile - 1), "ka_experts_sort: a list of %d rows is too short", capacity);
    hipLaunchKernelGGL(experts_sort_kernel, dim3(1), dim3(1024), 0, stream, chosen, n_pairs, E, tile, capacity, sorted, tile_expert);
    KA_LAUNCH_CHECK();
    return 0;
}
