// Kernels of a residual stream that is several copies (hyper-connections): x [n, S, dim] fp32. One launch stands between two
// sublayers: it writes the output y of the one before into the streams, all of them at once from the old ones,
//     x_t <- sum_s mix[s, t] x_s + out[t] y,
// reads what the next sublayer sees, u = sum_t into[t] x_t, and leaves that sublayer's norm of u in h. All arithmetic is fp32.
// What computes y is the caller's business: a load, or the weighted sum of a routed mixture's experts.
#include "ka_common.h"
#include "ka_route.h"
#include "ka_rows.h"

// A workgroup has a row. Of many rows each gets 256 threads and a thread several pieces of it; where there are fewer rows than two a
// CU (a decode step) a row gets a thread per piece, up to 1,024: it then waits for memory once (48 rows of four streams of
// 4,096: 11 -> 5.1 us between sublayers and 24 -> 8.3 behind six experts).
constexpr int ST_THREADS = KA_ROW_THREADS;
constexpr int ST_MAX_STREAMS = 16;

struct StreamArgs {
    float* x;                   // [rows of the stream, S, dim]
    const float* embedded;      // [n, dim]: every stream starts as this row (x is written only); null: x is read
    const float* mix;           // [S, S] from, to; null: nothing is written into the streams
    const float* out;           // [S]
    const float* into;          // [S]; null: the sum of the streams is read
    const int* rows;            // rows of x that are read (nothing is written then), all inside x; null: row i
    const float* gain;
    const float* bias;          // may be null
    float eps;
    int rms;                    // 0: layer norm, 1: root mean square alone
    void* h;                    // [n, dim]; null: nothing is read
    int h_bf16;
    int S, dim;
};

__device__ __forceinline__ float4 st_fma4(float a, const float4& b, const float4& c) {
    return make_float4(fmaf(a, b.x, c.x), fmaf(a, b.y, c.y), fmaf(a, b.z, c.z), fmaf(a, b.w, c.w));
}

// S streams in registers, PIECES pieces of four channels a thread (dim a multiple of 4 and at most 4 PIECES THREADS, rows
// 16-byte aligned). `piece(c)` gives y of the channels c .. c + 3. `early()` runs behind the first requests, `keep(c, b)` sees the bf16 rows of h.
typedef __attribute__((ext_vector_type(4))) __bf16 st_bf16x4;

template <int S, int PIECES, int THREADS, typename Piece, typename Early, typename Keep>
__device__ __forceinline__ void st_step_regs(const StreamArgs& a, Piece piece, float* smem, Early early, Keep keep) {
    const int i = blockIdx.x, dim = a.dim;
    float* row = a.x + (size_t)(a.rows ? a.rows[i] : i) * S * dim;
    float m[S][S], o[S], in[S];
    const bool writes = a.mix != nullptr;
    // The numbers of the streams and (of short rows) the norm's are asked for behind the row and arrive with it; where they are used they would come behind what `early`
    // asks for. (A step without that: 2.8 us at one row of four streams of 2,048 either way.)
    auto numbers = [&] {
        if (writes) {
#pragma unroll
            for (int s = 0; s < S; ++s) {
#pragma unroll
                for (int t = 0; t < S; ++t) m[s][t] = a.mix[s * S + t];
                o[s] = a.out[s];
            }
        }
#pragma unroll
        for (int s = 0; s < S; ++s) in[s] = a.into ? a.into[s] : 1.f;
    };
    constexpr bool NORM_EARLY = PIECES <= 2;
    float4 gain[PIECES], bias[PIECES];
    auto norm_of = [&](int p) {
        const int c = min(ka_row_channel<THREADS>(p), dim - 4);
        const float* const g = a.h ? a.gain : row;                  // (without a norm any address; not used)
        gain[p] = *reinterpret_cast<const float4*>(g + c);
        bias[p] = *reinterpret_cast<const float4*>((a.h && a.bias ? a.bias : g) + c);
    };
    float4 u[PIECES];
    float sum[PIECES], ss[PIECES];
    // (all that a few pieces need is asked for before anything is stored)
    constexpr int AT_ONCE = PIECES < 4 ? PIECES : 4;
#pragma unroll
    for (int p0 = 0; p0 < PIECES; p0 += AT_ONCE) {
        float4 v[AT_ONCE][S], y[AT_ONCE];
#pragma unroll
        for (int p = 0; p < AT_ONCE; ++p) {
            const int c = ka_row_channel<THREADS>(p0 + p);
            if (c >= dim) continue;
            if (a.embedded) {
                v[p][0] = *reinterpret_cast<const float4*>(a.embedded + (size_t)i * dim + c);
            } else {
#pragma unroll
                for (int s = 0; s < S; ++s) v[p][s] = *reinterpret_cast<const float4*>(row + (size_t)s * dim + c);
            }
            if (writes) y[p] = piece(c);
        }
        if (p0 == 0) {
            if constexpr (NORM_EARLY) {
#pragma unroll
                for (int p = 0; p < PIECES; ++p) norm_of(p);
            }
            numbers();
            early();
        }
#pragma unroll
        for (int p = 0; p < AT_ONCE; ++p) {
            const int c = ka_row_channel<THREADS>(p0 + p);
            float4& sums = u[p0 + p];
            sums = make_float4(0.f, 0.f, 0.f, 0.f);
            sum[p0 + p] = 0.f;
            if (c >= dim) continue;
            if (a.embedded) {
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    v[p][s] = v[p][0];
                    *reinterpret_cast<float4*>(row + (size_t)s * dim + c) = v[p][0];
                }
            }
            if (writes) {
#pragma unroll
                for (int t = 0; t < S; ++t) {
                    float4 w = make_float4(o[t] * y[p].x, o[t] * y[p].y, o[t] * y[p].z, o[t] * y[p].w);
#pragma unroll
                    for (int s = 0; s < S; ++s) w = st_fma4(m[s][t], v[p][s], w);
                    *reinterpret_cast<float4*>(row + (size_t)t * dim + c) = w;
                    sums = st_fma4(in[t], w, sums);
                }
            } else {
#pragma unroll
                for (int s = 0; s < S; ++s) sums = st_fma4(in[s], v[p][s], sums);
            }
            sum[p0 + p] = (sums.x + sums.y) + (sums.z + sums.w);
        }
    }
    if (a.h == nullptr) return;
    const float mean = a.rms ? 0.f : ka_pieces_sum<PIECES, THREADS>(sum, smem) / (float)dim;
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
        ss[p] = 0.f;
        if (ka_row_channel<THREADS>(p) < dim) {
            u[p] = make_float4(u[p].x - mean, u[p].y - mean, u[p].z - mean, u[p].w - mean);
            ss[p] = ka_squares(u[p]);
        }
    }
    const float r = 1.0f / sqrtf(ka_pieces_sum<PIECES, THREADS>(ss, smem) / (float)dim + a.eps);
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
        const int c = ka_row_channel<THREADS>(p);
        if (c < dim) {
            if constexpr (!NORM_EARLY) norm_of(p);
            const float4 g = gain[p];
            float4 v = make_float4(u[p].x * r * g.x, u[p].y * r * g.y, u[p].z * r * g.z, u[p].w * r * g.w);
            if (a.bias) v = make_float4(v.x + bias[p].x, v.y + bias[p].y, v.z + bias[p].z, v.w + bias[p].w);
            if (a.h_bf16) {
                st_bf16x4 b;
                b[0] = (bf16_t)v.x;
                b[1] = (bf16_t)v.y;
                b[2] = (bf16_t)v.z;
                b[3] = (bf16_t)v.w;
                *reinterpret_cast<st_bf16x4*>(reinterpret_cast<bf16_t*>(a.h) + (size_t)i * dim + c) = b;
                keep(c, b);
            } else {
                *reinterpret_cast<float4*>(reinterpret_cast<float*>(a.h) + (size_t)i * dim + c) = v;
            }
        }
    }
}

template <int S, int PIECES, int THREADS, typename Piece>
__device__ __forceinline__ void st_step_regs(const StreamArgs& a, Piece piece, float* smem) {
    st_step_regs<S, PIECES, THREADS>(a, piece, smem, [] {}, [](int, const st_bf16x4&) {});
}

// Any number of streams up to ST_MAX_STREAMS, any dim. `one(c)` gives y of channel c.
template <typename One>
__device__ __forceinline__ void st_step_any(const StreamArgs& a, One one, float* smem) {
    const int i = blockIdx.x, tid = threadIdx.x, dim = a.dim, S = a.S;
    float* row = a.x + (size_t)(a.rows ? a.rows[i] : i) * S * dim;
    const bool writes = a.mix != nullptr;
    auto read = [&](int c) {
        float u = 0.f;
        for (int s = 0; s < S; ++s) u = fmaf(a.into ? a.into[s] : 1.f, row[(size_t)s * dim + c], u);
        return u;
    };
    float sum = 0.f;
    for (int c = tid; c < dim; c += ST_THREADS) {
        if (a.embedded) {
            const float e = a.embedded[(size_t)i * dim + c];
            for (int s = 0; s < S; ++s) row[(size_t)s * dim + c] = e;
        }
        if (writes) {
            float v[ST_MAX_STREAMS];
#pragma unroll
            for (int s = 0; s < ST_MAX_STREAMS; ++s) v[s] = s < S ? row[(size_t)s * dim + c] : 0.f;
            const float y = one(c);
            for (int t = 0; t < S; ++t) {
                float w = a.out[t] * y;
#pragma unroll
                for (int s = 0; s < ST_MAX_STREAMS; ++s)
                    if (s < S) w = fmaf(a.mix[s * S + t], v[s], w);
                row[(size_t)t * dim + c] = w;
            }
        }
        if (a.h) sum += read(c);              // (a thread reads its own writes)
    }
    if (a.h == nullptr) return;
    const float mean = a.rms ? 0.f : ka_row_sum(sum, smem) / (float)dim;
    float ss = 0.f;
    for (int c = tid; c < dim; c += ST_THREADS) {
        const float u = read(c) - mean;
        ss += u * u;
    }
    const float r = 1.0f / sqrtf(ka_row_sum(ss, smem) / (float)dim + a.eps);
    for (int c = tid; c < dim; c += ST_THREADS) {
        float v = (read(c) - mean) * r * a.gain[c];
        if (a.bias) v += a.bias[c];
        if (a.h_bf16) reinterpret_cast<bf16_t*>(a.h)[(size_t)i * dim + c] = (bf16_t)v;
        else reinterpret_cast<float*>(a.h)[(size_t)i * dim + c] = v;
    }
}

template <int S, int PIECES, int THREADS>
__global__ void __launch_bounds__(THREADS) streams_step_kernel(StreamArgs a, const float* __restrict__ y) {
    __shared__ float smem[THREADS / KA_WAVE];
    const float* yr = y ? y + (size_t)blockIdx.x * a.dim : nullptr;
    if constexpr (S > 0)
        st_step_regs<S, PIECES, THREADS>(a, [&](int c) { return *reinterpret_cast<const float4*>(yr + c); }, smem);
    else
        st_step_any(a, [&](int c) { return yr[c]; }, smem);
}

// The step in front of a routed mixture, of few rows: the same row's router logits and its choice in the launch that leaves h. The router's linear of few rows is a
// handful of workgroups that wait for memory, and the choice behind it a wave a row that waits again; here the router's weights (120 to 500 KB, from L2 for all rows
// but the first) are asked for beside the streams, in registers, and h meets them out of LDS: a wave takes every (THREADS / 64)-th output.
// A row's numbers depend on that row alone. One CU brings the weights at 30 to 40 GB/s beyond the first trip, so long rows gain only where the linear alone is slow
// (us, 30 outputs of 2,048, one row: step, linear and choice 9.4, this 7.5; 62 of 4,096: 11.9 and 15.7, 40 rows 21.4 and 16.5). 1,024 threads leave 128 registers,
// which one output ahead takes up (eight values spill); with two ahead 25.8 us.
struct StreamRoute {
    const bf16_t* router;       // [outputs, dim], rows ld apart
    long ld;
    int outputs;                // rows of the router's linear: those of the choice, and what else rides along
    const float* bias;          // [outputs] or null
    float* logits;              // [n, >= outputs], rows logits_ld apart
    long logits_ld;
};
constexpr int ST_ROUTE_OUTPUTS = 128;

template <int S, int THREADS>
__global__ void __launch_bounds__(THREADS) streams_route_kernel(StreamArgs a, const float* __restrict__ y, StreamRoute q, RouteArgs choice) {
    typedef __attribute__((ext_vector_type(8))) __bf16 st_bf16x8;
    constexpr int WAVES = THREADS / KA_WAVE, LOADS = THREADS * 4 / (8 * KA_WAVE), AHEAD = THREADS == 512 ? 4 : 1;     // loads of 16 bytes a lane and output; outputs asked for ahead
    __shared__ float smem[WAVES], logits[ST_ROUTE_OUTPUTS];
    __shared__ __attribute__((aligned(16))) bf16_t row[THREADS * 4];
    __shared__ RouteRoom<1> room;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KA_WAVE), lane = threadIdx.x % KA_WAVE, dim = a.dim;
    const float* yr = y + (size_t)blockIdx.x * dim;
    st_bf16x8 w[AHEAD][LOADS];
    auto ask = [&](st_bf16x8 (&to)[LOADS], int r) {
        const bf16_t* from = q.router + (size_t)min(r, q.outputs - 1) * q.ld;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) to[i] = *reinterpret_cast<const st_bf16x8*>(from + min((i * KA_WAVE + lane) * 8, dim - 8));
    };
    st_step_regs<S, 1, THREADS>(
        a, [&](int c) { return *reinterpret_cast<const float4*>(yr + c); }, smem,
        [&] {
#pragma unroll
            for (int g = 0; g < AHEAD; ++g) ask(w[g], wave + g * WAVES);
        },
        [&](int c, const st_bf16x4& b) { *reinterpret_cast<st_bf16x4*>(row + c) = b; });
    __syncthreads();
    st_bf16x8 h[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) h[i] = *reinterpret_cast<const st_bf16x8*>(row + (i * KA_WAVE + lane) * 8);
    for (int r0 = wave; r0 < q.outputs; r0 += AHEAD * WAVES) {
#pragma unroll
        for (int g = 0; g < AHEAD; ++g) {
            const int r = r0 + g * WAVES;
            float sum = 0.f;
#pragma unroll
            for (int i = 0; i < LOADS; ++i) {
                float part = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) part = fmaf((float)w[g][i][e], (float)h[i][e], part);
                sum += (i * KA_WAVE + lane) * 8 < dim ? part : 0.f;
            }
            ask(w[g], r + AHEAD * WAVES);
            sum = ka_wave_sum(sum);
            if (r < q.outputs && lane == 0) {
                if (q.bias) sum += q.bias[r];
                logits[r] = sum;
                q.logits[(size_t)blockIdx.x * q.logits_ld + r] = sum;
            }
        }
    }
    __syncthreads();
    if (wave > 0) return;
    choice.logits = logits;
    choice.stride = 0;
    ka_route_token<1>(choice, blockIdx.x, lane, room);
}

// y = sum_k weights[t, k] * (chosen[t, k] < E ? pairs[t top + k] : h_in[t]) + sigmoid(shared_gate[t]) * shared[t], as
// ka_experts_combine makes it, in its order.
struct StreamExperts {
    const float* pairs;         // [n top, dim]
    const void* h_in;
    long h_stride;
    const int* chosen;
    const float* weights;
    int top, E;
    const float* shared;
    const float* shared_gate;
    long gate_stride;
};

template <typename T, int S, int PIECES, int THREADS>
__global__ void __launch_bounds__(THREADS) streams_experts_kernel(StreamArgs a, StreamExperts e) {
    __shared__ float smem[THREADS / KA_WAVE];
    const int t = blockIdx.x, dim = a.dim;
    const T* hp = reinterpret_cast<const T*>(e.h_in) + (size_t)t * e.h_stride;
    const float sg = e.shared ? (e.shared_gate ? 1.0f / (1.0f + expf(-e.shared_gate[(size_t)t * e.gate_stride])) : 1.f) : 0.f;
    if constexpr (S > 0) {
        st_step_regs<S, PIECES, THREADS>(a, [&](int c) {
            float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
            // (everything is asked for at once, eight choices at a time and nothing behind a branch; a choice without weights of
            // its own has a row in `pairs` too, which is not used)
            const float4 own = make_float4(ka_to_float(hp[c]), ka_to_float(hp[c + 1]), ka_to_float(hp[c + 2]), ka_to_float(hp[c + 3]));
            const float4 common = e.shared ? *reinterpret_cast<const float4*>(e.shared + (size_t)t * dim + c) : make_float4(0.f, 0.f, 0.f, 0.f);
            constexpr int AHEAD = PIECES == 1 ? 8 : 4;
            for (int k0 = 0; k0 < e.top; k0 += AHEAD) {
                float4 v[AHEAD];
                float w[AHEAD];
                bool has[AHEAD];
#pragma unroll
                for (int k = 0; k < AHEAD; ++k) {
                    const size_t at = (size_t)t * e.top + min(k0 + k, e.top - 1);
                    w[k] = e.weights[at];
                    has[k] = e.chosen[at] < e.E;
                    v[k] = *reinterpret_cast<const float4*>(e.pairs + at * dim + c);
                }
#pragma unroll
                for (int k = 0; k < AHEAD; ++k)
                    if (k0 + k < e.top) acc = st_fma4(w[k], has[k] ? v[k] : own, acc);
            }
            return e.shared ? st_fma4(sg, common, acc) : acc;
        }, smem);
    } else {
        st_step_any(a, [&](int c) {
            float acc = 0.f;
            for (int k = 0; k < e.top; ++k) {
                const float v = e.chosen[(size_t)t * e.top + k] < e.E ? e.pairs[((size_t)t * e.top + k) * dim + c] : ka_to_float(hp[c]);
                acc = fmaf(e.weights[(size_t)t * e.top + k], v, acc);
            }
            return e.shared ? fmaf(sg, e.shared[(size_t)t * dim + c], acc) : acc;
        }, smem);
    }
}

// Pieces of four channels a thread holds in the form with registers, times ten, with 1 or 2 added where a row gets 512 or 1,024 threads
// (few rows); 0: the general form.
static int st_pieces(const StreamArgs& a, int n, const void* y, const void* shared) {
    const uintptr_t all = (uintptr_t)a.x | (uintptr_t)a.embedded | (uintptr_t)a.gain | (uintptr_t)a.bias | (uintptr_t)y | (uintptr_t)shared;
    if (a.S > 4 || a.dim % 4 != 0 || all % 16 != 0 || (uintptr_t)a.h % (a.h_bf16 ? 8 : 16) != 0) return 0;
    const int need = ka_cdiv(a.dim, 4 * ST_THREADS);
    if (n < 2 * ka_compute_units()) {
        if (need == 2) return 11;
        if (need > 2 && need <= 4) return 12;
        if (need > 4 && need <= 8) return 22;
    }
    for (int p : {1, 2, 4, 8})
        if (need <= p) return p * 10;
    return 0;
}

#define ST_CASES(LAUNCH, S)                \
    switch (pieces) {                      \
        case 10: LAUNCH(S, 1, 256); break; \
        case 20: LAUNCH(S, 2, 256); break; \
        case 40: LAUNCH(S, 4, 256); break; \
        case 11: LAUNCH(S, 1, 512); break; \
        case 12: LAUNCH(S, 1, 1024); break;\
        case 22: LAUNCH(S, 2, 1024); break;\
        default: LAUNCH(S, 8, 256); break; \
    }
#define ST_DISPATCH(LAUNCH)                       \
    if (pieces == 0) { LAUNCH(0, 0, 256); }       \
    else if (a.S == 1) { ST_CASES(LAUNCH, 1) }    \
    else if (a.S == 2) { ST_CASES(LAUNCH, 2) }    \
    else if (a.S == 3) { ST_CASES(LAUNCH, 3) }    \
    else { ST_CASES(LAUNCH, 4) }

static int st_check(const char* who, const StreamArgs& a, int n, int h_dtype) {
    KA_CHECK(n >= 0 && a.S > 0 && a.S <= ST_MAX_STREAMS && a.dim > 0 && a.eps >= 0.f, "%s: bad sizes (%d streams of %d)", who, a.S, a.dim);
    KA_CHECK(h_dtype == KA_F32 || h_dtype == KA_BF16, "%s: unsupported dtype %d", who, h_dtype);
    KA_CHECK((a.mix == nullptr) == (a.out == nullptr), "%s: writing needs both mix and out", who);
    KA_CHECK(a.h == nullptr || a.gain != nullptr, "%s: the norm needs its gains", who);
    KA_CHECK(a.rows == nullptr || (a.mix == nullptr && a.embedded == nullptr), "%s: chosen rows are only read", who);
    return 0;
}

KA_API int ka_streams_step(float* x, const float* embedded, const float* y, const float* mix, const float* out, const float* into,
                           const int* rows, const float* gain, const float* bias, float eps, int rms, void* h, int h_dtype, int n, int S,
                           int dim, hipStream_t stream) {
    const char* who = "ka_streams_step";
    const StreamArgs a{x, embedded, mix, out, into, rows, gain, bias, eps, rms, h, h_dtype == KA_BF16, S, dim};
    if (const int status = st_check(who, a, n, h_dtype)) return status;
    KA_CHECK((mix == nullptr) == (y == nullptr), "%s: writing needs a sublayer's output", who);
    if (n == 0) return 0;
    const int pieces = st_pieces(a, n, y, nullptr);
#define ST_LAUNCH(S_, P_, T_) hipLaunchKernelGGL((streams_step_kernel<S_, P_, T_>), dim3(n), dim3(T_), 0, stream, a, y)
    ST_DISPATCH(ST_LAUNCH)
#undef ST_LAUNCH
    KA_LAUNCH_CHECK();
    return 0;
}

// ka_streams_step of rows that are written and read, and ka_route of the logits h router^T (+ router_bias) in the same launch. 1: not covered, nothing was run.
KA_API int ka_streams_step_route(float* x, const float* y, const float* mix, const float* out, const float* into, const float* gain, const float* bias, float eps,
                                 int rms, void* h, int n, int S, int dim, const void* router, long ldr, int outputs, const float* router_bias,
                                 float* logits, long stride, const float* correction, int tokens, int R, int top, int n_groups, int keep, int group_best, float scale,
                                 int mode, int always, int* chosen, float* weights, hipStream_t stream) {
    const char* who = "ka_streams_step_route";
    const StreamArgs a{x, nullptr, mix, out, into, nullptr, gain, bias, eps, rms, h, 1, S, dim};
    if (const int status = st_check(who, a, n, KA_BF16)) return status;
    KA_CHECK(mix != nullptr && y != nullptr && h != nullptr, "%s: a step that writes and reads", who);
    const RouteArgs choice{logits, stride, correction, R, top, n_groups, keep, group_best, mode, always, scale, chosen, weights};
    if (ka_route_check(who, choice, tokens)) return -1;
    KA_CHECK(tokens == n && outputs >= R && stride >= outputs && ldr >= dim, "%s: %d outputs of which %d are chosen among, %d of %d rows", who, outputs, R, tokens, n);
    const int pieces = st_pieces(a, n, y, nullptr);
    if ((pieces != 11 && pieces != 12) || R > KA_WAVE || outputs > ST_ROUTE_OUTPUTS || dim % 8 || ldr % 8 || (uintptr_t)router % 16) return 1;
    if (n == 0) return 0;
    const StreamRoute q{(const bf16_t*)router, ldr, outputs, router_bias, logits, stride};
#define ST_ROUTE(S_)                                                                                                                  \
    case S_:                                                                                                                          \
        if (pieces == 11) hipLaunchKernelGGL((streams_route_kernel<S_, 512>), dim3(n), dim3(512), 0, stream, a, y, q, choice);        \
        else hipLaunchKernelGGL((streams_route_kernel<S_, 1024>), dim3(n), dim3(1024), 0, stream, a, y, q, choice);                   \
        break;
    switch (S) {
        ST_ROUTE(1)
        ST_ROUTE(2)
        ST_ROUTE(3)
        ST_ROUTE(4)
    }
#undef ST_ROUTE
    KA_LAUNCH_CHECK();
    return 0;
}

KA_API int ka_streams_experts(float* x, const float* pairs, const void* h_in, long h_stride, int dtype, const int* chosen,
                              const float* weights, int top, int E, const float* shared, const float* shared_gate, long gate_stride,
                              const float* mix, const float* out, const float* into, const float* gain, const float* bias, float eps,
                              int rms, void* h, int h_dtype, int n, int S, int dim, hipStream_t stream) {
    const char* who = "ka_streams_experts";
    const StreamArgs a{x, nullptr, mix, out, into, nullptr, gain, bias, eps, rms, h, h_dtype == KA_BF16, S, dim};
    if (const int status = st_check(who, a, n, h_dtype)) return status;
    KA_CHECK(mix != nullptr && top > 0 && h_stride >= dim, "%s: bad sizes", who);
    KA_CHECK(dtype == KA_F32 || dtype == KA_BF16, "%s: unsupported dtype %d", who, dtype);
    if (n == 0) return 0;
    const StreamExperts e{pairs, h_in, h_stride, chosen, weights, top, E, shared, shared_gate, gate_stride};
    const int pieces = st_pieces(a, n, pairs, shared);
#define ST_LAUNCH_F32(S_, P_, T_) hipLaunchKernelGGL((streams_experts_kernel<float, S_, P_, T_>), dim3(n), dim3(T_), 0, stream, a, e)
#define ST_LAUNCH_BF16(S_, P_, T_) hipLaunchKernelGGL((streams_experts_kernel<bf16_t, S_, P_, T_>), dim3(n), dim3(T_), 0, stream, a, e)
    if (dtype == KA_F32) { ST_DISPATCH(ST_LAUNCH_F32) } else { ST_DISPATCH(ST_LAUNCH_BF16) }
#undef ST_LAUNCH_F32
#undef ST_LAUNCH_BF16
    KA_LAUNCH_CHECK();
    return 0;
}
