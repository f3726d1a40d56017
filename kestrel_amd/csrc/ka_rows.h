// Finishing a row of the fp32 residual stream: a sublayer's output d is normalised and added, x += d / rms(d) * gain with
// rms(d) = sqrt(mean(d^2) + eps), and the norm that the next reader of the stream begins with is computed from the new
// row, h = x / rms(x) * gain2, in the same pass (without gain2 the new row itself is left there, rounded). A workgroup takes a row, of
// KA_ROW_THREADS threads where there are many rows, of a thread per four channels, up to 1,024, where there are few; what
// computes d is the caller's business (a load, a weighted sum). All arithmetic is fp32. Eight rows of 2,048 behind four experts: 4.5 us, where
// the sum, its norm into the stream and the rounding for the next reader were three launches of 13.4, 6.2 and 4.5.
#pragma once

#include "ka_common.h"

constexpr int KA_ROW_THREADS = 256;
constexpr int KA_ROW_MAX_PIECES = 8;        // pieces of four channels a thread keeps in registers: rows of up to 8192 channels

struct KaRowNorms {
    const float* gain;      // of the norm of d
    float eps;
    const float* gain2;     // of the norm of the new row; null: the row as it is
    float eps2;
    void* h;                // where that goes, rows of dim numbers; null: nowhere
    int h_bf16;
};

// However many threads a row has, its sums have the order of KA_ROW_THREADS of them, so that a row's bits do not depend on how many
// rows a step has: "thread" t of that order owns the pieces (four channels each) t, t + KA_ROW_THREADS and so on. Where a row has
// GROUP times as many threads, GROUP lanes of a wave share one of those: they hand each other their numbers before the wave's sum,
// and GROUP waves make one of that order's. It costs nothing that shows: eight rows of four streams of 4,096 channels 3.9 us, as with
// an order for each number of threads.
template <int THREADS>
struct KaRowLanes {
    static constexpr int GROUP = THREADS / KA_ROW_THREADS, WIDTH = KA_WAVE / GROUP, WAVES = THREADS / KA_WAVE;
    static_assert(GROUP == 1 || GROUP == 2 || GROUP == 4, "256, 512 or 1,024 threads");
};

// First channel of this thread's piece j.
template <int THREADS>
__device__ __forceinline__ int ka_row_channel(int j) {
    using L = KaRowLanes<THREADS>;
    const int wave = threadIdx.x / KA_WAVE, lane = threadIdx.x % KA_WAVE;
    return ((j * L::GROUP + lane / L::WIDTH) * KA_ROW_THREADS + wave * L::WIDTH + lane % L::WIDTH) * 4;
}

// Sum over the row of `q`, a number for each of this thread's pieces; the same bits in every thread. `smem` holds a float a wave.
template <int PIECES, int THREADS>
__device__ __forceinline__ float ka_pieces_sum(const float (&q)[PIECES], float* smem) {
    using L = KaRowLanes<THREADS>;
    float v = 0.f;
#pragma unroll
    for (int j = 0; j < PIECES; ++j) {
        if constexpr (L::GROUP == 1) {
            v += q[j];
        } else if constexpr (L::GROUP == 2) {
            float a, b;
            ka_lanes_pair<32>(q[j], a, b);
            v += a;
            v += b;
        } else {
            float a, b, c[4];
            ka_lanes_pair<16>(q[j], a, b);
            ka_lanes_pair<32>(a, c[0], c[2]);
            ka_lanes_pair<32>(b, c[1], c[3]);
#pragma unroll
            for (int p = 0; p < 4; ++p) v += c[p];
        }
    }
    v = ka_lanes_reduce<1, L::WIDTH>(v, KaSum{});
    __syncthreads();
    if (threadIdx.x % KA_WAVE == 0) smem[threadIdx.x / KA_WAVE] = v;
    __syncthreads();
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < L::WAVES; w += L::GROUP) {
        if constexpr (L::GROUP == 1) total += smem[w];
        else if constexpr (L::GROUP == 2) total += smem[w] + smem[w + 1];
        else total += (smem[w] + smem[w + 1]) + (smem[w + 2] + smem[w + 3]);
    }
    return total;
}

// The same of one number a thread, KA_ROW_THREADS threads.
__device__ __forceinline__ float ka_row_sum(float v, float* smem) {
    const float q[1] = {v};
    return ka_pieces_sum<1, KA_ROW_THREADS>(q, smem);
}

// Of four squares: the order is written out, so that every kernel has the same.
__device__ __forceinline__ float ka_squares(const float4& d) { return fmaf(d.w, d.w, fmaf(d.z, d.z, fmaf(d.x, d.x, d.y * d.y))); }

__device__ __forceinline__ void ka_row_store_h(const KaRowNorms& a, size_t at, float v) {
    if (a.h_bf16) reinterpret_cast<bf16_t*>(a.h)[at] = (bf16_t)v;
    else reinterpret_cast<float*>(a.h)[at] = v;
}

// PIECES > 0: dim is a multiple of 4 and at most 4 PIECES THREADS, rows are 16-byte aligned; `piece(c)` gives d of the
// channels c .. c + 3. PIECES = 0: any dim; `one(c)` gives d of channel c (asked for twice).
// Either may read the row of x that is finished: of the thread's own channels, before these are written.
template <int PIECES, int THREADS, typename Piece, typename One>
__device__ __forceinline__ void ka_finish_row(float* x, int row, int dim, const KaRowNorms& a, Piece piece, One one,
                                              float* smem) {
    const int tid = threadIdx.x;
    const size_t at = (size_t)row * dim;
    if constexpr (PIECES > 0) {
        typedef __attribute__((ext_vector_type(4))) __bf16 row_bf16x4;
        float4 d[PIECES], y[PIECES];
        float s[PIECES], s2[PIECES];
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            const int c = ka_row_channel<THREADS>(p);
            s[p] = 0.f;
            if (c < dim) {
                d[p] = piece(c);
                y[p] = *reinterpret_cast<const float4*>(x + at + c);
                s[p] = ka_squares(d[p]);
            }
        }
        const float r = 1.0f / sqrtf(ka_pieces_sum<PIECES, THREADS>(s, smem) / (float)dim + a.eps);
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            const int c = ka_row_channel<THREADS>(p);
            s2[p] = 0.f;
            if (c < dim) {
                const float4 g = *reinterpret_cast<const float4*>(a.gain + c);
                y[p].x += d[p].x * r * g.x;
                y[p].y += d[p].y * r * g.y;
                y[p].z += d[p].z * r * g.z;
                y[p].w += d[p].w * r * g.w;
                *reinterpret_cast<float4*>(x + at + c) = y[p];
                s2[p] = ka_squares(y[p]);
            }
        }
        if (a.h == nullptr) return;
        const float r2 = a.gain2 ? 1.0f / sqrtf(ka_pieces_sum<PIECES, THREADS>(s2, smem) / (float)dim + a.eps2) : 1.f;
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            const int c = ka_row_channel<THREADS>(p);
            if (c < dim) {
                float4 v = y[p];
                if (a.gain2) {
                    const float4 g = *reinterpret_cast<const float4*>(a.gain2 + c);
                    v = make_float4(v.x * r2 * g.x, v.y * r2 * g.y, v.z * r2 * g.z, v.w * r2 * g.w);
                }
                if (a.h_bf16) {
                    row_bf16x4 b;
                    b[0] = (bf16_t)v.x;
                    b[1] = (bf16_t)v.y;
                    b[2] = (bf16_t)v.z;
                    b[3] = (bf16_t)v.w;
                    *reinterpret_cast<row_bf16x4*>(reinterpret_cast<bf16_t*>(a.h) + at + c) = b;
                } else {
                    *reinterpret_cast<float4*>(reinterpret_cast<float*>(a.h) + at + c) = v;
                }
            }
        }
    } else {
        static_assert(THREADS == KA_ROW_THREADS, "the general form has one number of threads");
        float s = 0.f;
        for (int c = tid; c < dim; c += THREADS) {
            const float d = one(c);
            s += d * d;
        }
        const float r = 1.0f / sqrtf(ka_row_sum(s, smem) / (float)dim + a.eps);
        float s2 = 0.f;
        for (int c = tid; c < dim; c += THREADS) {
            const float y = x[at + c] + one(c) * r * a.gain[c];
            x[at + c] = y;
            s2 += y * y;
        }
        if (a.h == nullptr) return;
        const float r2 = a.gain2 ? 1.0f / sqrtf(ka_row_sum(s2, smem) / (float)dim + a.eps2) : 1.f;
        for (int c = tid; c < dim; c += THREADS) ka_row_store_h(a, at + c, x[at + c] * r2 * (a.gain2 ? a.gain2[c] : 1.f));      // (its own writes)
    }
}

// Pieces of four channels a thread holds of rows of `dim` channels in the form with registers, times ten, with 1 or 2 added where a
// row gets 512 or 1,024 threads (fewer rows than two a CU); 0: the general form.
static inline int ka_row_pieces(int n, int dim, const void* x, const void* d, const KaRowNorms& a) {
    const uintptr_t all = (uintptr_t)x | (uintptr_t)d | (uintptr_t)a.gain | (uintptr_t)a.gain2;
    if (dim % 4 != 0 || all % 16 != 0 || (uintptr_t)a.h % (a.h_bf16 ? 8 : 16) != 0) return 0;
    const int need = (dim + 4 * KA_ROW_THREADS - 1) / (4 * KA_ROW_THREADS);
    if (n < 2 * ka_compute_units()) {
        if (need == 2) return 11;
        if (need > 2 && need <= 4) return 12;
        if (need > 4 && need <= 8) return 22;
    }
    for (int p : {1, 2, 4, 8})
        if (need <= p) return p * 10;
    return 0;
}

// LAUNCH(pieces, threads) of the form that ka_row_pieces named.
#define KA_ROW_CASES(PIECES, LAUNCH)   \
    switch (PIECES) {                  \
        case 10: LAUNCH(1, 256); break; \
        case 20: LAUNCH(2, 256); break; \
        case 40: LAUNCH(4, 256); break; \
        case 80: LAUNCH(8, 256); break; \
        case 11: LAUNCH(1, 512); break; \
        case 12: LAUNCH(1, 1024); break;\
        case 22: LAUNCH(2, 1024); break;\
        default: LAUNCH(0, 256); break; \
    }
