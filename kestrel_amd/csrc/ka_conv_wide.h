// The short causal convolution with rotation and cache write (sequence_parts.hip) for bf16 rows as a function of a workgroup's place, so that
// more than one kernel can hold it: the plain launch and the launch that runs it beside the step of a recurrence (both in sequence_parts.hip).
#pragma once
#include "ka_common.h"

constexpr int SP_THREADS = 256;

struct ConvArgs {
    const void* u;
    long u_stride;
    const float* taps;
    float* state;
    long state_stride;      // from one slot's rows to the next slot's
    int K, C;
    const int* cu_q;
    const int* row_slot;
    const int* token_row;
    const int* positions;
    const int* slots;
    void* q_out;
    long q_stride;
    void* k_cache;
    void* v_cache;
    int Hq, Hk, hd, Hv, hdv, page_size;
    const float* freqs;
    int rot, interleaved;
    int normed;
    float eps;
    // the form of eight channels a thread: the tokens cut into runs of at most page_size (null: every token by itself), and
    // whether every row brings one token, row t token t (its thread then moves the state on as well)
    const int* run_first;
    const int* run_count;
    int single_tokens;
};

// The short convolution, rotation and cache write of sequence_parts.hip for bf16 rows, up to SP_WIDE_TAPS taps, and query and key heads of 8 LPH channels, LPH a power of two: a thread
// keeps eight neighbouring channels, their taps and the rows the taps still reach in registers and walks over the tokens of a
// run, one 16-byte load a token; a head's sum of squares meets inside its LPH lanes, and the lanes of a rotated pair of
// halves exchange their numbers. Grid (blocks of 2,048 channels: queries and keys, then values; runs; parts of a run). Eight values
// of a channel that lie side by side in a page leave together. rot is a multiple of 16 for pairs of halves.
typedef __attribute__((ext_vector_type(8))) __bf16 sp_bf16x8;
typedef __attribute__((ext_vector_type(4))) float sp_floatx4;
constexpr int SP_WIDE_TAPS = 4;
constexpr int SP_WIDE_RUN = 16;                     // tokens of a run at most
constexpr int SP_WIDE_QK = 4, SP_WIDE_V = 8;        // tokens of a run a workgroup takes, of queries and keys and of values
constexpr int SP_WIDE_MAX_ROT = 256;

// Whatever `back` = 1 .. SP_WIDE_TAPS - 1 rows before token t hold of channels c .. c + 7, into hist[back - 1].
__device__ __forceinline__ void sp_wide_history(const ConvArgs& a, int t, int local, int slot, int c, float (&hist)[SP_WIDE_TAPS - 1][8]) {
    const bf16_t* u = reinterpret_cast<const bf16_t*>(a.u);
#pragma unroll
    for (int back = 1; back < SP_WIDE_TAPS; ++back) {
        if (back < a.K && back <= local) {
            const sp_bf16x8 x = *reinterpret_cast<const sp_bf16x8*>(u + (size_t)(t - back) * a.u_stride + c);
#pragma unroll
            for (int e = 0; e < 8; ++e) hist[back - 1][e] = (float)x[e];
        } else if (back < a.K && slot >= 0) {
            const float* st = a.state + (size_t)slot * a.state_stride + (size_t)(local - back + a.K - 1) * a.C + c;
            const sp_floatx4 x0 = *reinterpret_cast<const sp_floatx4*>(st), x1 = *reinterpret_cast<const sp_floatx4*>(st + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) { hist[back - 1][e] = x0[e]; hist[back - 1][4 + e] = x1[e]; }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) hist[back - 1][e] = 0.f;
        }
    }
}

// The taps of channels c .. c + 7 as w[back]: the tap that reads `back` rows before (0: behind the last). K numbers a channel, side
// by side.
template <int K>
__device__ __forceinline__ void sp_wide_taps(const float* taps, int c, float (&w)[SP_WIDE_TAPS][8]) {
    float flat[8 * K];
    const float* src = taps + (size_t)c * K;
#pragma unroll
    for (int i = 0; i < 2 * K; ++i) {
        const sp_floatx4 v = *reinterpret_cast<const sp_floatx4*>(src + 4 * i);
#pragma unroll
        for (int e = 0; e < 4; ++e) flat[4 * i + e] = v[e];
    }
#pragma unroll
    for (int back = 0; back < SP_WIDE_TAPS; ++back)
#pragma unroll
        for (int e = 0; e < 8; ++e) w[back][e] = back < K ? flat[e * K + (back < K ? K - 1 - back : 0)] : 0.f;
}

// ONE: every run is one token (a step of single tokens), which takes 70 registers less.
template <int LPH, bool ONE>
__device__ __forceinline__ void conv_prepare_wide_body(const ConvArgs& a, const int bx, const int by, const int bz) {
    __shared__ __attribute__((aligned(16))) float cs[ONE ? 1 : SP_WIDE_QK][SP_WIDE_MAX_ROT / 2], sn[ONE ? 1 : SP_WIDE_QK][SP_WIDE_MAX_ROT / 2];
    __shared__ int row_s[SP_WIDE_V], at_s[SP_WIDE_V];
    constexpr int HD = 8 * LPH, QK = ONE ? 1 : SP_WIDE_QK, VALUES = ONE ? 1 : SP_WIDE_V;      // tokens of a workgroup
    const int tid = threadIdx.x;
    const int Cqk = (a.Hq + a.Hk) * HD, Cv = a.Hv * a.hdv;
    const int qk_blocks = (Cqk + 8 * SP_THREADS - 1) / (8 * SP_THREADS);
    const bool values = bx >= qk_blocks;
    // this workgroup's tokens of the run
    const int part = values ? VALUES : QK;
    const int first = (a.run_first ? a.run_first[by] : by) + bz * part;
    const int count = min((a.run_first ? min(a.run_count[by], SP_WIDE_RUN) : 1) - bz * part, part);
    if (count <= 0) return;
    // (threads behind the last channel do the work of the first ones and store nothing: all lanes of a wave stay together)
    const int mine = (bx - (values ? qk_blocks : 0)) * SP_THREADS + tid;
    const bool live = 8 * mine < (values ? Cv : Cqk);
    const int within = live ? 8 * mine : 8 * (tid % LPH);
    const int c = values ? Cqk + (live ? 8 * mine : 0) : within;
    const bf16_t* u = reinterpret_cast<const bf16_t*>(a.u) + c;
    sp_bf16x8 rows[VALUES];
#pragma unroll
    for (int i = 0; i < VALUES; ++i)
        if (i < count) rows[i] = *reinterpret_cast<const sp_bf16x8*>(u + (size_t)(first + i) * a.u_stride);
    float w[SP_WIDE_TAPS][8];
    switch (a.K) {
        case 1: sp_wide_taps<1>(a.taps, c, w); break;
        case 2: sp_wide_taps<2>(a.taps, c, w); break;
        case 3: sp_wide_taps<3>(a.taps, c, w); break;
        default: sp_wide_taps<4>(a.taps, c, w); break;
    }
    float hist[SP_WIDE_TAPS - 1][8];
    int row, slot;
    if (a.single_tokens) {                          // (row t brings token t, its first)
        row = first;
        slot = a.row_slot[row];
        sp_wide_history(a, first, 0, slot, c, hist);
    } else {
        row = a.token_row[first];
        slot = a.row_slot[row];
        sp_wide_history(a, first, first - a.cu_q[row], slot, c, hist);
    }
    const int half = a.rot / 2;
    if (tid < count) {
        row_s[tid] = a.single_tokens ? row : a.token_row[first + tid];
        at_s[tid] = a.slots ? a.slots[first + tid] : -1;
    }
    if (a.freqs && !values)
        for (int e = tid; e < count * half; e += SP_THREADS)
            sincosf((float)a.positions[first + e / half] * a.freqs[e % half], &sn[e / half][e % half], &cs[e / half][e % half]);
    __syncthreads();
    // the rows before token i of the run, where it is not the one behind the last token of its row
    auto enter = [&](int i) {
        const int r = row_s[i];
        if (r == row) return;
        row = r;
        slot = a.row_slot[r];
        sp_wide_history(a, first + i, first + i - a.cu_q[r], slot, c, hist);
    };
    auto convolve = [&](const sp_bf16x8& x, float (&y)[8]) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float s = 0.f;
#pragma unroll
            for (int back = SP_WIDE_TAPS - 1; back >= 1; --back) s = fmaf(w[back][e], hist[back - 1][e], s);
            y[e] = fmaf(w[0][e], (float)x[e], s);
        }
#pragma unroll
        for (int back = SP_WIDE_TAPS - 2; back >= 1; --back)
#pragma unroll
            for (int e = 0; e < 8; ++e) hist[back][e] = hist[back - 1][e];
#pragma unroll
        for (int e = 0; e < 8; ++e) hist[0][e] = (float)x[e];
    };
    // (the row's only token: entry s of the state is now what stands K - 2 - s rows before the next token's predecessor)
    auto move_state = [&]() {
        if (!a.single_tokens || slot < 0 || !live) return;
        float* st = a.state + (size_t)slot * a.state_stride + c;
#pragma unroll
        for (int back = 0; back < SP_WIDE_TAPS - 1; ++back) {
            if (back >= a.K - 1) continue;
            sp_floatx4 v0, v1;
#pragma unroll
            for (int e = 0; e < 4; ++e) { v0[e] = hist[back][e]; v1[e] = hist[back][4 + e]; }
            *reinterpret_cast<sp_floatx4*>(st + (size_t)(a.K - 2 - back) * a.C) = v0;
            *reinterpret_cast<sp_floatx4*>(st + (size_t)(a.K - 2 - back) * a.C + 4) = v1;
        }
    };
    if (!values) {
        const int head = within / HD, sub = within % HD / 8;
        const bool is_q = head < a.Hq;
        // (what a channel's rotation does is the same for every token)
        const int apart = a.rot / 16;
        const bool low = sub < apart, turned = a.freqs && !a.interleaved && sub < 2 * apart;
        const int partner = (turned ? (tid % KA_WAVE) + (low ? apart : -apart) : tid % KA_WAVE);
        const int j0 = (low ? sub : sub - apart) * 8;
#pragma unroll
        for (int i = 0; i < QK; ++i) {
            if (i >= count) break;
            float y[8];
            enter(i);
            convolve(rows[i], y);
            if (a.normed) {
                float ss = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) ss = fmaf(y[e], y[e], ss);
                const float scale = 1.0f / sqrtf(ka_lanes_reduce<1, LPH>(ss, KaSum{}) / (float)HD + a.eps);
#pragma unroll
                for (int e = 0; e < 8; ++e) y[e] *= scale;
            }
            if (a.freqs && a.interleaved) {
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    const int j = sub * 4 + p;
                    if (2 * j < a.rot) {
                        const float v0 = y[2 * p], v1 = y[2 * p + 1];
                        y[2 * p] = v0 * cs[i][j] - v1 * sn[i][j];
                        y[2 * p + 1] = v1 * cs[i][j] + v0 * sn[i][j];
                    }
                }
            } else if (a.freqs) {
                float other[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) other[e] = __shfl(y[e], partner);
                if (turned) {
                    const sp_floatx4 c0 = *reinterpret_cast<const sp_floatx4*>(&cs[i][j0]), c1 = *reinterpret_cast<const sp_floatx4*>(&cs[i][j0 + 4]);
                    const sp_floatx4 s0 = *reinterpret_cast<const sp_floatx4*>(&sn[i][j0]), s1 = *reinterpret_cast<const sp_floatx4*>(&sn[i][j0 + 4]);
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float co = e < 4 ? c0[e % 4] : c1[e % 4], si = e < 4 ? s0[e % 4] : s1[e % 4];
                        y[e] = low ? y[e] * co - other[e] * si : y[e] * co + other[e] * si;
                    }
                }
            }
            sp_bf16x8 o;
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = (bf16_t)y[e];
            if (!live) continue;
            if (is_q) {
                *reinterpret_cast<sp_bf16x8*>(reinterpret_cast<bf16_t*>(a.q_out) + (size_t)(first + i) * a.q_stride + within) = o;
            } else {
                const int at = at_s[i];
                if (at >= 0)
                    *reinterpret_cast<sp_bf16x8*>(reinterpret_cast<bf16_t*>(a.k_cache) + (((size_t)(at / a.page_size) * a.Hk + (head - a.Hq)) * a.page_size +
                                                  at % a.page_size) * HD + sub * 8) = o;
            }
        }
        move_state();
        return;
    }
    if (!live) return;                              // (nothing below meets other lanes)
    const int vc = 8 * mine, vhead = vc / a.hdv, vd = vc % a.hdv;
    bf16_t* vbase = reinterpret_cast<bf16_t*>(a.v_cache);
    const int at0 = at_s[0];
    if constexpr (!ONE) if (count == SP_WIDE_V && a.page_size % SP_WIDE_V == 0 && at0 >= 0 && at0 % SP_WIDE_V == 0 && at_s[SP_WIDE_V - 1] == at0 + SP_WIDE_V - 1 &&
        row_s[SP_WIDE_V - 1] == row_s[0]) {
        sp_bf16x8 page[8];                          // (places side by side in a page: 16 bytes a channel)
#pragma unroll
        for (int i = 0; i < SP_WIDE_V; ++i) {
            float y[8];
            convolve(rows[i], y);
#pragma unroll
            for (int e = 0; e < 8; ++e) page[e][i] = (bf16_t)y[e];
        }
        bf16_t* dst = vbase + (((size_t)(at0 / a.page_size) * a.Hv + vhead) * a.hdv + vd) * a.page_size + at0 % a.page_size;
#pragma unroll
        for (int e = 0; e < 8; ++e) *reinterpret_cast<sp_bf16x8*>(dst + (size_t)e * a.page_size) = page[e];
        return;
    }
#pragma unroll
    for (int i = 0; i < VALUES; ++i) {
        if (i >= count) break;
        float y[8];
        enter(i);
        convolve(rows[i], y);
        const int at = at_s[i];
        if (at < 0) continue;
        bf16_t* dst = vbase + (((size_t)(at / a.page_size) * a.Hv + vhead) * a.hdv + vd) * a.page_size + at % a.page_size;
#pragma unroll
        for (int e = 0; e < 8; ++e) dst[(size_t)e * a.page_size] = (bf16_t)y[e];
    }
    move_state();
}
