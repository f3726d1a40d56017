// A router's choice by one wave a token, as a function, so that it can be a launch of its own (experts.hip) or go along in the launch of a linear
// (gemv_bf16.hip).
#pragma once
#include "ka_common.h"

constexpr int EX_MAX_OUTPUTS = 512;             // router outputs a wave can hold (8 a lane)
constexpr int EX_MAX_GROUPS = 64;

// The lowest index that holds the largest value of a wave (of at most `last`), in every lane.
__device__ __forceinline__ int ex_wave_argmax(float v, int i, int last) {
    const float best = ka_wave_max(v);
    const int found = ka_lanes_reduce<1, KA_WAVE>(v == best ? i : 0x7fffffff, KaIntMin{});
    return __builtin_amdgcn_readfirstlane(min(found, last));
}

// The router's choice, a wave per token. logits fp32 [n, >= R] (rows `stride` apart), R router outputs.
//     s = softmax(logits), or sigmoid(logits) one by one;  choice = s + correction (correction optional)
//     n_groups > 0: the outputs form n_groups equal groups of neighbours, a group's score is its largest choice score, or the
//       sum of its two largest (group_best 2), and only outputs of the `keep` best groups can be chosen;
//     the `top` outputs with the largest choice scores are chosen (the lower index wins a tie);
//     weights: their s divided by the sum of the chosen s (+ 1e-20), times scale.
// mode 0: softmax scores, 2: sigmoid scores; 1 (by the logits): the choice goes by the logits themselves (no correction, no groups); the weights are the softmax over the chosen
// logits, times scale.
// chosen int32 [n, top], weights fp32 [n, top]; always >= 0: the rows are one longer and end in that output with weight 1 (a
// feed-forward that every token uses, laid behind the experts).
struct RouteArgs {
    const float* logits;
    long stride;
    const float* correction;
    int R, top, n_groups, keep, group_best, mode, always;
    float scale;
    int* chosen;
    float* weights;
};

template <int PER_LANE>          // outputs a lane holds
struct RouteRoom {               // LDS of a wave
    float choice[PER_LANE * KA_WAVE], group[EX_MAX_GROUPS];
    int allowed[EX_MAX_GROUPS];
};

// What the wave's lanes wrote to LDS before is seen by its lanes after.
__device__ __forceinline__ void ka_route_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Token t by this wave, all lanes active.
template <int PER_LANE>
__device__ __forceinline__ void ka_route_token(const RouteArgs& job, int t, int lane, RouteRoom<PER_LANE>& room) {
    const int R = job.R, top = job.top, n_groups = job.n_groups, keep = job.keep, group_best = job.group_best, always = job.always;
    const float* const correction = job.correction;
    const bool by_logits = job.mode == 1, sigmoids = job.mode == 2;
    const float* z = job.logits + (size_t)t * job.stride;
    float s[PER_LANE], c[PER_LANE];
    float top_z = -INFINITY;
#pragma unroll
    for (int q = 0; q < PER_LANE; ++q) {
        const int r = lane + q * KA_WAVE;
        s[q] = r < R ? z[r] : -INFINITY;
        top_z = fmaxf(top_z, s[q]);
    }
    top_z = ka_wave_max(top_z);
    float total = 0.f;
#pragma unroll
    for (int q = 0; q < PER_LANE; ++q) {
        c[q] = s[q];
        if (sigmoids) s[q] = lane + q * KA_WAVE < R ? 1.0f / (1.0f + expf(-s[q])) : 0.f;
        else s[q] = lane + q * KA_WAVE < R ? expf(s[q] - top_z) : 0.f;
        total += s[q];
    }
    total = ka_wave_sum(total);
#pragma unroll
    for (int q = 0; q < PER_LANE; ++q) {
        const int r = lane + q * KA_WAVE;
        if (by_logits) continue;      // (the largest logit is among the chosen: e^(z - top) over their sum is their softmax)
        if (!sigmoids) s[q] = s[q] / total;
        c[q] = r < R ? s[q] + (correction ? correction[r] : 0.f) : -INFINITY;
        if (r < R) room.choice[r] = c[q];
    }
    if (n_groups > 0) {
        const int per = R / n_groups;
        ka_route_sync();
        if (lane < n_groups) {
            float best = -INFINITY, second = -INFINITY;
            for (int m = 0; m < per; ++m) {
                const float v = room.choice[lane * per + m];
                second = fmaxf(second, fminf(v, best));
                best = fmaxf(best, v);
            }
            room.group[lane] = group_best == 2 && per > 1 ? best + second : best;
        }
        ka_route_sync();
        if (lane < n_groups) {
            const float own = room.group[lane];
            int ahead = 0;              // groups that are kept before this one (the lower index wins a tie)
            for (int g = 0; g < n_groups; ++g) ahead += room.group[g] > own || (room.group[g] == own && g < lane);
            room.allowed[lane] = ahead < keep;
        }
        ka_route_sync();
#pragma unroll
        for (int q = 0; q < PER_LANE; ++q) {
            const int r = lane + q * KA_WAVE;
            if (r < R && !room.allowed[r / per]) c[q] = -INFINITY;
        }
    }
    float sum = 0.f;
    float mine_w = 0.f;          // lane k keeps the k-th chosen score
    int mine_i = 0;
    unsigned taken = 0;          // bit q: this lane's entry q is chosen already
    for (int k = 0; k < top; ++k) {
        float v = -INFINITY;
        int i = 0x7fffffff;
#pragma unroll
        for (int q = 0; q < PER_LANE; ++q) {
            const int r = lane + q * KA_WAVE;
            if (r < R && !(taken >> q & 1) && (c[q] > v || i == 0x7fffffff)) {
                v = c[q];
                i = r;
            }
        }
        i = ex_wave_argmax(v, i, R - 1);
        float sv = 0.f;
#pragma unroll
        for (int q = 0; q < PER_LANE; ++q)
            if (lane + q * KA_WAVE == i) {
                taken |= 1u << q;
                sv = s[q];
            }
        sv = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(sv), i % KA_WAVE));       // (one lane holds it)
        sum += sv;
        if (lane == k % KA_WAVE) {
            // (more than a wave of choices would need more than one register a lane: the entry point refuses it)
            mine_w = sv;
            mine_i = i;
        }
    }
    const size_t at = (size_t)t * (always >= 0 ? top + 1 : top);
    if (lane < top) {
        job.chosen[at + lane] = mine_i;
        job.weights[at + lane] = mine_w / (by_logits ? sum : sum + 1e-20f) * job.scale;
    }
    if (always >= 0 && lane == 0) {
        job.chosen[at + top] = always;
        job.weights[at + top] = 1.f;
    }
}

static inline int ka_route_check(const char* who, const RouteArgs& r, int n) {
    KA_CHECK(r.mode >= 0 && r.mode <= 2 && (r.group_best == 1 || r.group_best == 2), "%s: unknown mode %d or group score %d", who, r.mode, r.group_best);
    KA_CHECK(r.mode != 1 || (r.n_groups == 0 && r.correction == nullptr), "%s: a choice by the logits alone has no groups and no correction", who);
    KA_CHECK(n >= 0 && r.R > 0 && r.R <= EX_MAX_OUTPUTS && r.stride >= r.R, "%s: %d router outputs (at most %d)", who, r.R, EX_MAX_OUTPUTS);
    KA_CHECK(r.top > 0 && r.top <= r.R && r.top <= KA_WAVE, "%s: %d choices of %d", who, r.top, r.R);
    KA_CHECK(r.n_groups >= 0 && r.n_groups <= EX_MAX_GROUPS && (r.n_groups == 0 || (r.R % r.n_groups == 0 && r.keep > 0 && r.keep <= r.n_groups)),
             "%s: %d groups of which %d are kept do not divide %d outputs", who, r.n_groups, r.keep, r.R);
    KA_CHECK(r.n_groups == 0 || r.keep * (r.R / r.n_groups) >= r.top, "%s: %d kept groups hold fewer than %d outputs", who, r.keep, r.top);
    return 0;
}
