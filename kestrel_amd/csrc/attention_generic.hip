// Generic paged attention, all arithmetic in fp32: one wavefront per (token, query head), any head size up
// to 1024, any page size, fp32 or bf16 storage; and a second kernel for fp32 storage in steps of four keys and channels, which reads whole lines.
//
// Every token t of the packed batch belongs to request row token_row[t] and sees
// the cached keys at positions [kv_lo[t], kv_hi[t]) of that row (kv_lo optional,
// default 0). A causal token at position p has kv_hi = p + 1; a token inside a
// bidirectional block has kv_hi = end of its block; a window of w has
// kv_lo = max(0, p + 1 - w). The keys of this step are already in the cache.
// Key position k of row r lies at page block_table[r, k / page_size], offset
// k % page_size; key cache [pages, Hkv, page_size, hd], value cache [pages, Hkv, hdv, page_size]:
// values may have another size than queries and keys (hdv channels; the output is [n, H hdv]).
//
// Two optional terms of the scores, for mixers that encode order by distance instead of by a
// rotation, and that let a query attend to nothing:
//  * slopes (fp32 [H]) with positions (int32 [n], the place of every query in its row): the score
//    of query position i against key position j is lowered by slopes[h] * (i - j);
//  * a distance table (fp32 [H, bias_len]) with positions: the score of query position i against key position j is
//    raised by table[h, min(i - j, bias_len - 1)] (a learned bias per head and distance, constant from some distance on);
//  * an output gate (rows of the activation type, [n, H hdv] with a row stride of their own): the output is multiplied
//    element by element by the sigmoid of it;
//  * a sink: one more term exp(sink_score) in the softmax's denominator that carries no value
//    (has_sink != 0). The running maximum and sum then start from that term instead of from nothing.
//    `sinks` (fp32 [H]) gives every head a score of its own for that term;
//  * kept first keys: a query also sees the keys [0, min(keep_first, kv_lo)) of its row, before its window;
//  * several maps per head (maps > 1): query heads and key heads come in groups of `maps` neighbours, map m of a
//    query head reads map m of its key head, and all maps of a key head share one value head: H and Hkv count maps,
//    the value cache has Hkv / maps heads;
//  * values inside the keys (values_in_keys != 0): the value of a key is the first hdv channels of its key row
//    (a cache of latents that are both); v_cache is then not read;
//  * out_f32 != 0: the output is written as fp32 whatever the type of queries and cache;
//  * softcap > 0: the scaled score passes through softcap * tanh(score / softcap) before any bias and the softmax;
//  * gate_per_head != 0: the gate holds one number per head ([n, H]) instead of one per channel.
#include "ka_common.h"

constexpr int ATT_MAX_HD = 1024;

// Four neighbouring elements with one load (the address must be a multiple of 4 elements).
template <typename T>
__device__ __forceinline__ void att_load4(const T* p, float v[4]) {
    typedef __attribute__((ext_vector_type(4))) T vec4;
    const vec4 x = *reinterpret_cast<const vec4*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = ka_to_float(x[i]);
}

template <typename T>
__global__ void __launch_bounds__(KA_WAVE)
attention_generic_kernel(const T* __restrict__ q, long q_row_stride, const T* __restrict__ k_cache,
                         const T* __restrict__ v_cache, const int* __restrict__ block_table,
                         int max_pages, const int* __restrict__ token_row,
                         const int* __restrict__ kv_lo, const int* __restrict__ kv_hi,
                         T* __restrict__ out, long out_row_stride, float scale, int H, int Hkv,
                         int hd, int hdv, int page_size, const int* __restrict__ positions,
                         const float* __restrict__ slopes, int has_sink, float sink_score,
                         const float* __restrict__ bias_table, int bias_len, const T* __restrict__ gate,
                         long gate_row_stride, const float* __restrict__ sinks, int keep_first, int maps,
                         int values_in_keys, int out_f32, float softcap, int gate_per_head) {
    __shared__ float qs[ATT_MAX_HD];
    __shared__ float ps[KA_WAVE];
    __shared__ long offs[KA_WAVE];   // value cache offset of channel 0 of each key of the chunk
    int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
    // (maps == 1: query head h reads kv head h / (H / Hkv), keys and values alike)
    const int vh = h / maps / (H / Hkv);
    const int kvh = vh * maps + h % maps;
    const int Hv = Hkv / maps;
    int row = token_row[t];
    int lo = kv_lo ? kv_lo[t] : 0, hi = kv_hi[t];
    const T* qp = q + (size_t)t * q_row_stride + (size_t)h * hd;
    for (int d = lane; d < hd; d += KA_WAVE) qs[d] = ka_to_float(qp[d]) * scale;
    const float slope = slopes ? slopes[h] : 0.f;
    const int place = (slopes || bias_table) ? positions[t] : 0;
    const float* bias_row = bias_table ? bias_table + (size_t)h * bias_len : nullptr;
    __syncthreads();
    const int* bt = block_table + (size_t)row * max_pages;
    const bool k_vectors = hd % 4 == 0 && reinterpret_cast<uintptr_t>(k_cache) % (4 * sizeof(T)) == 0;
    const bool v_vectors = page_size % 4 == 0 && reinterpret_cast<uintptr_t>(v_cache) % (4 * sizeof(T)) == 0;
    if (sinks) sink_score = sinks[h];
    float m = has_sink ? sink_score : -INFINITY, l = has_sink ? 1.f : 0.f;
    float o[ATT_MAX_HD / KA_WAVE];
#pragma unroll
    for (int i = 0; i < ATT_MAX_HD / KA_WAVE; ++i) o[i] = 0.f;
    const int kept = min(keep_first, lo);            // keys [0, kept) before the window, then [lo, hi)
    for (int part = kept > 0 ? 0 : 1; part < 2; ++part)
    for (int base = part ? lo : 0, hi_here = part ? hi : kept; base < hi_here; base += KA_WAVE) {
        const int hi = hi_here;
        int key = base + lane;
        bool valid = key < hi;
        float s = -INFINITY;
        long off = 0;
        if (valid) {
            int page = bt[key / page_size];
            const T* kp = k_cache + (((long)page * Hkv + kvh) * page_size + key % page_size) * hd;
            off = values_in_keys ? (long)(kp - k_cache) : ((long)page * Hv + vh) * hdv * page_size + key % page_size;
            float acc = 0.f;
            if (k_vectors) {
                // four channels with one load, added in the same order as one by one
                for (int d = 0; d < hd; d += 4) {
                    float k4[4];
                    att_load4(kp + d, k4);
#pragma unroll
                    for (int u = 0; u < 4; ++u) acc = fmaf(qs[d + u], k4[u], acc);
                }
            } else {
                for (int d = 0; d < hd; ++d) acc = fmaf(qs[d], ka_to_float(kp[d]), acc);
            }
            if (softcap > 0.f) acc = softcap * tanhf(acc / softcap);
            s = slopes ? acc - slope * (float)(place - key) : acc;
            if (bias_row) s += bias_row[min(max(place - key, 0), bias_len - 1)];
        }
        float m_new = fmaxf(m, ka_wave_max(s));
        float corr = expf(m - m_new);  // m = -inf at the first chunk gives 0
        float p = valid ? expf(s - m_new) : 0.f;
        l = l * corr + ka_wave_sum(p);
        m = m_new;
        __syncthreads();
        ps[lane] = p;
        offs[lane] = off;
        __syncthreads();
        int count = min(KA_WAVE, hi - base);
#pragma unroll
        for (int i = 0; i < ATT_MAX_HD / KA_WAVE; ++i) {
            int d = lane + i * KA_WAVE;
            if (d < hdv) {
                float acc = o[i] * corr;
                const T* vd = values_in_keys ? k_cache + d : v_cache + (long)d * page_size;
                int j = 0;
                // A chunk that starts on a multiple of four keys: every four keys from there lie in
                // one page, their values side by side in the cache: one load, added in the same
                // order as one by one.
                if (v_vectors && !values_in_keys && (base & 3) == 0) {
                    for (; j + 3 < count; j += 4) {
                        float v4[4];
                        att_load4(vd + offs[j], v4);
#pragma unroll
                        for (int u = 0; u < 4; ++u) acc = fmaf(ps[j + u], v4[u], acc);
                    }
                }
                for (; j < count; ++j) acc = fmaf(ps[j], ka_to_float(vd[offs[j]]), acc);
                o[i] = acc;
            }
        }
    }
    float inv = l > 0.f ? 1.0f / l : 0.f;
    const size_t out_at = (size_t)t * out_row_stride + (size_t)h * hdv;
    const float head_gate = gate && gate_per_head ? 1.0f / (1.0f + expf(-ka_to_float(gate[(size_t)t * gate_row_stride + h]))) : 1.f;
#pragma unroll
    for (int i = 0; i < ATT_MAX_HD / KA_WAVE; ++i) {
        int d = lane + i * KA_WAVE;
        if (d < hdv) {
            float y = o[i] * inv * head_gate;
            // (an output gate: the head's channels times the sigmoid of the gate's pre-activations of the same token)
            if (gate && !gate_per_head) y *= 1.0f / (1.0f + expf(-ka_to_float(gate[(size_t)t * gate_row_stride + (size_t)h * hdv + d])));
            if (out_f32) reinterpret_cast<float*>(out)[out_at + d] = y;
            else out[out_at + d] = ka_from_float<T>(y);
        }
    }
}

// ----------------------------------------------------------------------------
// The same for fp32 heads of up to 256 channels (keys a multiple of four) and pages of a multiple of four keys, values in a cache of their own.
//
// Bound by trips to memory one behind the other. In the kernel above a lane owns a key, so a load touches 64 rows with 16 bytes each and comes
// back to each of them for every four channels, and the values are asked for when the scores are known; one wave walks all keys. Here
// G = 16, 32 or 64 lanes share a key (a row is one load's piece), 16 keys each; a lane's sixteen partial scores are added up across its row of 16
// lanes so that each lane ends with one key's (fifteen lane moves for 16 keys); values come as four neighbouring keys of one channel, whole
// pieces of a page, asked for together with the keys. A token's chunks of CK keys are dealt out to AS_PARTS parts, which meet in LDS at the end; a wave takes
// one part or all of them one behind the other, and the sums are the same: a token's numbers do not depend on the tokens beside it.
// 32 heads of 64, eight layers' caches in turn, us, there and here: 3 tokens behind 160 keys 17.3 and 6.6, 6 behind 400 46 and 13.7, 64 behind 400 106 and 74
// (5.7 TB/s); prompts of 17 5.6 and 5.2, six of 20 10.6 and 9.2, three of 64 32 and 13, one of 200 67 and 24, of 2,048 5,373 and 1,078; heads of 128: 6 behind
// 400 85 and 20, a prompt of 400 454 and 101. (All chunks in one sequence where a wave takes a token alone: 137 registers instead of 126 with heads of 64, a wave
// less a SIMD, six of 20 12.6, three of 64 15.6; heads of 128 up to 5 % faster, a prompt of 200 35.4 against 37.3. Places behind the last key left out of the
// loads: 172 registers, six of 20 10.2, three of 64 17.4.) Errors against 64 bits are no larger: a score is the sum of sixteen or more
// partial ones instead of one chain.
// ----------------------------------------------------------------------------
struct SpreadArgs {
    const float* q;
    long q_row_stride;
    const float *k_cache, *v_cache;
    const int* block_table;
    int max_pages;
    const int *token_row, *kv_lo, *kv_hi;
    float* out;
    long out_row_stride;
    float scale;
    int H, Hkv, hd, hdv, page_size;
    const int* positions;
    const float* slopes;
    int has_sink;
    float sink_score;
    const float* bias_table;
    int bias_len;
    const float* gate;
    long gate_row_stride;
    const float* sinks;
    int keep_first, maps;
    float softcap;
    int gate_per_head;
    // a step of single tokens whose keys and values are not cached yet: they lie behind the queries of `q`
    const int* slots;           // where they go (< 0: nowhere)
    const float* table;         // [places, rot]: cosines, then sines
    int rot, interleaved;
};

typedef __attribute__((ext_vector_type(4))) float as_floatx4;

// What a wave's lanes wrote to LDS before is seen by its lanes after.
__device__ __forceinline__ void as_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Sixteen values a lane, added up over the 16 lanes of a row: lane i of the row ends with the sum of value i. A step leaves a lane the half of the
// values that its own bit names and adds the partner's (the lane mirrored in the row, in the half row, then two and one further).
template <int LEFT>
__device__ __forceinline__ void as_scatter_sums(float (&v)[16], int lane) {
    if constexpr (LEFT >= 1) {
        constexpr int CTRL = LEFT == 8 ? 0x140 : LEFT == 4 ? 0x141 : LEFT == 2 ? 0x4E : 0xB1;
        const bool upper = lane & LEFT;
#pragma unroll
        for (int i = 0; i < LEFT; ++i) {
            const float keep = upper ? v[i + LEFT] : v[i], give = upper ? v[i] : v[i + LEFT];
            v[i] = keep + ka_dpp_move<CTRL>(give);
        }
        as_scatter_sums<LEFT / 2>(v, lane);
    }
}

constexpr int AS_PARTS = 4;

// Four channels of a head from `d` on, the first `rot` of them rotated (as rope_cache_kernel does).
__device__ __forceinline__ as_floatx4 as_rotated(const float* head, const float* cs, int rot, int interleaved, int d) {
    as_floatx4 y = *reinterpret_cast<const as_floatx4*>(head + d);
    const int half = rot / 2;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int c = d + e;
        if (c >= rot) continue;
        const int i = interleaved ? c / 2 : (c < half ? c : c - half), ia = interleaved ? 2 * i : i, ib = interleaved ? 2 * i + 1 : i + half;
        const float a = head[ia], b = head[ib], co = cs[i], si = cs[half + i];
        y[e] = c == ia ? a * co - b * si : b * co + a * si;
    }
    return y;
}

// NW waves take the parts in turn: the sums of a token are the same whatever NW is. STEP: the token's own key and value come from the projected row, rotated here, and the first
// head that reads them puts them into the cache; in a chunk of keys they take the place of what the cache holds there. (As a launch in front and this
// one, us, 32 heads of 64: three tokens behind 160 keys 9.6 and 8.0, six behind 400 17.1 and 14.8, six behind 2,000 48.8 and 42.9; heads of 80, three behind 160 10.6 and 10.4.)
template <int G, int NW, bool STEP>
__global__ void __launch_bounds__(KA_WAVE * NW) attention_spread_kernel(SpreadArgs g) {
    constexpr int GROUPS = KA_WAVE / G, CK = 16 * GROUPS, R = G / 4;         // groups of 16 keys in a chunk of CK; channels in sixteens
    __shared__ long k_at[NW][CK], v_at[NW][CK];
    __shared__ __attribute__((aligned(16))) float ps[NW][CK];
    __shared__ float sums[AS_PARTS][R * 16], tops[AS_PARTS], totals[AS_PARTS];
    const int t = blockIdx.x, h = blockIdx.y, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KA_WAVE), lane = threadIdx.x % KA_WAVE;
    const int vh = h / g.maps / (g.H / g.Hkv), kvh = vh * g.maps + h % g.maps, Hv = g.Hkv / g.maps;
    const int lo = g.kv_lo ? g.kv_lo[t] : 0, hi = g.kv_hi[t];
    const int* bt = g.block_table + (size_t)g.token_row[t] * g.max_pages;
    const int in_row = lane % G, group = lane / G;
    const bool owns = in_row < 16;                       // (the other rows of a group hold the same keys' scores once more)
    as_floatx4 q4 = {0.f, 0.f, 0.f, 0.f};
    as_floatx4 own_k = {0.f, 0.f, 0.f, 0.f};
    float own_v[R];
    const int slot = STEP ? g.slots[t] : -1;
    if constexpr (STEP) {
        const float *row = g.q + (size_t)t * g.q_row_stride, *krow = row + (size_t)g.H * g.hd + (size_t)kvh * g.hd, *vrow = row + (size_t)(g.H + g.Hkv) * g.hd + (size_t)kvh * g.hd;
        const float* cs = g.rot ? g.table + (size_t)g.positions[t] * g.rot : nullptr;
#pragma unroll
        for (int r = 0; r < R; ++r) own_v[r] = vrow[min(r * 16 + lane / 4, g.hdv - 1)];
        if (in_row * 4 < g.hd) {
            q4 = as_rotated(row + (size_t)h * g.hd, cs, g.rot, g.interleaved, in_row * 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) q4[i] *= g.scale;
            own_k = as_rotated(krow, cs, g.rot, g.interleaved, in_row * 4);
        }
        if (slot >= 0 && wave == 0 && h % (g.H / g.Hkv) == 0) {
            const long page = slot / g.page_size;
            const int off = slot % g.page_size;
            if (group == 0 && in_row * 4 < g.hd)
                *reinterpret_cast<as_floatx4*>(const_cast<float*>(g.k_cache) + ((page * g.Hkv + kvh) * g.page_size + off) * g.hd + in_row * 4) = own_k;
            if (lane % 4 == 0)
#pragma unroll
                for (int r = 0; r < R; ++r)
                    if (r * 16 + lane / 4 < g.hdv) const_cast<float*>(g.v_cache)[((page * g.Hkv + kvh) * g.hdv + r * 16 + lane / 4) * g.page_size + off] = own_v[r];
        }
    } else if (in_row * 4 < g.hd) {
        const float* qp = g.q + (size_t)t * g.q_row_stride + (size_t)h * g.hd + in_row * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) q4[i] = qp[i] * g.scale;
    }
    const float slope = g.slopes ? g.slopes[h] : 0.f;
    const int place = (g.slopes || g.bias_table) ? g.positions[t] : 0;
    const float* bias_row = g.bias_table ? g.bias_table + (size_t)h * g.bias_len : nullptr;
    const float sink = g.sinks ? g.sinks[h] : g.sink_score;

    // chunks of the kept first keys, then of the window's, whose first chunk starts on a multiple of four keys; part p has every AS_PARTS-th from chunk p on
    const int kept = min(g.keep_first, lo), kept_chunks = kept > 0 ? (kept + CK - 1) / CK : 0;
    const int start = lo & ~3, chunks = kept_chunks + (hi > lo ? (hi - start + CK - 1) / CK : 0);
    const int parts = max(1, min(AS_PARTS, chunks));     // (the first one also without a key, for the sink)
    for (int part = wave; part < parts; part += NW) {
        const bool sinks_here = g.has_sink && part == 0;
        float m = sinks_here ? sink : -INFINITY, l = sinks_here ? 1.f : 0.f;
        float o[R];
#pragma unroll
        for (int r = 0; r < R; ++r) o[r] = 0.f;
        for (int c = part; c < chunks; c += AS_PARTS) {
            const bool first = c < kept_chunks;
            const int base = first ? c * CK : start + (c - kept_chunks) * CK, from = first ? 0 : lo, to = first ? kept : hi;
            const int key = base + group * 16 + lane % 16;
            const bool valid = key >= from && key < to;
            int own = -1;                                // STEP: the place in the chunk of the token's own key
            {
                const int near = min(max(key, from), to - 1), page = bt[near / g.page_size], at = near % g.page_size;
                if constexpr (STEP) {
                    const unsigned long long hit = __ballot(owns && valid && page * g.page_size + at == slot);
                    if (hit) own = (int)__builtin_ctzll(hit) / G * 16 + (int)__builtin_ctzll(hit) % G;
                }
                as_wave_sync();                          // the chunk before has been read
                if (owns) {
                    k_at[wave][group * 16 + in_row] = (((long)page * g.Hkv + kvh) * g.page_size + at) * g.hd;
                    v_at[wave][group * 16 + in_row] = ((long)page * Hv + vh) * g.hdv * g.page_size + (at & ~3);
                }
                as_wave_sync();
            }
            as_floatx4 k4[16], v4[GROUPS][R];
            const int channel = min(in_row * 4, g.hd - 4);
#pragma unroll
            for (int i = 0; i < 16; ++i) k4[i] = *reinterpret_cast<const as_floatx4*>(g.k_cache + k_at[wave][group * 16 + i] + channel);
#pragma unroll
            for (int x = 0; x < GROUPS; ++x) {
                const float* vp = g.v_cache + v_at[wave][x * 16 + lane % 4 * 4];
#pragma unroll
                for (int r = 0; r < R; ++r) v4[x][r] = *reinterpret_cast<const as_floatx4*>(vp + (long)min(r * 16 + lane / 4, g.hdv - 1) * g.page_size);
            }
            if (STEP && own >= 0) {
#pragma unroll
                for (int i = 0; i < 16; ++i) k4[i] = group * 16 + i == own ? own_k : k4[i];
#pragma unroll
                for (int x = 0; x < GROUPS; ++x)
#pragma unroll
                    for (int r = 0; r < R; ++r)
#pragma unroll
                        for (int i = 0; i < 4; ++i) v4[x][r][i] = x * 16 + lane % 4 * 4 + i == own ? own_v[r] : v4[x][r][i];
            }
            float part_s[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) part_s[i] = fmaf(q4[3], k4[i][3], fmaf(q4[2], k4[i][2], fmaf(q4[1], k4[i][1], q4[0] * k4[i][0])));
            as_scatter_sums<8>(part_s, lane);
            float s = ka_lanes_reduce<16, G>(part_s[0], KaSum{});
            if (g.softcap > 0.f) s = g.softcap * tanhf(s / g.softcap);
            if (g.slopes) s -= slope * (float)(place - key);
            if (bias_row) s += bias_row[min(max(place - key, 0), g.bias_len - 1)];
            if (!valid) s = -INFINITY;
            const float m_new = fmaxf(m, ka_wave_max(s));
            const float corr = m == m_new ? 1.f : expf(m - m_new);
            const float p = s == -INFINITY ? 0.f : expf(s - m_new);      // (a table may shut out all keys of a chunk: m_new is -inf as well)
            l = l * corr + ka_wave_sum(owns ? p : 0.f);
            m = m_new;
            if (owns) ps[wave][group * 16 + in_row] = p;
            as_wave_sync();
            const bool whole = base >= from && base + CK <= to;
#pragma unroll
            for (int r = 0; r < R; ++r) o[r] *= corr;
#pragma unroll
            for (int x = 0; x < GROUPS; ++x) {
                const int j = x * 16 + lane % 4 * 4;
                const as_floatx4 p4 = *reinterpret_cast<const as_floatx4*>(&ps[wave][j]);
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    as_floatx4 v = v4[x][r];
                    if (!whole) {                        // (a place without a key may hold anything)
#pragma unroll
                        for (int i = 0; i < 4; ++i) v[i] = base + j + i >= from && base + j + i < to ? v[i] : 0.f;
                    }
                    o[r] += fmaf(p4[3], v[3], fmaf(p4[2], v[2], fmaf(p4[1], v[1], p4[0] * v[0])));
                }
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float y = ka_lanes_reduce<1, 4>(o[r], KaSum{});
            if (lane % 4 == 0) sums[part][r * 16 + lane / 4] = y;
        }
        if (lane == 0) {
            tops[part] = m;
            totals[part] = l;
        }
    }
    __syncthreads();
    float top = -INFINITY, total = 0.f, share[AS_PARTS];
#pragma unroll
    for (int w = 0; w < AS_PARTS; ++w) top = w < parts ? fmaxf(top, tops[w]) : top;
#pragma unroll
    for (int w = 0; w < AS_PARTS; ++w) {
        if (w >= parts) break;
        share[w] = tops[w] == top ? 1.f : expf(tops[w] - top);           // (a part without a key: exp(-inf), or nothing at all)
        total += totals[w] * share[w];
    }
    const float inv = total > 0.f ? 1.0f / total : 0.f;
    const float head_gate = g.gate && g.gate_per_head ? 1.0f / (1.0f + expf(-g.gate[(size_t)t * g.gate_row_stride + h])) : 1.f;
    for (int d = threadIdx.x; d < g.hdv; d += KA_WAVE * NW) {
        float y = 0.f;
#pragma unroll
        for (int w = 0; w < AS_PARTS; ++w) {
            if (w >= parts) break;
            y += sums[w][d] * share[w];
        }
        y *= inv * head_gate;
        if (g.gate && !g.gate_per_head) y *= 1.0f / (1.0f + expf(-g.gate[(size_t)t * g.gate_row_stride + (size_t)h * g.hdv + d]));
        g.out[(size_t)t * g.out_row_stride + (size_t)h * g.hdv + d] = y;
    }
}

template <int G>
static void launch_spread(const SpreadArgs& g, int n, hipStream_t stream) {
    // A wave a part where workgroups of four waves are two a CU at the most, else one wave for all: heads of 64, us, four waves and one: 3 tokens behind 160
    // keys 6.5 and 8.7, 16 behind 200 14.2 and 17.3, but 32 behind 64 8.9 and 8.6, a prompt of 33 9.4 and 6.4, six of 20 21 and 9.3. Long rows
    // of many tokens do not care (64 behind 400 76 and 74).
    if ((long)n * g.H <= 2L * ka_compute_units()) hipLaunchKernelGGL((attention_spread_kernel<G, AS_PARTS, false>), dim3(n, g.H), dim3(AS_PARTS * KA_WAVE), 0, stream, g);
    else hipLaunchKernelGGL((attention_spread_kernel<G, 1, false>), dim3(n, g.H), dim3(KA_WAVE), 0, stream, g);
}

KA_API int ka_attention_generic(const void* q, int dtype, long q_row_stride, const void* k_cache,
                                const void* v_cache, const int* block_table, int max_pages,
                                const int* token_row, const int* kv_lo, const int* kv_hi, void* out,
                                long out_row_stride, float scale, int n, int H, int Hkv, int hd,
                                int page_size, int hdv, const int* positions, const float* slopes,
                                int has_sink, float sink_score, const float* bias_table, int bias_len,
                                const void* gate, long gate_row_stride, const float* sinks, int keep_first, int maps,
                                int values_in_keys, int out_f32, float softcap, int gate_per_head, hipStream_t stream) {
    KA_CHECK(softcap >= 0.f, "ka_attention_generic: a cap on the scores must be positive");
    KA_CHECK(maps >= 1 && H % maps == 0 && Hkv % maps == 0 && keep_first >= 0, "ka_attention_generic: %d maps do not divide the heads %d and %d", maps, H, Hkv);
    KA_CHECK(!values_in_keys || hdv <= hd, "ka_attention_generic: values inside keys of %d channels cannot have %d", hd, hdv);
    KA_CHECK(sinks == nullptr || has_sink, "ka_attention_generic: sink scores without a sink");
    KA_CHECK(bias_table == nullptr || (positions != nullptr && bias_len > 0), "ka_attention_generic: a distance table needs the queries' positions");
    KA_CHECK(n >= 0 && H > 0 && Hkv > 0 && hd > 0 && hdv > 0, "ka_attention_generic: bad sizes");
    KA_CHECK(hdv <= ATT_MAX_HD, "ka_attention_generic: value size %d above %d", hdv, ATT_MAX_HD);
    KA_CHECK(slopes == nullptr || positions != nullptr, "ka_attention_generic: slopes need the queries' positions");
    KA_CHECK(H % Hkv == 0, "ka_attention_generic: %d query heads do not divide into %d kv heads", H, Hkv);
    KA_CHECK(hd <= ATT_MAX_HD, "ka_attention_generic: head size %d above %d", hd, ATT_MAX_HD);
    KA_CHECK(H <= 65535, "ka_attention_generic: too many heads %d", H);
    KA_CHECK(page_size > 0 && max_pages > 0, "ka_attention_generic: bad paging %d %d", page_size, max_pages);
    if (n == 0) return 0;
    dim3 grid(n, H), block(KA_WAVE);
    if (dtype == KA_F32 && !values_in_keys && hd % 4 == 0 && hd <= 256 && hdv <= 256 && page_size % 4 == 0 &&
        ((uintptr_t)k_cache | (uintptr_t)v_cache) % 16 == 0) {
        const SpreadArgs g{(const float*)q, q_row_stride, (const float*)k_cache, (const float*)v_cache, block_table, max_pages, token_row, kv_lo, kv_hi,
                           (float*)out, out_row_stride, scale, H, Hkv, hd, hdv, page_size, positions, slopes, has_sink, sink_score, bias_table, bias_len,
                           (const float*)gate, gate_row_stride, sinks, keep_first, maps, softcap, gate_per_head, nullptr, nullptr, 0, 0};
        const int wide = hd > hdv ? hd : hdv;
        if (wide <= 64) launch_spread<16>(g, n, stream);
        else if (wide <= 128) launch_spread<32>(g, n, stream);
        else launch_spread<64>(g, n, stream);
    } else if (dtype == KA_F32)
        hipLaunchKernelGGL(attention_generic_kernel<float>, grid, block, 0, stream, (const float*)q, q_row_stride,
                           (const float*)k_cache, (const float*)v_cache, block_table, max_pages, token_row, kv_lo,
                           kv_hi, (float*)out, out_row_stride, scale, H, Hkv, hd, hdv, page_size, positions, slopes, has_sink,
                           sink_score, bias_table, bias_len, (const float*)gate, gate_row_stride, sinks, keep_first, maps, values_in_keys, out_f32, softcap, gate_per_head);
    else if (dtype == KA_BF16)
        hipLaunchKernelGGL(attention_generic_kernel<bf16_t>, grid, block, 0, stream, (const bf16_t*)q, q_row_stride,
                           (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_table, max_pages, token_row, kv_lo,
                           kv_hi, (bf16_t*)out, out_row_stride, scale, H, Hkv, hd, hdv, page_size, positions, slopes, has_sink,
                           sink_score, bias_table, bias_len, (const bf16_t*)gate, gate_row_stride, sinks, keep_first, maps, values_in_keys, out_f32, softcap, gate_per_head);
    else
        KA_CHECK(false, "ka_attention_generic: unsupported dtype %d", dtype);
    KA_LAUNCH_CHECK();
    return 0;
}

// A step of single tokens in 32 bits: rotation, cache write and attention in one launch. qkv rows: [H hd q | Hkv hd k | Hkv hd v], not changed. 1: done; 0: not covered,
// nothing was run; -1: an error.
KA_API int ka_attention_step_f32(const float* qkv, long row_stride, float* k_cache, float* v_cache, const int* block_table, int max_pages, const int* token_row, const int* kv_lo,
                                 const int* kv_hi, float* out, long out_row_stride, float scale, int n, int H, int Hkv, int hd, int page_size, const int* positions,
                                 const int* slots, const float* table, int table_rows, int rot, int interleaved, hipStream_t stream) {
    const char* who = "ka_attention_step_f32";
    KA_CHECK(n > 0 && H > 0 && Hkv > 0 && hd > 0 && H % Hkv == 0 && H <= 65535, "%s: n=%d heads %d, %d of %d", who, n, H, Hkv, hd);
    KA_CHECK(page_size > 0 && max_pages > 0 && slots && row_stride >= (long)(H + 2 * Hkv) * hd && out_row_stride >= (long)H * hd, "%s: pages of %d, %d a row, strides %ld and %ld", who,
             page_size, max_pages, row_stride, out_row_stride);
    KA_CHECK(rot >= 0 && rot <= hd && rot % 2 == 0 && (rot == 0 || (table && table_rows > 0 && positions)), "%s: rotation of %d channels", who, rot);
    // (one workgroup a CU at the most: with 214 to 240 registers instead of 126 to 160 two of them share a CU worse; 16 tokens of 32 heads behind 200 keys 19.5 us, the two launches 18.3)
    if ((long)n * H > ka_compute_units() || hd % 4 || hd > 256 || page_size % 4 || row_stride % 4 || ((uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)qkv) % 16) return 0;
    const SpreadArgs g{qkv, row_stride, k_cache, v_cache, block_table, max_pages, token_row, kv_lo, kv_hi, out, out_row_stride, scale, H, Hkv, hd, hd, page_size, positions,
                       nullptr, 0, 0.f, nullptr, 0, nullptr, 0, nullptr, 0, 1, 0.f, 0, slots, table, rot, interleaved};
    if (hd <= 64) hipLaunchKernelGGL((attention_spread_kernel<16, AS_PARTS, true>), dim3(n, H), dim3(AS_PARTS * KA_WAVE), 0, stream, g);
    else if (hd <= 128) hipLaunchKernelGGL((attention_spread_kernel<32, AS_PARTS, true>), dim3(n, H), dim3(AS_PARTS * KA_WAVE), 0, stream, g);
    else hipLaunchKernelGGL((attention_spread_kernel<64, AS_PARTS, true>), dim3(n, H), dim3(AS_PARTS * KA_WAVE), 0, stream, g);
    KA_LAUNCH_CHECK();
    return 1;
}
