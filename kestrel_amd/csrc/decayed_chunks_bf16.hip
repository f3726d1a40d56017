// The decaying matrix memory (recurrent_parts.hip) over prompt portions: the walk over a row's tokens, cut into chunks of 64 that run at
// once. All arithmetic is fp32 and is the walk's: per head and token
//     o_j = sum_i r_i (S_ij + u_i k_i v_j),   S_ij <- w_i S_ij + k_i v_j,   w_i = e^(-e^(pre_i)).
// Three launches meet in a buffer of the caller's (per chunk and head S [d, d], then per chunk and head the factors [d]):
//  * LOCAL walks over every chunk but a row's last from S = 0 and leaves what the chunk adds to the state, and prod w, the part of a
//    state that outlives it;
//  * SCAN takes a row's chunks in order and turns those into the state that every chunk starts from;
//  * READ walks over every chunk from there with the read-outs; a row's last chunk leaves the request's state.
// A row of one chunk needs the last alone. Decays meet as factors, never as logarithms, so a decay of any size leaves what comes after
// it untouched; a token's numbers depend on tokens before it alone, whatever they hold.
//
// A thread keeps 4 key channels of 4 value channels (16 numbers of S): a token's r, k and w of four channels and v of four cost it four
// LDS reads for 48 (LOCAL 32) multiply-adds; with one value channel a thread, as the walk of whole rows has it, LDS bounds the loop.
// The KEYS lanes that hold the key channels of a value channel are neighbours: their read-outs meet by lane moves.
//
// Bound by the multiply-adds of the vector unit, five a number of S and token in both walks, where chunks fill the chip, and by the 64
// tokens of a chunk one after the other where they do not (0.28 us each with read-outs, 0.16 without). Measured, us, 32 heads of 64, one walk of a row and the
// norm's launch -> here: 2,048 tokens of one row 613 -> 70; two rows of 800 248 -> 65; eight of 100 78 -> 41; 128 tokens 44 -> 30; 65 27 -> 29; 16 heads of
// 128, 512 tokens 188 -> 50. On the matrix cores, where keys and queries meet as scores and carry powers of differences of logarithms: 90, 85, 50,
// 33, 33 and 68, with sixteen bits of what carries a power, fewer behind a run of small decays, and later tokens' values multiplied with zeros.
#include "ka_common.h"

typedef __attribute__((ext_vector_type(4))) __bf16 dc_bf16x4;

constexpr int DC_CHUNK = 64;
constexpr int DC_BLOCK = 16;                // tokens staged at once
constexpr int DC_THREADS = 256;
constexpr int DC_MAX_D = 224;

struct DecayedChunkArgs {
    const bf16_t* r;
    const bf16_t* k;
    const bf16_t* v;
    const bf16_t* gate;
    long stride;                // of the rows of r, k, v and gate
    const float* pre;           // [n, H d]
    const float* u;             // [H d]
    const float* gain;          // [H d]
    float* state;               // [slots, state_stride]: S [H, d, d], then the kept row [dim]
    long state_stride;
    const float* x;             // [n, dim]: the rows whose last one a request keeps, or null
    int dim;
    const int* cu_q;
    const int* row_slot;
    bf16_t* out;                // rows of out_stride, normalised and gated; null: read-outs to raw
    long out_stride;
    float* raw;                 // [n, H d]
    float* chunks;              // [chunks, H, d, d]
    float* factors;             // [chunks, H, d]
    int n_rows, H, d;
    float eps;
};

// The row of chunk `g` of the step (chunks numbered row by row), its first and last token, the chunk's place among the row's and the
// number of the row's first chunk; false: behind the last chunk. A lane looks at a row, 64 rows at a time.
__device__ __forceinline__ bool dc_find_chunk(const DecayedChunkArgs& a, int g, int& row, int& t0, int& t1, int& place) {
    const int lane = threadIdx.x % KA_WAVE;
    int base = 0;
    for (int r0 = 0; r0 < a.n_rows; r0 += KA_WAVE) {
        const int r = r0 + lane;
        const int first = r < a.n_rows ? a.cu_q[r] : 0, end = r < a.n_rows ? a.cu_q[r + 1] : 0;
        const int nc = (end - first + DC_CHUNK - 1) / DC_CHUNK;
        const int upto = base + (int)ka_wave_running_sum((float)nc);          // (counts of chunks: exact in fp32)
        const unsigned long long hit = __builtin_amdgcn_ballot_w64(g < upto && g >= upto - nc);
        if (hit != 0) {
            const int src = __builtin_ctzll(hit);
            row = r0 + src;
            place = g - __builtin_amdgcn_readlane(upto - nc, src);
            t0 = __builtin_amdgcn_readlane(first, src);
            t1 = __builtin_amdgcn_readlane(end, src);
            return true;
        }
        base = __builtin_amdgcn_readlane(upto, KA_WAVE - 1);
    }
    return false;
}

// The sum over groups of KEYS lanes of four numbers each; lane l ends with number (l % 4): 0 2 1 3.
template <int KEYS>
__device__ __forceinline__ float dc_lanes_sum(const float4& q) {
    const int lane = threadIdx.x;
    const bool odd = lane & 1, second = lane & 2;
    const float a = (odd ? q.z : q.x) + ka_dpp_move<0xB1>(odd ? q.x : q.z);            // quad_perm [1,0,3,2]
    const float b = (odd ? q.w : q.y) + ka_dpp_move<0xB1>(odd ? q.y : q.w);
    float s = (second ? b : a) + ka_dpp_move<0x4E>(second ? a : b);                    // quad_perm [2,3,0,1]
    s += ka_dpp_move<0x128>(s);                                                        // row_ror:8
    s += ka_dpp_move<0x124>(s);                                                        // row_ror:4
    return ka_lanes_reduce<16, KEYS>(s, KaSum{});
}
__device__ __forceinline__ int dc_lane_channel() { return (threadIdx.x & 1) * 2 + (threadIdx.x >> 1 & 1); }

// KEYS lanes hold the key channels (4 each, zeros behind the last), DC_THREADS / KEYS groups of them four value channels each. Grid (H,
// chunks, slices of value channels).
template <int KEYS, bool READ>
__global__ void __launch_bounds__(DC_THREADS) __attribute__((amdgpu_waves_per_eu(KEYS == 16 ? 4 : KEYS == 32 ? 3 : 2)))
decayed_chunk_kernel(DecayedChunkArgs a) {
    constexpr int WIDTH = KEYS * 4, GROUPS = DC_THREADS / KEYS, SLICE = GROUPS * 4;
    constexpr int LOADS = KEYS / 16;                     // pieces of four channels a thread brings of a block's r, k and w
    constexpr int STEP = DC_THREADS / KEYS;              // tokens that one of them covers for all threads
    __shared__ __attribute__((aligned(16))) float rs[READ ? DC_BLOCK * WIDTH : 4], ks[DC_BLOCK * WIDTH], ws[DC_BLOCK * WIDTH];
    // (of two blocks in turn: the read-outs of one are finished while the next one is staged)
    __shared__ __attribute__((aligned(16))) float vs[2][DC_BLOCK * SLICE], os[READ ? 2 : 1][READ ? DC_BLOCK * SLICE : 4], bonus[2][DC_BLOCK];
    int row, t0, t1, place;
    if (!dc_find_chunk(a, blockIdx.y, row, t0, t1, place)) return;
    const int c0 = t0 + place * DC_CHUNK, c1 = min(c0 + DC_CHUNK, t1);
    const bool last = c1 == t1;
    if (!READ && last) return;
    const int head = blockIdx.x, tid = threadIdx.x, wave = tid / KA_WAVE, lane = tid % KA_WAVE, d = a.d, j0 = blockIdx.z * SLICE;
    const int slot = a.row_slot[row];
    if (slot < 0) {
        if (READ)
            for (int e = tid; e < (c1 - c0) * SLICE; e += DC_THREADS) {
                const int t = c0 + e / SLICE, j = j0 + e % SLICE;
                if (j >= d) continue;
                if (a.out) a.out[(size_t)t * a.out_stride + (size_t)head * d + j] = (bf16_t)0.f;
                else a.raw[(size_t)t * a.H * d + (size_t)head * d + j] = 0.f;
            }
        return;
    }
    const int p = tid % KEYS, group = tid / KEYS, i0 = p * 4, jl = group * 4, j = j0 + jl;
    const bool mine = i0 < d && j < d;
    float* const S_mem = a.state + (size_t)slot * a.state_stride + (size_t)head * d * d;
    float* const record = a.chunks + ((size_t)blockIdx.y * a.H + head) * d * d;
    float S[4][4];
    {
        const float* from = place == 0 && last ? S_mem : record;
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) {
            const float* at = from + (size_t)(i0 + ii) * d + j;
            // (a request's state may start anywhere)
            if (READ && mine)
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) S[ii][jj] = at[jj];
            else
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) S[ii][jj] = 0.f;
        }
    }
    // what a thread brings of a block: the channels of lane p, of tokens tid / KEYS, STEP further and so on; four value channels of a token
    const dc_bf16x4 none = {(bf16_t)0.f, (bf16_t)0.f, (bf16_t)0.f, (bf16_t)0.f};
    const bool brings = i0 < d;
    const int v_tok = tid / GROUPS, v_at = j0 + tid % GROUPS * 4;
    const bool brings_v = v_tok < DC_BLOCK && v_at < d;
    const float4 u4 = READ && brings ? *reinterpret_cast<const float4*>(a.u + (size_t)head * d + i0) : make_float4(0.f, 0.f, 0.f, 0.f);
    dc_bf16x4 fr[LOADS], fk[LOADS], fv = none;
    float4 fw[LOADS];
    auto fetch = [&](int tb) {
#pragma unroll
        for (int m = 0; m < LOADS; ++m) {
            const int t = tb + group + m * STEP;
            fr[m] = none;
            fk[m] = none;
            fw[m] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (brings && t < c1) {
                const size_t at = (size_t)t * a.stride + (size_t)head * d + i0;
                if (READ) fr[m] = *reinterpret_cast<const dc_bf16x4*>(a.r + at);
                fk[m] = *reinterpret_cast<const dc_bf16x4*>(a.k + at);
                fw[m] = *reinterpret_cast<const float4*>(a.pre + (size_t)t * a.H * d + (size_t)head * d + i0);
            }
        }
        fv = none;
        if (brings_v && tb + v_tok < c1) fv = *reinterpret_cast<const dc_bf16x4*>(a.v + (size_t)(tb + v_tok) * a.stride + (size_t)head * d + v_at);
    };
    // (a token behind the chunk's last: r and k are 0 and the decay is 1, which leaves S as it is without a branch)
    auto decay = [](float z, bool in) { return in ? __expf(-__expf(z)) : 1.f; };
    auto barrier = [] {                                  // (LDS alone: the next block's numbers stay on their way)
        __builtin_amdgcn_s_waitcnt(0xc07f);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    float4 kept = make_float4(1.f, 1.f, 1.f, 1.f);       // LOCAL: the product of the decays
    fetch(c0);
    int buf = 0;
    for (int tb = c0; tb < c1; tb += DC_BLOCK, buf ^= 1) {
        const int nb = min(DC_BLOCK, c1 - tb);
#pragma unroll
        for (int m = 0; m < LOADS; ++m) {
            const int at = (group + m * STEP) * WIDTH + i0;
            const bool in = tb + group + m * STEP < c1;
            const float4 k = make_float4((float)fk[m][0], (float)fk[m][1], (float)fk[m][2], (float)fk[m][3]);
            *reinterpret_cast<float4*>(ks + at) = k;
            *reinterpret_cast<float4*>(ws + at) = make_float4(decay(fw[m].x, in), decay(fw[m].y, in), decay(fw[m].z, in), decay(fw[m].w, in));
            if constexpr (READ) {
                const float4 r = make_float4((float)fr[m][0], (float)fr[m][1], (float)fr[m][2], (float)fr[m][3]);
                *reinterpret_cast<float4*>(rs + at) = r;
                const float part = ((r.x * u4.x * k.x + r.y * u4.y * k.y) + r.z * u4.z * k.z) + r.w * u4.w * k.w;
                const float sum = ka_lanes_reduce<1, KEYS>(part, KaSum{});
                if (p == 0) bonus[buf][group + m * STEP] = sum;
            }
        }
        if (v_tok < DC_BLOCK) *reinterpret_cast<float4*>(&vs[buf][v_tok * SLICE + tid % GROUPS * 4]) = make_float4((float)fv[0], (float)fv[1], (float)fv[2], (float)fv[3]);
        if (tb + DC_BLOCK < c1) fetch(tb + DC_BLOCK);
        barrier();
        // (two tokens ahead: a trip through LDS takes as long as the sums of about one)
        constexpr int AHEAD = 2;
        float4 rq[AHEAD], kq[AHEAD], wq[AHEAD], vq[AHEAD];
        auto ask = [&](int tt) {
            const int q = tt % AHEAD;
            if constexpr (READ) rq[q] = *reinterpret_cast<const float4*>(rs + tt * WIDTH + i0);
            kq[q] = *reinterpret_cast<const float4*>(ks + tt * WIDTH + i0);
            wq[q] = *reinterpret_cast<const float4*>(ws + tt * WIDTH + i0);
            vq[q] = *reinterpret_cast<const float4*>(&vs[buf][tt * SLICE + jl]);
        };
#pragma unroll
        for (int q = 0; q < AHEAD; ++q) ask(q);
        float sums[DC_BLOCK / 4];                        // of the lane's tokens, every fourth
#pragma unroll
        for (int tt = 0; tt < DC_BLOCK; ++tt) {
            const int q = tt % AHEAD;
            const float k[4] = {kq[q].x, kq[q].y, kq[q].z, kq[q].w}, w[4] = {wq[q].x, wq[q].y, wq[q].z, wq[q].w};
            const float v[4] = {vq[q].x, vq[q].y, vq[q].z, vq[q].w};
            float r[4] = {0.f, 0.f, 0.f, 0.f};
            if constexpr (READ) { r[0] = rq[q].x; r[1] = rq[q].y; r[2] = rq[q].z; r[3] = rq[q].w; }
            if (tt + AHEAD < DC_BLOCK) ask(tt + AHEAD);
            float o[4];
#pragma unroll
            for (int ii = 0; ii < 4; ++ii)
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) {
                    if constexpr (READ) o[jj] = ii == 0 ? r[0] * S[0][jj] : fmaf(r[ii], S[ii][jj], o[jj]);
                    S[ii][jj] = fmaf(w[ii], S[ii][jj], k[ii] * v[jj]);
                }
            if constexpr (READ) {
                const float sum = dc_lanes_sum<KEYS>(make_float4(o[0], o[1], o[2], o[3]));
                sums[tt / 4] = tt % 4 == 0 || p / 4 % 4 == tt % 4 ? sum : sums[tt / 4];
            } else {
                kept = make_float4(kept.x * w[0], kept.y * w[1], kept.z * w[2], kept.w * w[3]);
            }
        }
        if constexpr (READ) {
            if (p < 16)
#pragma unroll
                for (int q = 0; q < DC_BLOCK / 4; ++q) os[buf][(q * 4 + p / 4) * SLICE + jl + dc_lane_channel()] = sums[q];
        }
        barrier();
        if constexpr (READ) {
            if (a.out != nullptr) {
                // (one slice: a wave finishes a token's head)
                for (int tt = wave; tt < nb; tt += DC_THREADS / KA_WAVE) {
                    const bool in = lane < d;
                    const float o = in ? fmaf(bonus[buf][tt], vs[buf][tt * SLICE + lane % SLICE], os[buf][tt * SLICE + lane % SLICE]) : 0.f;
                    const float inv = 1.0f / sqrtf(ka_wave_sum(o * o) / (float)d + a.eps);
                    const size_t c = (size_t)head * d + lane;
                    if (in) a.out[(size_t)(tb + tt) * a.out_stride + c] = (bf16_t)(o * inv * a.gain[c] * (float)a.gate[(size_t)(tb + tt) * a.stride + c]);
                }
            } else {
                for (int e = tid; e < nb * SLICE; e += DC_THREADS) {
                    const int tt = e / SLICE, c = e % SLICE;
                    if (j0 + c < d)
                        a.raw[(size_t)(tb + tt) * a.H * d + (size_t)head * d + j0 + c] = fmaf(bonus[buf][tt], vs[buf][e], os[buf][e]);
                }
            }
        }
    }
    if (READ && !last) return;
    if (mine) {
        float* to = READ ? S_mem : record;
#pragma unroll
        for (int ii = 0; ii < 4; ++ii)
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) to[(size_t)(i0 + ii) * d + j + jj] = S[ii][jj];
        if (!READ && group == 0 && blockIdx.z == 0) *reinterpret_cast<float4*>(a.factors + ((size_t)blockIdx.y * a.H + head) * d + i0) = kept;
    }
    if (READ && head == 0 && blockIdx.z == 0 && a.x != nullptr)
        for (int c = tid; c < a.dim; c += DC_THREADS) a.state[(size_t)slot * a.state_stride + (size_t)a.H * d * d + c] = a.x[(size_t)(t1 - 1) * a.dim + c];
}

// Grid (H, rows, pieces of 1,024 numbers of S): four numbers a thread.
__global__ void __launch_bounds__(DC_THREADS) decayed_scan_kernel(DecayedChunkArgs a) {
    const int head = blockIdx.x, row = blockIdx.y, tid = threadIdx.x, lane = tid % KA_WAVE, d = a.d;
    const int nc = (a.cu_q[row + 1] - a.cu_q[row] + DC_CHUNK - 1) / DC_CHUNK, slot = a.row_slot[row];
    if (nc < 2 || slot < 0) return;
    int before = 0;
    for (int r = lane; r < row; r += KA_WAVE) before += (a.cu_q[r + 1] - a.cu_q[r] + DC_CHUNK - 1) / DC_CHUNK;
    const int base = (int)ka_wave_sum((float)before);
    const int e = (blockIdx.z * DC_THREADS + tid) * 4;
    if (e >= d * d) return;
    const float* st = a.state + (size_t)slot * a.state_stride + (size_t)head * d * d + e;
    float4 cur = make_float4(st[0], st[1], st[2], st[3]);
    const size_t step = (size_t)a.H * d * d, step_f = (size_t)a.H * d;
    float* rec = a.chunks + ((size_t)base * a.H + head) * d * d + e;
    const float* fac = a.factors + ((size_t)base * a.H + head) * d + e / d;
    constexpr int AHEAD = 4;                             // chunks whose numbers are asked for at once
    for (int c = 0; c < nc; c += AHEAD) {
        float4 x[AHEAD];
        float f[AHEAD];
#pragma unroll
        for (int q = 0; q < AHEAD; ++q) {
            const int at = min(c + q, nc - 2);           // (the last chunk has left nothing)
            x[q] = *reinterpret_cast<const float4*>(rec + at * step);
            f[q] = fac[at * step_f];
        }
#pragma unroll
        for (int q = 0; q < AHEAD; ++q) {
            if (c + q >= nc) break;
            *reinterpret_cast<float4*>(rec + (c + q) * step) = cur;
            cur = make_float4(fmaf(f[q], cur.x, x[q].x), fmaf(f[q], cur.y, x[q].y), fmaf(f[q], cur.z, x[q].z), fmaf(f[q], cur.w, x[q].w));
        }
    }
}

KA_API int ka_decayed_chunks_supported(int d) { return d > 0 && d % 16 == 0 && d <= DC_MAX_D ? 1 : 0; }

template <int KEYS>
static void decayed_chunks_launch(const DecayedChunkArgs& a, int n, int n_chunks, hipStream_t stream) {
    const int slices = ka_cdiv(a.d, DC_THREADS / KEYS * 4);
    if (n > DC_CHUNK) {                                  // (else no row has two chunks)
        hipLaunchKernelGGL((decayed_chunk_kernel<KEYS, false>), dim3(a.H, n_chunks, slices), dim3(DC_THREADS), 0, stream, a);
        hipLaunchKernelGGL(decayed_scan_kernel, dim3(a.H, a.n_rows, ka_cdiv(a.d * a.d, 4 * DC_THREADS)), dim3(DC_THREADS), 0, stream, a);
    }
    hipLaunchKernelGGL((decayed_chunk_kernel<KEYS, true>), dim3(a.H, n_chunks, slices), dim3(DC_THREADS), 0, stream, a);
}

// Operands as ka_decayed_memory's; `scratch`: a state [d, d] and its factors [d] per chunk (n / DC_CHUNK + n_rows of them) and head. Heads of up to 64 channels leave normalised and gated, in `out` (returns 0, `raw` is not written); the
// read-outs of larger ones are left in `raw` (returns 1: ka_decayed_readout finishes them).
KA_API int ka_decayed_chunks_bf16(const void* r, const void* k, const void* v, const void* gate, long stride, const float* pre, const float* u,
                                  const float* gain, float* state, long state_stride, const float* x, int dim, const int* cu_q, const int* row_slot,
                                  void* out, long out_stride, float* raw, float* scratch, int n, int n_rows, int H, int d, float eps,
                                  hipStream_t stream) {
    const char* who = "ka_decayed_chunks_bf16";
    KA_CHECK(n >= 0 && n_rows >= 0 && H > 0 && eps >= 0.f && ka_decayed_chunks_supported(d), "%s: heads of %d not covered", who, d);
    KA_CHECK(pre != nullptr && u != nullptr && dim >= 0, "%s: a decay needs its pre-activations, a token its bonus", who);
    KA_CHECK(((uintptr_t)r | (uintptr_t)k | (uintptr_t)v) % 8 == 0 && stride % 4 == 0 && ((uintptr_t)pre | (uintptr_t)u | (uintptr_t)scratch) % 16 == 0,
             "%s: operands must be 16-byte aligned", who);
    KA_CHECK(state_stride >= (long)H * d * d + (x ? dim : 0) && stride >= (long)H * d && out_stride >= (long)H * d, "%s: rows are shorter than their heads", who);
    const long n_chunks = n / DC_CHUNK + n_rows;
    KA_CHECK(H <= 65535 && n_rows <= 65535 && n_chunks <= 65535 && scratch != nullptr, "%s: too many heads, rows or chunks", who);
    if (n == 0 || n_rows == 0) return 0;
    const bool finishes = d <= 64;
    const DecayedChunkArgs a{(const bf16_t*)r, (const bf16_t*)k, (const bf16_t*)v, (const bf16_t*)gate, stride, pre, u, gain, state, state_stride, x, dim, cu_q,
                             row_slot, finishes ? (bf16_t*)out : nullptr, out_stride, raw, scratch, scratch + n_chunks * H * d * d, n_rows, H, d, eps};
    if (d <= 64) decayed_chunks_launch<16>(a, n, (int)n_chunks, stream);
    else if (d <= 128) decayed_chunks_launch<32>(a, n, (int)n_chunks, stream);
    else decayed_chunks_launch<64>(a, n, (int)n_chunks, stream);
    KA_LAUNCH_CHECK();
    return finishes ? 0 : 1;
}
