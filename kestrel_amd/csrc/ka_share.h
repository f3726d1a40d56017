// Linears of at most eight rows whose workgroups hold their whole share of the weights: all of it is asked for at once.
//
// The products are those of ka_skinny.h: strips of 8 weight rows, eight waves that take the k-blocks of a strip in turn, the waves' sums added in their
// order, rows with a norm in front summed by sk_row_statistics. So a row has the bits that the persistent kernel gives it, and those of the split kernel where
// that one has eight waves over K. What differs is that nothing of a workgroup's way depends on a number known at
// run time only: strips and blocks are unrolled, so that every load can be issued where it stands and waited for by count. A loop over
// strips cannot have that here: what a round has asked for moves to other registers for the next one, and the compiler waits for all of it
// to do so; a value chosen as soon as it is loaded (no bias: zero) waits for it there too. With few strips a workgroup, which is what a
// layer's linears have, such waits are all there is of a loop.
// The strips' sums meet in LDS behind one barrier at the end instead of one a strip.
#pragma once
#include "ka_skinny.h"

constexpr int SH_ROWS = 8;                        // most rows
__host__ __device__ constexpr int sh_threads(bool ln) { return (SP_WAVES + (ln ? 4 : 0)) * KA_WAVE; }
// LDS: the strips' sums [NS][SP_WAVES][KA_WAVE]; with a norm, in their place before there are any, the rows in fp32, [M][K], and behind them
// three counts of waves (16 bytes), each row's mean and reciprocal deviation, and the normalised rows, [M][K + SK_PAD] in bf16.
constexpr int SH_NORM = 4;                        // waves that normalise, beside the eight that multiply
__host__ __device__ constexpr int sh_min(int a, int b) { return a < b ? a : b; }
__host__ __device__ constexpr int sh_first_bytes(int NS, bool ln, int M, int K) {
    const int sums = NS * SP_WAVES * KA_WAVE * 16, rows = ln ? M * K * 4 : 0;
    return sums > rows ? sums : rows;
}
constexpr int SH_STATS_BYTES = 16 + SH_ROWS * 8;

// Workgroup `block` of `grid`: strips block, block + grid, ... (NS of them; past the last strip it reads the last one again and stores nothing).
// U: k-blocks of a wave. AHEAD: blocks asked for before the first is multiplied (all NS * U, or as many as registers hold).
// PAIR: two segments of K, one strip.
// X_BESIDE: the activations come block by block beside the weights (one strip of a long K), else all before them.
// LN: the rows are fp32 and normalised here, by waves of their own: a wave is held where it asks for more than the memory takes, so one that first asked
// for its weights would begin with the norm when most of them have come (stamps, 14,336 outputs of 2,048, 8 rows: rows normalised 10.6 us into
// 12.7), and one that asks for them behind it leaves the memory idle. These waves share the channels, not the rows: scale and shift are then read once a
// workgroup (with a row a wave, once a row: 16 K bytes of every 16 K + 8 M K at eight rows). The sums of a row have the order of sk_row_statistics, as in every
// kernel with a norm in front, so a row's numbers do not depend on the rows beside it: the channels that the waves have brought meet in LDS, and a wave
// takes the sums of whole rows from there (sums by the waves' own channels: 0.1 to 0.3 us less up to 2,048 wide, up to 1.2 less at 2,560 and eight rows of
// few outputs, nothing from 8,192 outputs on). A wave that multiplies waits for the rows and not for the other waves: at a barrier it would wait for the
// last one's requests.
template <int U, int NS, int AHEAD, bool LN, bool PAIR, bool X_BESIDE>
__device__ __forceinline__ void skinny_share_body(const SkinnyArgs& p, const int total_strips, const int block, const int grid, unsigned char* lds) {
    static_assert(AHEAD <= NS * U && AHEAD > 0, "blocks ahead");
    static_assert(!X_BESIDE || (NS == 1 && !LN), "activations beside the weights: one strip, no norm");
    static_assert(!PAIR || (NS == 1 && !LN), "two segments: one strip, no norm");
    constexpr bool ACCUMULATES = NS == 1 && !LN;
    constexpr int WAVES = sh_threads(LN) / KA_WAVE, ADDENDS = (NS + WAVES - 1) / WAVES;
    floatx4* const red = reinterpret_cast<floatx4*>(lds);
    float* const raw = reinterpret_cast<float*>(lds);                                  // [M][K]
    unsigned char* const behind = lds + sh_first_bytes(NS, LN, p.M, p.K[0]);
    int* const raw_done = reinterpret_cast<int*>(behind);                              // waves whose part of the fp32 rows is in LDS
    int* const stats_done = raw_done + 1;                                              // waves whose rows' statistics are
    int* const rows_done = raw_done + 2;                                               // waves whose part of the normalised rows is
    float2* const stats = reinterpret_cast<float2*>(raw_done + 4);                     // [SH_ROWS]
    bf16_t* const xs = reinterpret_cast<bf16_t*>(behind + SH_STATS_BYTES);
    auto await = [](const int* count) {
        while (__hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < SH_NORM) __builtin_amdgcn_s_sleep(1);
        asm volatile("" ::: "memory");
    };
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KA_WAVE), lane = threadIdx.x % KA_WAVE;
    const int r = lane % 16, g = lane / 16, m = r % 8;
    const int koff = (r / 8) * 32 + g * 8, M = p.M;
    const int K0 = sk_pinned(p.K[0]), K1 = sk_pinned(p.K[1]);
    const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
    const floatx4 zero4 = {0.f, 0.f, 0.f, 0.f};
    const bf16_t* const Wa = sk_pinned(p.a.W);
    const bf16_t* const Wb = sk_pinned(PAIR ? p.W2 : p.b.W);
    const long ldwa = sk_pinned(p.a.ldw), ldwb = sk_pinned(PAIR ? p.ldw2 : p.b.ldw);
    const int Na = sk_pinned(p.a.N), Nb = sk_pinned(p.b.N), strips_a = sk_pinned(p.strips_a);
    const float* const biasa = sk_pinned(p.a.bias);
    const float* const biasb = sk_pinned(PAIR ? p.bias2 : p.b.bias);
    const int accumulate = sk_pinned(p.a.accumulate);
    const int nb0 = (K0 + SK_KBLOCK - 1) / SK_KBLOCK, nb = PAIR ? nb0 + (K1 + SK_KBLOCK - 1) / SK_KBLOCK : nb0;

    auto strip_of = [&](int s) { return min(block + s * grid, total_strips - 1); };
    // what the finishing lanes add (biases, the output's old value): asked for first, chosen at the end
    floatx4 addend[ADDENDS][2], old;
    sk_static_for<ADDENDS>([&](auto i) {
        const int strip = strip_of(WAVES - 1 - wave + i.value * WAVES);
        const bool second = !PAIR && strip >= strips_a;
        const int N = second ? Nb : Na, n = min((second ? strip - strips_a : strip) * SK_STRIP + (g & 1) * 4, N - 4);
        const float* const bias = second ? biasb : biasa;
        addend[i.value][0] = *(const SK_GLOBAL floatx4*)(bias ? bias + n : reinterpret_cast<const float*>(Wa));
        if constexpr (PAIR) addend[i.value][1] = *(const SK_GLOBAL floatx4*)(biasb ? biasb + n : reinterpret_cast<const float*>(Wa));
        if constexpr (ACCUMULATES)
            old = *(const SK_GLOBAL floatx4*)(accumulate ? reinterpret_cast<const float*>(p.a.out) + (size_t)min(m, M - 1) * p.a.ldo + n : reinterpret_cast<const float*>(Wa));
    });

    // block u of this wave: its segment, first k, and whether there is one (past the end: the last one again, times zeros)
    struct Place { bool live, seg; int k, K; };
    auto place = [&](int u) {
        const int b = wave + u * SP_WAVES, bc = min(b, nb - 1);
        Place at;
        at.live = b < nb;
        at.seg = PAIR && bc >= nb0;
        at.k = (at.seg ? bc - nb0 : bc) * SK_KBLOCK;
        at.K = at.seg ? K1 : K0;
        return at;
    };
    auto covered = [&](const Place& at) { return at.live && at.k + koff < at.K; };
    bf16x8 w[AHEAD], x[X_BESIDE ? AHEAD : U];
    const bf16_t* const A0 = sk_pinned(p.A[0]);
    const bf16_t* const A1 = sk_pinned(p.A[1]);
    const int lda0 = (int)sk_pinned(p.lda[0]), lda1 = (int)sk_pinned(p.lda[1]);
    // (bytes from the operand's or the strip's first row fit in 32 bits: the host's check)
    auto load_x = [&](int u) {
        const Place at = place(u);
        const unsigned off = (unsigned)(min(m, M - 1) * (at.seg ? lda1 : lda0) + min(at.k + koff, at.K - 8)) * 2u;
        return *(const SK_GLOBAL bf16x8*)((const SK_GLOBAL char*)(at.seg ? A1 : A0) + off);
    };
    auto kept_x = [&](int u, bf16x8 v) { return m < M && covered(place(u)) ? v : zero; };
    auto issue = [&](auto i) {
        constexpr int s = i.value / U, u = i.value % U, slot = i.value % AHEAD;
        const int strip = strip_of(s);
        const Place at = place(u);
        const bool second = !PAIR && strip >= strips_a;
        const int n0 = (second ? strip - strips_a : strip) * SK_STRIP;
        const bool other = PAIR ? at.seg : second;
        const long ldw = other ? ldwb : ldwa;
        const int last = (second ? Nb : Na) - 1 - n0;
        const SK_GLOBAL char* const base = (const SK_GLOBAL char*)((other ? Wb : Wa) + (size_t)n0 * ldw);
        const unsigned off = ((unsigned)min(r % 8, last) * (unsigned)ldw + (unsigned)min(at.k + koff, at.K - 8)) * 2u;
        w[slot] = __builtin_nontemporal_load((const SK_GLOBAL bf16x8*)(base + off));
        if constexpr (X_BESIDE) x[slot] = load_x(u);
    };
    if (LN && wave >= SP_WAVES) {
        if constexpr (LN) {
            constexpr int XJ = (2 * U + SH_NORM - 1) / SH_NORM;       // pieces of four channels a lane and row
            constexpr bool KEPT = XJ <= 2;                             // (else read once more: 24 pieces beside a whole row spill)
            const int part = wave - SP_WAVES;
            auto channel = [&](int j) { return ((j * SH_NORM + part) * KA_WAVE + lane) * 4; };
            const float* const shift = p.ln_beta ? p.ln_beta : p.ln_gamma;        // (no shift: the scale once more, left out below)
            floatx4 xf[SH_ROWS][XJ], gamma[XJ], beta[XJ];
#pragma unroll
            for (int of = 0; of < SH_ROWS; ++of)
                if (of < M) {
#pragma unroll
                    for (int j = 0; j < XJ; ++j) xf[of][j] = *(const SK_GLOBAL floatx4*)(p.ln_x + (size_t)of * K0 + min(channel(j), K0 - 4));
                }
#pragma unroll
            for (int j = 0; j < XJ; ++j) {
                gamma[j] = *(const SK_GLOBAL floatx4*)(p.ln_gamma + min(channel(j), K0 - 4));
                beta[j] = *(const SK_GLOBAL floatx4*)(shift + min(channel(j), K0 - 4));
            }
            if (part == 0 && lane == 0) *rows_done = *raw_done = *stats_done = 0;
            sk_lds_barrier();
            auto report = [&](int* count) {
                __builtin_amdgcn_s_waitcnt(0xc07f);                    // (what this wave wrote is in LDS)
                asm volatile("" ::: "memory");
                if (lane == 0) __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            };
#pragma unroll
            for (int of = 0; of < SH_ROWS; ++of)
                if (of < M) {
#pragma unroll
                    for (int j = 0; j < XJ; ++j)
                        if (channel(j) < K0) *reinterpret_cast<floatx4*>(raw + of * K0 + channel(j)) = xf[of][j];
                }
            report(raw_done);
            await(raw_done);
#pragma unroll 1
            for (int of = part; of < M; of += SH_NORM) {
                floatx4 row[2 * U];
#pragma unroll
                for (int j = 0; j < 2 * U; ++j) row[j] = *reinterpret_cast<const floatx4*>(raw + of * K0 + min((j * KA_WAVE + lane) * 4, K0 - 4));
                const float2 mean_rstd = sk_row_statistics(p, K0, lane, row);
                if (lane == 0) stats[of] = mean_rstd;
            }
            report(stats_done);
            await(stats_done);
            const bool shifted = p.ln_beta != nullptr, stored = p.ln_store != nullptr && block == 0;
#pragma unroll
            for (int j = 0; j < XJ; ++j)
                if (!shifted) beta[j] = zero4;
#pragma unroll
            for (int of = 0; of < SH_ROWS; ++of)
                if (of < M) {
                    const float mean = stats[of].x, rstd = stats[of].y;
#pragma unroll
                    for (int j = 0; j < XJ; ++j) {
                        if constexpr (!KEPT) xf[of][j] = *reinterpret_cast<const floatx4*>(raw + of * K0 + min(channel(j), K0 - 4));
                        bf16x4 y;
#pragma unroll
                        for (int i = 0; i < 4; ++i) y[i] = (bf16_t)((xf[of][j][i] - mean) * rstd * gamma[j][i] + beta[j][i]);
                        if (channel(j) < K0) {
                            *reinterpret_cast<bf16x4*>(xs + of * (K0 + SK_PAD) + channel(j)) = y;
                            // (every workgroup normalises the same rows; one of them leaves them for later launches)
                            if (stored) *reinterpret_cast<bf16x4*>(p.ln_store + (size_t)of * p.ln_store_ld + channel(j)) = y;
                        }
                    }
                }
            report(rows_done);
        }
    } else {
        if constexpr (!LN && !X_BESIDE) sk_static_for<U>([&](auto u) { x[u.value] = load_x(u.value); });
        __builtin_amdgcn_sched_barrier(0);
        sk_static_for<AHEAD>([&](auto i) {
            issue(i);
            if constexpr (LN && i.value == sh_min(2, AHEAD) - 1) {
                __builtin_amdgcn_sched_barrier(0);
                sk_lds_barrier();                    // (the counts are set)
                __builtin_amdgcn_sched_barrier(0);
            }
        });
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (LN) {
            await(rows_done);
            sk_static_for<U>([&](auto u) {
                const Place at = place(u.value);
                x[u.value] = *reinterpret_cast<const bf16x8*>(xs + min(m, M - 1) * (K0 + SK_PAD) + min(at.k + koff, at.K - 8));
            });
        }
        if constexpr (!X_BESIDE) sk_static_for<U>([&](auto u) { x[u.value] = kept_x(u.value, x[u.value]); });
        floatx4 sum = zero4;
        sk_static_for<NS * U>([&](auto i) {
            constexpr int s = i.value / U, u = i.value % U, slot = i.value % AHEAD;
            const bf16x8 xv = X_BESIDE ? kept_x(u, x[slot]) : x[X_BESIDE ? 0 : u];
            sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[slot], xv, u == 0 ? zero4 : sum, 0, 0, 0);
            if constexpr (i.value + AHEAD < NS * U) issue(std::integral_constant<int, i.value + AHEAD>{});
            if constexpr (u == U - 1) red[(s * SP_WAVES + wave) * KA_WAVE + lane] = sum;
        });
    }
    sk_lds_barrier();
    // strip s is finished by the last wave but s (with a norm: by the waves that have least to do)
    if (lane >= 32 || r >= 8) return;
    sk_static_for<ADDENDS>([&](auto i) {
        const int s = WAVES - 1 - wave + i.value * WAVES, strip = block + s * grid;
        if (s >= NS || strip >= total_strips) return;
        const bool second = !PAIR && strip >= strips_a;
        const int n0 = (second ? strip - strips_a : strip) * SK_STRIP;
        floatx4 add[1] = {zero4};
        if (second ? biasb != nullptr : biasa != nullptr) add[0] = addend[i.value][0];
        if constexpr (PAIR) {
            if (biasb != nullptr) add[0] += addend[i.value][1];
        }
        if constexpr (ACCUMULATES) {
            if (accumulate) add[0] += old;
        }
        sk_finish<1, true, SP_WAVES>(reinterpret_cast<const floatx4(*)[1][KA_WAVE]>(red + s * SP_WAVES * KA_WAVE), add, second ? p.b : p.a, n0, M, lane,
                                     [](int) { return true; });
    });
}

template <int U, int NS, int AHEAD, bool LN, bool PAIR, bool X_BESIDE>
__global__ void __launch_bounds__(sh_threads(LN))
skinny_share_kernel(SkinnyArgs p, int strips) {
    extern __shared__ __attribute__((aligned(16))) unsigned char sh_lds[];
    skinny_share_body<U, NS, AHEAD, LN, PAIR, X_BESIDE>(p, strips, blockIdx.x, gridDim.x, sh_lds);
}

template <int U, int NS, int AHEAD, bool LN, bool PAIR, bool X_BESIDE>
static int launch_share(const SkinnyArgs& args, int strips, hipStream_t stream) {
    auto kernel = skinny_share_kernel<U, NS, AHEAD, LN, PAIR, X_BESIDE>;
    const int lds = sh_first_bytes(NS, LN, args.M, args.K[0]) + (LN ? SH_STATS_BYTES + args.M * (args.K[0] + SK_PAD) * (int)sizeof(bf16_t) : 0);
    static int reserved = 64 * 1024;
    if (lds > reserved) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        KA_CHECK(e == hipSuccess, "linear of few rows: cannot reserve %d bytes of LDS: %s", lds, hipGetErrorString(e));
        reserved = lds;
    }
    hipLaunchKernelGGL(kernel, dim3(ka_cdiv(strips, NS)), dim3(sh_threads(LN)), lds, stream, args, strips);
    KA_LAUNCH_CHECK();
    return 0;
}

