// Launches of linears of at most eight rows whose workgroups hold their whole share of the weights (ka_share.h).
#include "ka_share.h"

// Blocks asked for ahead: a lane has 256 registers, with the waves for a norm beside it 168.
constexpr int sh_ahead(int U, int NS, bool ln) { return sh_min(NS * U, ln ? (U <= 4 ? 28 : 24) : 32); }

template <int U, bool LN>
static int launch_strips(int NS, const SkinnyArgs& args, int strips, hipStream_t stream) {
    switch (NS) {
        case 1: return launch_share<U, 1, sh_ahead(U, 1, LN), LN, false, false>(args, strips, stream);
        case 2: return launch_share<U, 2, sh_ahead(U, 2, LN), LN, false, false>(args, strips, stream);
        case 3: return launch_share<U, 3, sh_ahead(U, 3, LN), LN, false, false>(args, strips, stream);
        case 4: return launch_share<U, 4, sh_ahead(U, 4, LN), LN, false, false>(args, strips, stream);
        case 5: return launch_share<U, 5, sh_ahead(U, 5, LN), LN, false, false>(args, strips, stream);
        case 6: return launch_share<U, 6, sh_ahead(U, 6, LN), LN, false, false>(args, strips, stream);
        case 7: return launch_share<U, 7, sh_ahead(U, 7, LN), LN, false, false>(args, strips, stream);
        case 8: return launch_share<U, 8, sh_ahead(U, 8, LN), LN, false, false>(args, strips, stream);
        case 9: return launch_share<U, 9, sh_ahead(U, 9, LN), LN, false, false>(args, strips, stream);
    }
    return 1;
}

int ka_skinny_share_long(const SkinnyArgs& args, int strips, int per, bool crowded, hipStream_t stream);       // gemv_share_long_bf16.hip

// Which linears: those whose workgroups hold all of their strips at once, up to nine a CU (a layer's; the persistent kernel, two workgroups a CU, is ahead
// where they walk over more: 51,200 outputs 35 us either way), and one strip of a long K where the split kernel took it. Us, before -> here, weights
// from HBM: norm and 6,144 outputs of 2,048, one row 8.4 -> 7.3; norm and 14,336 14.9 -> 12.8, eight rows 16.6 -> 13.2; norm and 17,920 of 2,560, eight
// rows 22.0 -> 19.2; 9,280 of 2,048, one row 10.5 -> 9.3, eight 11.2 -> 9.0; 5,632 of 2,048 gated, eight 8.7 -> 7.0; 4,096 of 4,096, eight 9.7 -> 8.7;
// 2,048 of 2,048 4.2 -> 4.1; 2,048 of 2,048 + 8,192, one row 9.8 -> 9.3, eight 12.5 -> 12.1; 2,560 of 2,560 + 10,240, four rows 24.0 -> 21.7.
// What bounds them now: requests, which the memory takes at 5 to 5.5 TB/s once all CUs ask, and 2 us of a launch's start and end.
// split_waves: the waves over K that the split kernel would take, where that one has the call otherwise (else 0). With four of them there the call stays there:
// nine to sixteen rows have four as well, and eight here would be another order of a row's sums. (Where it would take sixteen, nine to sixteen rows have the eight of here; error
// of the fp32 sums against 64 bits, 256 to 1,488 outputs of 3,072 to 10,752: 1.147e-7 of their norm with eight waves, 1.131e-7 with sixteen.)
// 1: not covered, nothing was run.
int ka_skinny_share(const SkinnyArgs& args, int strips, int kblocks, bool ln, int split_waves, hipStream_t stream) {
    const bool pair = args.A[1] != nullptr;
    if (split_waves == 4) return 1;
    const int cus = ka_compute_units(), per = ka_cdiv(kblocks, SP_WAVES), NS = ka_cdiv(strips, cus);
    if (args.M > SH_ROWS || !persistent_bias_ok(args.a) || !persistent_bias_ok(args.b)) return 1;
    for (long ld : {args.a.ldw, args.b.ldw, args.ldw2, args.lda[0], args.lda[1]})
        if (ld >= 1L << 26) return 1;          // (offsets of eight rows in 32 bits)
    if (args.bias2 && (args.a.N % 4 || (uintptr_t)args.bias2 % 16)) return 1;
    if (args.a.accumulate && args.b.W) return 1;        // (the body adds a's old values, whichever target a strip has)
    if (args.a.accumulate && (args.a.N % 4 || args.a.ldo % 4 || (uintptr_t)args.a.out % 16)) return 1;
    if (ln) {
        // (rows of up to 1,024: the persistent kernel. In the form for two blocks the compiler keeps the rows in memory, 7.5 against 5.2 us)
        if (per <= 2) return 1;
        if (per <= 4) return launch_strips<4, true>(NS, args, strips, stream);
        if (per <= 5) return launch_strips<5, true>(NS, args, strips, stream);
        return 1;
    }
    if (pair || per > 8) return NS <= 2 && !args.b.W ? ka_skinny_share_long(args, strips, per, NS > 1, stream) : 1;
    if (args.a.accumulate && NS > 1) return 1;
    switch (per) {
        case 1: return launch_strips<1, false>(NS, args, strips, stream);
        case 2: return launch_strips<2, false>(NS, args, strips, stream);
        case 3: return launch_strips<3, false>(NS, args, strips, stream);
        case 4: return launch_strips<4, false>(NS, args, strips, stream);
        case 5: return launch_strips<5, false>(NS, args, strips, stream);
        case 6: return NS <= 8 ? launch_strips<6, false>(NS, args, strips, stream) : 1;
        case 7: return NS <= 7 ? launch_strips<7, false>(NS, args, strips, stream) : 1;
        case 8: return NS <= 6 ? launch_strips<8, false>(NS, args, strips, stream) : 1;
    }
    return 1;
}
