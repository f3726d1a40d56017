// Launches of linears of at most eight rows whose workgroups hold their whole share of the weights (ka_share.h).
#include "ka_share.h"

// Blocks asked for ahead: a lane has 256 registers, with the waves for a norm beside it 168.
constexpr int sh_ahead(int U, int NS, bool ln) { return sh_min(NS * U, ln ? (U <= 4 ? 28 : 24) : 32); }

// NS strips a workgroup, one of FIRST to LAST (else 1: not covered, nothing was run).
template <int U, bool LN, int FIRST, int LAST>
static int launch_strips(int NS, const SkinnyArgs& args, int strips, hipStream_t stream) {
    if constexpr (FIRST > LAST) {
        return 1;
    } else {
        if (NS == FIRST) return launch_share<U, FIRST, sh_ahead(U, FIRST, LN), LN, false, false>(args, strips, stream);
        return launch_strips<U, LN, FIRST + 1, LAST>(NS, args, strips, stream);
    }
}

int ka_skinny_share_long(const SkinnyArgs& args, int strips, int per, bool crowded, hipStream_t stream);       // gemv_share_long_bf16.hip

// Which linears: those whose workgroups hold all of their strips at once, up to nine a CU (a layer's; the persistent kernel, two workgroups a CU up to
// K = 2,048 and one beyond, is ahead where they walk over more: 51,200 outputs 35 us either way), and one strip of a long K where the split kernel took it.
// The lines within, by k-blocks a wave (`per`, K in steps of 512), strips a CU (NS) and rows, from both sides measured in turn over 1 to 8 rows, 256 to 18,432
// outputs, K of 64 to 10,752, weights from HBM (times here over times of the other kernel):
//  * with a norm, per 3 to 5: one strip a CU 1.06 to 1.45 (the rows are the longer way then: the persistent kernel's eight waves normalise a row each), two 0.79 to
//    0.96 up to four rows, 0.98 to 1.19 above; three 0.80 to 0.96, at 2,560 and eight rows 1.04; from four on 0.77 to 0.92. Rows of up to 1,024: the persistent
//    kernel (in the form for two blocks the compiler keeps the rows in memory, 7.5 against 5.2 us).
//  * per 1 and 2: one strip a CU 0.95 to 1.04, two 0.87 to 1.06, four at up to four rows 0.99 to 1.06 (where the persistent kernel has two even rounds of two
//    workgroups a CU); else 0.76 to 1.00.
//  * per 3: 0.67 to 0.94 throughout.
//  * per 4: four and eight strips a CU at up to four rows 0.97 to 1.08, as above; else 0.78 to 1.01.
//  * per 5: up to four strips a CU 0.97 to 1.05, five to seven 0.94 to 0.99, eight and nine 0.97 to 1.07.
//  * per 6: up to four rows 0.93 to 1.06 (1.01 on the average at one), eight rows 0.95 to 1.00.
//  * per 7: 0.85 to 0.98 up to seven strips. Beyond, per 7 and 8 do not fit in registers.
//  * per 8: up to three strips a CU 0.89 to 0.99; four to six, one row 0.97 to 1.03, four rows 0.95 to 1.00.
//  * accumulation (one strip a CU), K above 1,024: 0.84 to 1.01.
//  * one strip of a long K, or of two segments (gemv_share_long_bf16.hip): 0.71 to 1.00.
// Us, other kernel -> here: norm and 6,144 outputs of 2,048, one row 8.4 -> 7.5; norm and 14,336 14.2 -> 12.6, eight rows 15.9 -> 13.1; norm and 18,432 of 2,560,
// eight rows 22.0 -> 19.3; 9,280 of 2,048, one row 10.5 -> 9.3, eight 11.2 -> 9.0; 5,632 of 2,048 gated, eight 8.7 -> 7.0; 4,096 of 4,096, eight 9.9 -> 9.3;
// 2,048 of 2,048 + 8,192, one row 10.1 -> 9.9, eight 13.0 -> 12.8; 2,560 of 2,560 + 10,240, four rows 24.0 -> 21.7.
// What bounds them now: requests, which the memory takes at 5 to 5.5 TB/s once all CUs ask, and 2 us of a launch's start and end.
// split_waves: the waves over K that the split kernel would take, where that one has the call otherwise (else 0). With four of them there the call stays there:
// nine to sixteen rows have four as well, and eight here would be another order of a row's sums. (Where it would take sixteen, nine to sixteen rows have the
// eight of here; error of the fp32 sums against 64 bits, 256 to 1,488 outputs of 3,072 to 10,752: 1.147e-7 of their norm with eight waves, 1.131e-7 with
// sixteen.)
// 1: not covered, nothing was run.
int ka_skinny_share(const SkinnyArgs& args, int strips, int kblocks, bool ln, int split_waves, hipStream_t stream) {
    const bool pair = args.A[1] != nullptr;
    if (split_waves == 4) return 1;
    const int cus = ka_compute_units(), per = ka_cdiv(kblocks, SP_WAVES), NS = ka_cdiv(strips, cus), M = args.M;
    if (M > SH_ROWS || !persistent_bias_ok(args.a) || !persistent_bias_ok(args.b)) return 1;
    for (long ld : {args.a.ldw, args.b.ldw, args.ldw2, args.lda[0], args.lda[1]})
        if (ld >= 1L << 26) return 1;          // (offsets of eight rows in 32 bits)
    if (args.bias2 && (args.a.N % 4 || (uintptr_t)args.bias2 % 16)) return 1;
    if (args.a.accumulate && args.b.W) return 1;        // (the body adds a's old values, whichever target a strip has)
    if (args.a.accumulate && (args.a.N % 4 || args.a.ldo % 4 || (uintptr_t)args.a.out % 16)) return 1;
    if (ln) {
        if (M > 4 && NS < (per <= 4 ? 3 : 4)) return 1;
        if (per == 3 || per == 4) return launch_strips<4, true, 2, 9>(NS, args, strips, stream);
        if (per == 5) return launch_strips<5, true, 2, 9>(NS, args, strips, stream);
        return 1;
    }
    if (pair || per > 8) return NS <= 2 && !args.b.W ? ka_skinny_share_long(args, strips, per, NS > 1, stream) : 1;
    if (args.a.accumulate) {
        switch (per) {
            case 3: return launch_strips<3, false, 1, 1>(NS, args, strips, stream);
            case 4: return launch_strips<4, false, 1, 1>(NS, args, strips, stream);
            case 5: return launch_strips<5, false, 1, 1>(NS, args, strips, stream);
            case 6: return launch_strips<6, false, 1, 1>(NS, args, strips, stream);
            case 7: return launch_strips<7, false, 1, 1>(NS, args, strips, stream);
            case 8: return launch_strips<8, false, 1, 1>(NS, args, strips, stream);
        }
        return 1;
    }
    switch (per) {
        case 1: return NS == 4 && M <= 4 ? 1 : launch_strips<1, false, 3, 9>(NS, args, strips, stream);
        case 2: return NS == 4 && M <= 4 ? 1 : launch_strips<2, false, 3, 9>(NS, args, strips, stream);
        case 3: return launch_strips<3, false, 1, 9>(NS, args, strips, stream);
        case 4: return NS % 4 == 0 && M <= 4 ? 1 : launch_strips<4, false, 1, 9>(NS, args, strips, stream);
        case 5: return launch_strips<5, false, 5, 7>(NS, args, strips, stream);
        case 6: return M <= 4 ? 1 : launch_strips<6, false, 1, 8>(NS, args, strips, stream);
        case 7: return launch_strips<7, false, 1, 7>(NS, args, strips, stream);
        case 8: return NS > 3 && M < 4 ? 1 : launch_strips<8, false, 1, 6>(NS, args, strips, stream);
    }
    return 1;
}
