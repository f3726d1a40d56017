// Launches of linears of at most eight rows of a long K, or of K in two segments, a strip a workgroup (ka_share.h).
#include "ka_share.h"

// One strip a workgroup. More strips than compute units: two workgroups share one, which they can with 128 registers.
template <int U, bool PAIR>
static int launch_one(bool crowded, const SkinnyArgs& args, int strips, hipStream_t stream) {
    if (crowded) return launch_share<U, 1, sh_min(U, 10), false, PAIR, true>(args, strips, stream);
    return launch_share<U, 1, sh_min(U, 20), false, PAIR, true>(args, strips, stream);
}
template <bool PAIR>
static int launch_one_strip(int per, bool crowded, const SkinnyArgs& args, int strips, hipStream_t stream) {
#define SH_ONE(U) case U: return launch_one<U, PAIR>(crowded, args, strips, stream)
    switch (per) {
        SH_ONE(9); SH_ONE(10); SH_ONE(11); SH_ONE(12); SH_ONE(13); SH_ONE(14); SH_ONE(15); SH_ONE(16); SH_ONE(17);
        SH_ONE(18); SH_ONE(19); SH_ONE(20); SH_ONE(21); SH_ONE(22); SH_ONE(23); SH_ONE(24); SH_ONE(25); SH_ONE(26);
    }
#undef SH_ONE
    return 1;
}

// per: k-blocks of a wave, 9 to 26 (two segments: K of both). 1: not covered, nothing was run.
int ka_skinny_share_long(const SkinnyArgs& args, int strips, int per, bool crowded, hipStream_t stream) {
    return args.A[1] ? launch_one_strip<true>(per, crowded, args, strips, stream) : launch_one_strip<false>(per, crowded, args, strips, stream);
}
