// Linears of some hundred rows by four waves a tile (ka_quad_tiles.h), outputs in bf16.
#include "ka_quad_tiles.h"

int ka_quad_bf16(const KqLinears& p, int code, hipStream_t stream) {
#define KQ_LAUNCH(...) launch_quad<__VA_ARGS__, false>(p, stream)
    KQ_TILES(KQ_LAUNCH)
#undef KQ_LAUNCH
    KA_CHECK(false, "linears by tiles: unknown tile %d", code);
}
