// Instantiations of the ring tiles.
#include "fp8_gemm_tile_ring.h"
#include "tg_host.h"

namespace tg {

hipError_t run_tile_ring(int bm, int bn, bool split, const GemmParams& p, int gx, int gy, hipStream_t s) {
#define TG_CASE(BM, BN, STAGES) \
    if (bm == BM && bn == BN) return launch_tile_ring<BM, BN, STAGES, false>(split, p, gx, gy, s);
    TG_CASE(64, 128, 5)
    TG_CASE(96, 128, 4)
    TG_CASE(128, 128, 4)
    TG_CASE(160, 128, 4)
    TG_CASE(160, 192, 3)
    TG_CASE(192, 192, 3)
#undef TG_CASE
    return hipErrorInvalidConfiguration;
}

hipError_t run_tile_ring_block(int bm, bool split, const GemmParams& p, int gx, int gy, hipStream_t s) {
    if (bm == 64) return launch_tile_ring<64, 128, 5, true>(split, p, gx, gy, s);
    if (bm == 96) return launch_tile_ring<96, 128, 4, true>(split, p, gx, gy, s);
    if (bm == 128) return launch_tile_ring<128, 128, 4, true>(split, p, gx, gy, s);
    if (bm == 160) return launch_tile_ring<160, 128, 4, true>(split, p, gx, gy, s);
    if (bm == 192) return launch_tile_ring<192, 128, 3, true>(split, p, gx, gy, s);
    return hipErrorInvalidConfiguration;
}

}  // namespace tg
