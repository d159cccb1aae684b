// Instantiations of the ring tiles for weights that one launch reads once.
#include "fp8_gemm_tile_ring.h"
#include "tg_host.h"

namespace tg {

hipError_t run_tile_ring_once(bool block_scaled, int bm, int bn, const GemmParams& p, int gx, hipStream_t s) {
#define TG_CASE(BM, BN, STAGES, BLOCKSCALE) \
    if (bm == BM && bn == BN && block_scaled == BLOCKSCALE) return launch_tile_ring_once<BM, BN, STAGES, BLOCKSCALE>(p, gx, s);
    TG_CASE(32, 64, 12, false)
    TG_CASE(64, 64, 9, false)
    TG_CASE(32, 128, 7, false)
    TG_CASE(64, 128, 5, false)
    TG_CASE(96, 128, 4, false)
    TG_CASE(128, 128, 4, false)
    TG_CASE(160, 128, 4, false)
    TG_CASE(256, 128, 3, false)
    TG_CASE(32, 64, 8, true)
    TG_CASE(64, 64, 7, true)
    TG_CASE(32, 128, 7, true)
    TG_CASE(64, 128, 5, true)
    TG_CASE(96, 128, 4, true)
    TG_CASE(128, 128, 4, true)
    TG_CASE(160, 128, 4, true)
#undef TG_CASE
    return hipErrorInvalidConfiguration;
}

}  // namespace tg
