// Instantiations of the per-tensor ring tiles.
#include "fp8_gemm_tile_ring.h"
#include "tg_host.h"

namespace tg {

hipError_t run_tile_ring(int bm, int bn, bool split, const GemmParams& p, int gx, int gy, hipStream_t s) {
#define TG_CASE(BM, BN, STAGES) \
    if (bm == BM && bn == BN) return launch_tile_ring<BM, BN, STAGES>(split, p, gx, gy, s);
    TG_CASE(96, 128, 4)
    TG_CASE(128, 128, 4)
    TG_CASE(160, 128, 4)
    TG_CASE(160, 192, 3)
    TG_CASE(192, 192, 3)
#undef TG_CASE
    return hipErrorInvalidConfiguration;
}

}  // namespace tg
