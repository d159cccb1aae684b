// Instantiations of the persistent grouped ring tiles.
#include "fp8_gemm_grouped_ring.h"
#include "tg_host.h"

namespace tg {

hipError_t run_grouped_ring(int bm, int cols, int group, GemmParams p, hipStream_t s) {
    const int bn = cols == 192 || cols == 0 ? 256 : cols;
    p.tile_cols = cols;
    if (p.kblocks < grouped_ring_steps(bn) || p.K % kKBlock != 0 || !p.As || !p.Bs || (group == GROUP_RAGGED && p.E > kGroupedRingExperts) ||
        (group != GROUP_RAGGED && p.block_m % bm != 0)) return hipErrorInvalidValue;
    const int grid = compute_units() / 8 * 8;
    if (grid <= 0) return hipErrorInvalidDevice;
#define TG_CASE(BM, BN, STAGES, NC)                                                                                  \
    if (bm == BM && bn == BN) {                                                                                   \
        if (group == GROUP_RAGGED) return launch_grouped_ring<BM, BN, STAGES, NC, GROUP_RAGGED>(p, grid, s);          \
        if (group == GROUP_GATHER) return launch_grouped_ring<BM, BN, STAGES, NC, GROUP_GATHER>(p, grid, s);          \
    }
    if (bm == 32 && bn == 128 && group == GROUP_RAGGED) return launch_grouped_ring<32, 128, 6, 4, GROUP_RAGGED>(p, grid, s);
    TG_CASE(64, 128, 6, 4)
    TG_CASE(64, 256, 3, 8)
    TG_CASE(128, 256, 3, 8)
#undef TG_CASE
    if (group == GROUP_GATHER_ACT && bn == 256) {
        if (bm == 64) return launch_grouped_ring<64, 256, 3, 8, GROUP_GATHER_ACT>(p, grid, s);
        if (bm == 128) return launch_grouped_ring<128, 256, 3, 8, GROUP_GATHER_ACT>(p, grid, s);
    }
    return hipErrorInvalidConfiguration;
}

}  // namespace tg
