// Instantiations of the ring tiles.
#include "fp8_gemm_tile_ring.h"
#include "tg_host.h"

namespace tg {

hipError_t run_tile_ring(int bm, int bn, bool split, const GemmParams& p, int gx, int gy, hipStream_t s) {
#define TG_CASE(BM, BN, STAGES) \
    if (bm == BM && bn == BN) return launch_tile_ring<BM, BN, STAGES, false>(split, p, gx, gy, s);
    TG_CASE(64, 32, 12)
    TG_CASE(32, 64, 12)
    TG_CASE(64, 64, 9)
    TG_CASE(32, 128, 7)
    TG_CASE(64, 128, 5)
    TG_CASE(96, 128, 4)
    TG_CASE(128, 128, 4)
    TG_CASE(160, 128, 4)
    TG_CASE(160, 192, 3)
    TG_CASE(192, 192, 3)
    TG_CASE(256, 128, 3)
#undef TG_CASE
    return hipErrorInvalidConfiguration;
}

hipError_t run_tile_ring_kn(int bm, int bn, bool split, const GemmParams& p, int gx, int gy, hipStream_t s) {
    // 16-byte pieces of whole K rows, 32-bit offsets
    if (p.N < 16 || p.N % 16 != 0 || p.K % kKBlock != 0 || (int64_t)p.N * p.K >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
#define TG_CASE(BM, BN, STAGES) \
    if (bm == BM && bn == BN) return launch_tile_ring<BM, BN, STAGES, false, true>(split, p, gx, gy, s);
    TG_CASE(32, 64, 12)
    TG_CASE(64, 64, 9)
    TG_CASE(32, 128, 7)
    TG_CASE(64, 128, 5)
    TG_CASE(96, 128, 4)
    TG_CASE(128, 128, 4)
    TG_CASE(160, 128, 4)
    TG_CASE(256, 128, 3)
#undef TG_CASE
    return hipErrorInvalidConfiguration;
}

hipError_t run_tile_ring_block(int bm, int bn, bool split, const GemmParams& p, int gx, int gy, hipStream_t s) {
    if (bm == 32 && bn == 64) return launch_tile_ring<32, 64, 8, true>(split, p, gx, gy, s);
    if (bm == 64 && bn == 64) return launch_tile_ring<64, 64, 7, true>(split, p, gx, gy, s);
    if (bn != 128) return hipErrorInvalidConfiguration;
    if (bm == 32) return launch_tile_ring<32, 128, 7, true>(split, p, gx, gy, s);
    if (bm == 64) return launch_tile_ring<64, 128, 5, true>(split, p, gx, gy, s);
    if (bm == 96) return launch_tile_ring<96, 128, 4, true>(split, p, gx, gy, s);
    if (bm == 128) return launch_tile_ring<128, 128, 4, true>(split, p, gx, gy, s);
    if (bm == 160) return launch_tile_ring<160, 128, 4, true>(split, p, gx, gy, s);
    if (bm == 192) return launch_tile_ring<192, 128, 3, true>(split, p, gx, gy, s);
    return hipErrorInvalidConfiguration;
}

}  // namespace tg
