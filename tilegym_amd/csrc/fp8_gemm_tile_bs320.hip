// The 256 x 320 block-scaled tile.
#include "fp8_gemm_tile_bs320.h"

namespace tg {

hipError_t run_bs320(const GemmParams& p, int gx, hipStream_t s) {
    if (!p.As || !p.Bs || p.K != p.kblocks * kKBlock || !bs320_takes(p.M, p.N)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(fp8_gemm_bs320_kernel, dim3(gx, 1, 1), dim3(512, 1, 1), 0, s, p);
    return hipGetLastError();
}

}  // namespace tg
