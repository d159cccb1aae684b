// Instantiations and launchers of the decoding MoE layer (fp8_moe_decode.h).
#include "fp8_moe_decode.h"

#include <algorithm>
#include <cmath>

namespace tg {

namespace {

// Fills in row_cap and wscale_cap; false when the layer is not one for this kernel.
//
// An expert with more than row_cap rows is streamed more than once, so the rows that the fullest expert is likely to get
// decide: with m = slots / E rows on average and even routing about m + 3 sqrt(m).  The line lies where a batch half of which
// routes alike (padding rows, say) takes as long as on the row-tiled form.  Whole layer, 64 experts of (2048, 1408), top 6,
// against that form (in brackets), us:
//   tokens (m)    even routing   half alike     one expert in every token   all alike
//   40 (3.8)       94 (122)       98 (118)      100 (122)                   43 (37)
//   64 (6)         99 (124)      121 (122)      119 (123)                   56 (38)
//   75 (7.0)      101 (125)      127 (124)      117 (125)                   51 (43)     <- the last one taken
//   87 (8.2)      102 (125)      128 (126)      121 (126)                   72 (43)
// and 128 experts of (4096, 1536), top 8: 80 (5) 382 (454), 420 (438), 426 (454), 137 (61); 96 (6) 390 (462), 445 (443), 421
// (458), 175 (63); 130 (8.1) 401 (460), 494 (458), 429 (495), 251 (69).  32 rows held take even routing to 174 tokens (111
// against 127 at 160), but an expert over the line then costs more than the rest saves (143 - 158 against 130 - 136).
constexpr int kDecodeRows = 16;
constexpr float kDecodeLikely = 15.0f;
bool decode_plan(MoeDecodeParams& p, bool up, int tokens) {
    const int cols = up ? 8 : 16, groups = (up ? p.inter : p.N) / cols;
    const int nbs = (groups * cols + 127) / 128 + 1;   // block rows of a segment, at most
    p.wscale_cap = (nbs * (up ? 2 : 1) * p.kblocks + 63) / 64 * 64;
    p.pass_groups = 2 + 40 / p.kblocks;
    int cap = 1;
    while (cap < tokens && cap < kDecodeRows) cap *= 2;
    while (cap > 1) {
        p.row_cap = cap;
        if (MoeDecodeLds::of(p).total <= kLdsBytes) break;
        cap /= 2;
    }
    p.row_cap = cap;
    const float mean = (float)p.slots / (float)p.E, likely = mean + 3.0f * sqrtf(mean);
    return MoeDecodeLds::of(p).total <= kLdsBytes && (tokens <= cap || likely < fminf((float)(cap + 2), kDecodeLikely));
}

template <typename T, bool UP>
hipError_t launch_decode(const MoeDecodeParams& p, hipStream_t s) {
    // one workgroup per compute unit: each takes an equal share of the weights (at most 256, for the kernel's 32-bit shares)
    hipLaunchKernelGGL((moe_decode_kernel<T, UP>), dim3((unsigned)std::min(compute_units(), 256)), dim3(64 * (kDecodeWaves + kDecodeQuantWaves)),
                       (size_t)MoeDecodeLds::of(p).total, s, p);
    return hipGetLastError();
}

template <typename T>
hipError_t dispatch_decode(const MoeDecodeParams& p, bool up, hipStream_t s) {
    return up ? launch_decode<T, true>(p, s) : launch_decode<T, false>(p, s);
}

bool decode_shape_ok(const MoeDecodeParams& p, bool up) {
    return p.K > 0 && p.K % kKBlock == 0 && p.slots > 0 && p.slots <= kMoeDecodeSlots && p.E >= 1 && p.E <= 512 &&
           (up ? p.inter > 0 && p.inter % 128 == 0 && p.N == 2 * p.inter : p.N > 0 && p.N % 128 == 0) &&
           (int64_t)p.N * p.K < ((int64_t)1 << 31) && (int64_t)p.E * p.N < ((int64_t)1 << 23);   // (units in 32 bits)
}

}  // namespace

bool moe_decode_fits(MoeDecodeParams p, bool up, int tokens) { return decode_shape_ok(p, up) && decode_plan(p, up, tokens); }

int64_t moe_decode_lds_bytes(MoeDecodeParams p, bool up, int tokens) {
    return decode_shape_ok(p, up) && decode_plan(p, up, tokens) ? MoeDecodeLds::of(p).total : 0;
}

int64_t moe_decode_sum_lds_bytes(const MoeDecodeParams& p, int tokens) { return moe_decode_sum_fits(p, tokens) ? moe_decode_sum_lds(p.top_k, p.K) : 0; }

hipError_t run_moe_decode(MoeDecodeParams p, bool up, bool is_bf16, int tokens, hipStream_t s) {
    if (!decode_shape_ok(p, up) || !decode_plan(p, up, tokens)) return hipErrorInvalidConfiguration;
    return is_bf16 ? dispatch_decode<__bf16>(p, up, s) : dispatch_decode<_Float16>(p, up, s);
}

// One launch instead of two pays while hardly any expert serves two tokens: 2 tokens of 6 slots over 64 experts 11.3 us
// against 12.5 + 3.0, 4 tokens 21.7 against 17.0 + 4.0 (each token reads its experts' weights).
bool moe_decode_sum_fits(const MoeDecodeParams& p, int tokens) {
    return (tokens == 1 || (p.slots <= 16 && p.slots * 4 <= p.E)) && p.top_k >= 1 && p.top_k <= 8 && p.K % kKBlock == 0 && p.K <= 64 * kKBlock &&
           p.N % 128 == 0 && (int64_t)p.N * p.K < ((int64_t)1 << 31) && moe_decode_sum_lds(p.top_k, p.K) <= kLdsBytes;
}

hipError_t run_moe_decode_sum(const MoeDecodeParams& p, bool is_bf16, int tokens, hipStream_t s) {
    if (!moe_decode_sum_fits(p, tokens) || tokens <= 0 || p.slots != tokens * p.top_k) return hipErrorInvalidConfiguration;
    const dim3 grid((unsigned)(p.N / kDecodeSumRows), (unsigned)tokens), block(64u * p.top_k);
    const size_t lds = (size_t)moe_decode_sum_lds(p.top_k, p.K);
    if (is_bf16) hipLaunchKernelGGL(moe_decode_sum_kernel<__bf16>, grid, block, lds, s, p);
    else hipLaunchKernelGGL(moe_decode_sum_kernel<_Float16>, grid, block, lds, s, p);
    return hipGetLastError();
}

}  // namespace tg
