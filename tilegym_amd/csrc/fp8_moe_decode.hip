// Instantiations and launchers of the decoding MoE layer (fp8_moe_decode.h).
#include "fp8_moe_decode.h"

#include <cmath>

namespace tg {

namespace {

// Fills in row_cap and wscale_cap; false when the layer is not one for this kernel.
//
// An expert with more than row_cap rows is streamed more than once, so the rows that the fullest expert is likely to get
// decide: with m = slots / E rows on average and even routing about m + 3 sqrt(m).  Whole layer, (hidden, inter) =
// (2048, 1408), 64 experts, top 6, against the row-tiled form: 1 token 16.2 us (35.0), 16 tokens 84 (112), 64 tokens
// (m = 6) 99 (124); at 96 tokens (m = 9) 131 (125) with 16 rows held, so more rows are held from there on (two tiles of 16).
bool decode_plan(MoeDecodeParams& p, bool up, int tokens) {
    const int cols = up ? 8 : 16, groups = (up ? p.inter : p.N) / cols;
    const int nbs = (groups * cols + 127) / 128 + 1;   // block rows of a segment, at most
    p.wscale_cap = (nbs * (up ? 2 : 1) * p.kblocks + 63) / 64 * 64;
    const float mean = (float)p.slots / (float)p.E, likely = fminf(mean + 3.0f * sqrtf(mean), (float)tokens);
    const int most = likely < 18.0f ? 16 : 32;
    int cap = 1;
    while (cap < tokens && cap < most) cap *= 2;
    while (cap > 1) {
        p.row_cap = cap;
        if (MoeDecodeLds::of(p).total <= kLdsBytes) break;
        cap /= 2;
    }
    p.row_cap = cap;
    return MoeDecodeLds::of(p).total <= kLdsBytes && likely < (float)(cap + 2);
}

template <typename T, bool UP, int MT>
hipError_t launch_decode(const MoeDecodeParams& p, hipStream_t s) {
    // one workgroup per compute unit: each takes an equal share of the weights
    hipLaunchKernelGGL((moe_decode_kernel<T, UP, MT>), dim3((unsigned)compute_units()), dim3(64 * (kDecodeWaves + kDecodeQuantWaves)),
                       (size_t)MoeDecodeLds::of(p).total, s, p);
    return hipGetLastError();
}

template <typename T>
hipError_t dispatch_decode(const MoeDecodeParams& p, bool up, hipStream_t s) {
    if (p.row_cap > 16) return up ? launch_decode<T, true, 2>(p, s) : launch_decode<T, false, 2>(p, s);
    return up ? launch_decode<T, true, 1>(p, s) : launch_decode<T, false, 1>(p, s);
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
