// Device side of the per-token group quantizer (see quant.hip): shared by the stand-alone kernel and by the kernel that
// runs it beside moe_align_block_size (moe_prepare.hip).
#pragma once
#include <type_traits>

#include "tg_host.h"

typedef float v8f_q __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8_q __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_q __attribute__((ext_vector_type(8)));

namespace tg {

template <typename T>
__device__ __forceinline__ v8f_q load8(const T* p);
template <>
__device__ __forceinline__ v8f_q load8<__bf16>(const __bf16* p) {
    return __builtin_convertvector(*reinterpret_cast<const bf16x8_q*>(p), v8f_q);
}
template <>
__device__ __forceinline__ v8f_q load8<_Float16>(const _Float16* p) {
    return __builtin_convertvector(*reinterpret_cast<const f16x8_q*>(p), v8f_q);
}
template <>
__device__ __forceinline__ v8f_q load8<float>(const float* p) {
    const v4f lo = reinterpret_cast<const v4f*>(p)[0], hi = reinterpret_cast<const v4f*>(p)[1];
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// kQuantGroupsPerLane groups per lane, all loads issued before the first use (one 16-byte load per lane
// leaves too few bytes in flight per wave for an HBM-bound kernel).
constexpr int kQuantGroupsPerLane = 4;
// One group per lane below this many workgroups of four (67 M elements): four are worked through one after the other, and more
// waves hide more.  Kernel with launch, four -> one, bf16 in groups of 128: 16 x 5120 4.1 -> 2.2 us, 256 x 4096 4.3 -> 2.5,
// 1024 x 4096 6.4 -> 4.8, 4096 x 5120 19.9 -> 15.8, 4096 x 12288 36.5 -> 35.4; 8192 x 14336 70.8 -> 76.4 and 32000 x 16384
// 281 -> 307 with one, so four from there on.  Groups of 16, 4096 x 8192: 21.0 -> 18.5; f32 30.4 -> 28.9.
constexpr int64_t kQuantFewWorkgroups = 1 << 13;

enum QuantRule { QUANT_ZERO_TO_ONE = 0, QUANT_EPS = 1, QUANT_EPS_POW2 = 2 };

// Maximum over the LPG (2, 4, 8, 16) neighbouring lanes of a group, in every one of them: lane permutations inside the vector
// instruction, no trip through the LDS crossbar.
template <int CTRL>
__device__ __forceinline__ float dpp_max(float v) {
    return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true)));
}
template <int LPG>
__device__ __forceinline__ float group_max(float v) {
    static_assert(LPG == 2 || LPG == 4 || LPG == 8 || LPG == 16, "inside a row of 16 lanes");
    v = dpp_max<0xB1>(v);                             // quad_perm [1, 0, 3, 2]
    if constexpr (LPG >= 4) v = dpp_max<0x4E>(v);     // quad_perm [2, 3, 0, 1]
    if constexpr (LPG >= 8) v = dpp_max<0x141>(v);    // row_half_mirror: the other four of eight
    if constexpr (LPG >= 16) v = dpp_max<0x140>(v);   // row_mirror: the other eight of sixteen
    return v;
}

// Elements of a 16-bit type against the scale of their group's maximum: four fewer instructions per element than ScaleDivider.
// With s = amax / 448, |a| <= amax, r the reciprocal of s and t = a r, the quotient after ONE residual correction rounds to the
// same e4m3 code as the IEEE quotient a / s: checked for every pair of significands of a and amax (7 + 7 bits for bf16, 10 + 10
// for f16), 24 exponent differences, and r one unit in the last place off in either direction.  Beyond 24 binades both are
// zero.  (The kernel is bound by its vector instructions: 4096 x 12288 bf16 32.2 -> 26.1 us with this and the lane permutations
// above, 5.8 TB/s.)  The residual is taken as s t - a and subtracted, which keeps the sign of a zero.  The scale itself needs no general
// division either: amax times the rounded 1 / 448 with one correction is the IEEE quotient for every such amax.
constexpr float kShortMin = 0x1p-50f, kShortMax = 0x1p50f;   // amax inside: every intermediate is a normal number
__device__ __forceinline__ float short_scale(float amax) {
    const float q = amax * (1.0f / 448.0f);
    return __builtin_fmaf(-__builtin_fmaf(448.0f, q, -amax), 1.0f / 448.0f, q);
}
__device__ __forceinline__ float short_quotient(float a, float s, float r) {
    const float t = a * r;
    return __builtin_fmaf(-__builtin_fmaf(s, t, -a), r, t);
}

// LPG lanes per group (group size 8 * LPG).  STRIDED: the scale of group j of row r goes to
// scales[r * s_row + j * s_col] (groups < 2^31); otherwise to scales[g].
// I8: the destination is int8 instead of e4m3 (per_token_group_quant_8bit with dst_dtype=torch.int8,
// tests/suites/flashinfer/test_per_token_group_quant_8bit.py:41-68): scale = amax / 127, q = the quotient clamped to
// [-128, 127] and converted as a float -> integer cast does (toward zero).
// (body of 256-thread block `block`, thread `tid` of it: the kernel below runs it as such, the MoE preparation kernel
// runs four such blocks per 1024-thread workgroup)
template <typename T, int LPG, bool STRIDED, bool I8, int G = kQuantGroupsPerLane>
__device__ __forceinline__ void act_quant_group_body(const T* __restrict__ x, uint8_t* __restrict__ q,
                                                     float* __restrict__ scales, int64_t groups, float eps,
                                                     int rule, uint32_t groups_per_row, int64_t s_row, int64_t s_col,
                                                     const int64_t block, const int tid) {
    constexpr int GS = 8 * LPG, PASS = 256 / LPG;
    constexpr float QMAX = I8 ? 127.0f : 448.0f, QMIN = I8 ? -128.0f : -448.0f;
    const int sub = tid & (LPG - 1);
    const int64_t g0 = block * (PASS * G) + (tid / LPG);
    v8f_q v[G];
#pragma unroll
    for (int j = 0; j < G; ++j) {
        const int64_t g = g0 + j * PASS;
        // the LPG lanes of a group are in or out together: the shuffles below stay inside a group
        if (g < groups) v[j] = load8<T>(x + g * GS + sub * 8);
        else {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[j][i] = 0.f;
        }
    }
#pragma unroll
    for (int j = 0; j < G; ++j) {
        const int64_t g = g0 + j * PASS;
        float amax = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(v[j][i]));
        amax = group_max<LPG>(amax);
        if (g >= groups) continue;
        float s, c[8];
        if (!I8 && !std::is_same_v<T, float> && rule != QUANT_EPS_POW2 && amax >= kShortMin && amax <= kShortMax && (rule == QUANT_ZERO_TO_ONE || amax >= eps)) {
            s = short_scale(amax);
            const float r = ScaleDivider(s).r;
#pragma unroll
            for (int i = 0; i < 8; ++i) c[i] = short_quotient(v[j][i], s, r);
        } else {
            if (rule == QUANT_ZERO_TO_ONE) s = amax == 0.f ? 1.0f : amax / QMAX;
            else s = fmaxf(amax, eps) / QMAX;
            if (rule == QUANT_EPS_POW2) s = exp2f(ceilf(log2f(fmaxf(fabsf(s), 1e-10f))));
            const ScaleDivider div(s);
            if (div.fast) {
#pragma unroll
                for (int i = 0; i < 8; ++i) c[i] = div.quotient(v[j][i]);
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) c[i] = v[j][i] / s;
            }
        }
        int packed[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float cc[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) cc[i] = __builtin_amdgcn_fmed3f(c[4 * h + i], QMIN, QMAX);  // (NaN: QMIN, as fminf(fmaxf()))
            int w = 0;
            if constexpr (I8) {
#pragma unroll
                for (int i = 0; i < 4; ++i) w |= ((int)cc[i] & 0xFF) << (8 * i);
            } else {
                w = __builtin_amdgcn_cvt_pk_fp8_f32(cc[0], cc[1], w, false);
                w = __builtin_amdgcn_cvt_pk_fp8_f32(cc[2], cc[3], w, true);
            }
            packed[h] = w;
        }
        *reinterpret_cast<v2i*>(q + g * GS + sub * 8) = v2i{packed[0], packed[1]};
        if (sub == 0) {
            if constexpr (STRIDED) {
                const uint32_t row = (uint32_t)g / groups_per_row, col = (uint32_t)g - row * groups_per_row;
                scales[row * s_row + col * s_col] = s;
            } else {
                scales[g] = s;
            }
        }
    }
}

}  // namespace tg
