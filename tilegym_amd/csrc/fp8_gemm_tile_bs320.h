// 256 x 320 block-scaled tile: C[m,n] = sum_kb As[m,kb] * Bs[n/128,kb] * sum_{k in kb} A[m,k] * B[n,k], for problems whose 256 x 256
// tiles leave the last round of the chip mostly empty and whose 256 x 320 tiles do not.
//
// 4096 x 5120 is 320 tiles of 256 x 256 (a full round of 256 compute units and a quarter of one) and exactly 256 of 256 x 320.
// Schedule, slab layout, swizzles, fragment addressing and arithmetic are those of
// fp8_gemm_tile_kernel<256, 256, 4, 2, true, GROUP_DENSE, false> (see there): identical results.  What differs:
//   * a wave's part is 64 x 160: 160 accumulator registers.  To stay inside the register file (255 of 256) a wave keeps one per-lane
//     offset per operand, the pass of the loads being in the scalar offset.  There is no register left to clamp the rows of a last
//     tile, and the descriptors are not sized to the operands: what keeps every load inside them is that the last row and column
//     tiles are moved back to end with the operands (and store only what is theirs), which takes M >= 256, N >= 320 and
//     N % 32 == 0 (bs320_takes; a wave's edge between two weight scales lies at a multiple of 32 columns);
//   * the two stages take 144 KiB of LDS and the activation scales the other 16.  The weight scales come through scalar loads, one
//     step ahead.  A wave's 160 columns lie in two blocks of 128: the pairs of column tiles in front of the boundary take
//     the first block's scale, the others the second one's.
// Bound by power and issue like the 256 x 256 form (1.8 GHz on average over the launch, 0.57 of the matrix slots: the counters in
// profiles/ring_pair_bs320_pmc.txt); it moves a tenth fewer bytes to LDS per MFMA.  Quantizer and GEMM, us, side by side with the 256 x 256
// tiles, in two pieces where the last round was mostly empty, and the quantizer before it: 4096 x 5120 x 12288 278 -> 250,
// 4096 x 5120 x 4096 99 -> 85, 3000 x 6400 x 7168 168 -> 138, 8192 x 5120 x 5120 240 -> 219.  With whole rounds of 256 x 256 tiles
// that form is ahead (4096 x 12288 x 5120: 222 against 274 for the GEMM): the cost model decides.
#pragma once

#include "fp8_gemm_tile.h"
#include "fp8_gemm_tile_bs256.h"

namespace tg {

__global__ void __launch_bounds__(512, 1) fp8_gemm_bs320_kernel(const GemmParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int BM = 256, BN = 320, WGM = 4, WGN = 2, NW = 8;
    constexpr int WTN = BN / WGN, TM = 4, TN = WTN / 16, TP = TN / 2;
    constexpr int A_IT = BM / (8 * NW), B_IT = BN / (8 * NW);
    constexpr int S_GROUPS = BM / 8, S_PHASES = S_GROUPS / NW;
    static_assert(TN == 10 && A_IT == 4 && B_IT == 5 && S_PHASES <= kScaleChunk, "shape");

    __shared__ __align__(1024) uint8_t sA0[BM * kKBlock];
    __shared__ __align__(1024) uint8_t sA1[BM * kKBlock];
    __shared__ __align__(1024) uint8_t sB0[BN * kKBlock];
    __shared__ __align__(1024) uint8_t sB1[BN * kKBlock];
    __shared__ __align__(256) float sTab[2 * BM * kScaleChunk];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WGM, wn = wave / WGM;
    const int K = p.K, kblocks = p.kblocks, last = kblocks - 1;
    const int tiles_n = (p.N + BN - 1) / BN, tiles_m = (p.M + BM - 1) / BM;
    const int pid = xcd_remap((int)blockIdx.x, tiles_m * tiles_n);
    constexpr int GM = 8;
    const int width = GM * tiles_n;
    const int group = pid / width, first_m = group * GM;
    const int gsz = min(tiles_m - first_m, GM);
    const int m_first = (first_m + (pid % width) % gsz) * BM, n_first = ((pid % width) / gsz) * BN;
    // the last row and column tiles are moved back to end with the operands and store what is theirs
    const int m0 = min(m_first, p.M - BM), n0 = min(n_first, p.N - BN);

    const int lrow = lane >> 3;
    const uint32_t a_off = (uint32_t)(m0 + wave * 8 + lrow) * (uint32_t)K + ((lane & 7) ^ swz16(lrow)) * 16;
    const uint32_t b_off = (uint32_t)(n0 + wave * 8 + lrow) * (uint32_t)K + ((lane & 7) ^ swz_w(((wave & 1) << 3) | lrow)) * 16;
    const v4i rsrc_a = make_rsrc(p.A), rsrc_b = make_rsrc(p.B);
    const v4i rsrc_s = make_rsrc(p.As);
    auto load_a = [&](int i, int kstep, uint8_t* dA) { direct_load_b128(rsrc_a, lds_address(dA) + wave * 1024 + i * NW * 1024, a_off, kstep * kKBlock + i * 64 * K); };
    auto load_b = [&](int kstep, uint8_t* dB) {
#pragma unroll
        for (int i = 0; i < B_IT; ++i) direct_load_b128(rsrc_b, lds_address(dB) + wave * 1024 + i * NW * 1024, b_off, kstep * kKBlock + i * 64 * K);
    };
    // activation scales: chunks of eight K steps, one 8-row group per wave and step (layout: fp8_gemm_tile.h)
    const int s_kbi = ((lane & 7) - lrow) & 7;
    auto load_s = [&](int chunk, int ph) {
        const int g = ph * NW + wave;
        if (g < S_GROUPS) {
            const int row = m0 + g * 8 + lrow;
            const int kb = min(chunk * kScaleChunk + s_kbi, last);
            direct_load_b32(rsrc_s, lds_address(sTab) + ((chunk & 1) * BM * kScaleChunk + g * 64) * 4, ((uint32_t)row * (uint32_t)kblocks + (uint32_t)kb) * 4u, 0);
        }
    };

    const int li = lane & 15, lg = lane >> 4;
    const uint32_t frag0 = wm * 16 * kKBlock + li * kKBlock + ((lg ^ swz16(li)) << 4), frag1 = frag0 ^ 64;
    const int wrow = ((li >> 2) << 3) | (li & 3);
    const uint32_t wfrag0 = wn * WTN * kKBlock + wrow * kKBlock + ((lg ^ swz_w(wrow)) << 4), wfrag1 = wfrag0 ^ 64;
    // weight scales of the wave's two column blocks
    const int c0 = n0 + wn * WTN;
    const int edge = (128 - c0 % 128) / 32;  // pairs of column tiles in the first block: 1 .. 4
    const float* const bs0 = p.Bs + (int64_t)(c0 / 128) * kblocks;
    const float* const bs1 = p.Bs + (int64_t)(c0 / 128 + 1) * kblocks;
    float b0 = uniform_load_f32(bs0), b1 = uniform_load_f32(bs1);
    const int s_rbase = (wm * 2 + (li >> 3)) * 64 + (li & 7) * 8;

    v4f acc[TN][TM];
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) acc[tn][tm] = v4f{0.f, 0.f, 0.f, 0.f};

    constexpr int kWaitAllButA = 0x0F70 | A_IT, kWaitAll = 0x0F70, kWaitLds = 0xC07F;
#define TG_FENCE() __builtin_amdgcn_sched_barrier(0)
    load_b(0, sB0);
#pragma unroll
    for (int i = 0; i < A_IT; ++i) load_a(i, 0, sA0);
#pragma unroll
    for (int ph = 0; ph < S_PHASES; ++ph) load_s(0, ph);
#pragma unroll
    for (int i = 0; i < A_IT; ++i) load_a(i, min(1, last), sA1);
    __builtin_amdgcn_s_waitcnt(kWaitAllButA);
    __builtin_amdgcn_s_waitcnt(kWaitLds);
    __builtin_amdgcn_s_barrier();
    auto step = [&](int k, uint8_t* cA, const uint8_t* cB, uint8_t* oB) __attribute__((always_inline)) {
        load_b(min(k + 1, last), oB);
        load_s(k / kScaleChunk + 1, k % kScaleChunk);
        v8i af[TM], wf[2];
        float as[TM];
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
            const uint8_t* base = cA + tm * (WGM * 16 * kKBlock);
            af[tm] = join(*reinterpret_cast<const v4i*>(base + frag0), *reinterpret_cast<const v4i*>(base + frag1));
        }
        const float* cs = sTab + ((k / kScaleChunk) & 1) * (BM * kScaleChunk) + s_rbase + (((k % kScaleChunk) + li) & 7);
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) as[tm] = cs[tm * (WGM * 128)];
        auto read_w = [&](int tn) {
            const uint8_t* base = cB + ((tn >> 1) * 32 + (tn & 1) * 4) * kKBlock;
            wf[tn & 1] = join(*reinterpret_cast<const v4i*>(base + wfrag0), *reinterpret_cast<const v4i*>(base + wfrag1));
        };
        const float w0 = b0, w1 = b1;
        b0 = uniform_load_f32(bs0 + min(k + 1, last));
        b1 = uniform_load_f32(bs1 + min(k + 1, last));
        __builtin_amdgcn_s_waitcnt(kWaitLds);
        __builtin_amdgcn_s_barrier();
        TG_FENCE();
        v4f part[3];
        float sc[2][TM];  // of the current pair of column tiles and the one before
        auto add = [&](int j) __attribute__((always_inline)) {
            const int tn = j / TM, tm = j % TM;
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[tn][tm][r] = __builtin_fmaf(part[j % 3][r], sc[(tn >> 1) & 1][tm], acc[tn][tm][r]);
        };
        read_w(0);
#pragma unroll
        for (int j = 0; j < TN * TM; ++j) {
            const int tn = j / TM, tm = j % TM;
            part[j % 3] = mfma_e4m3(wf[tn & 1], af[tm], v4f{0.f, 0.f, 0.f, 0.f});
            if (tm == 0 && tn + 1 < TN) read_w(tn + 1);
            if (j >= 2) add(j - 2);
            if ((tn & 1) == 0 && tm == 1) {  // (behind the last use of this set, in front of its first new one)
                const float w = tn / 2 < edge ? w0 : w1;
#pragma unroll
                for (int t = 0; t < TM; ++t) sc[(tn >> 1) & 1][t] = as[t] * w;
            }
            TG_FENCE();
            if (tm == TM - 1 && tn < A_IT) {
                load_a(tn, min(k + 2, last), cA);
                TG_FENCE();
            }
        }
        add(TN * TM - 2);
        add(TN * TM - 1);
        // keep the scale-and-add chain inside this step (see fp8_gemm_tile.h)
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
#pragma unroll
            for (int tm = 0; tm < TM; ++tm) asm volatile("" : "+v"(acc[tn][tm]));
        __builtin_amdgcn_s_waitcnt(kWaitAllButA);
        __builtin_amdgcn_s_waitcnt(kWaitLds);
        __builtin_amdgcn_s_barrier();
    };
    int k = 0;
    for (; k + 1 < kblocks; k += 2) {
        step(k, sA0, sB0, sB1);
        step(k + 1, sA1, sB1, sB0);
    }
    if (k < kblocks) step(k, sA0, sB0, sB1);
#undef TG_FENCE
    __builtin_amdgcn_s_waitcnt(kWaitAll);  // the re-fetches past the end must land before the workgroup's LDS is released

    const bool vec_ok = p.vec_store != 0 && (p.N % 8) == 0;
    const float scale = p.alpha;
    auto emit = [&](auto type_tag) __attribute__((always_inline)) {
        constexpr int OT = decltype(type_tag)::value;
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
            const int row = m0 + (tm * WGM + wm) * 16 + li;
#pragma unroll
            for (int tp = 0; tp < TP; ++tp) {
                const int col = c0 + tp * 32 + lg * 8;
                if (row < m_first || col < n_first) continue;
                store8(p.C, OT, row, col, p.N, p.ldc, acc[2 * tp][tm] * scale, acc[2 * tp + 1][tm] * scale, p.beta, vec_ok);
            }
        }
    };
    if (p.out_type == OUT_BF16) emit(std::integral_constant<int, OUT_BF16>{});
    else if (p.out_type == OUT_F32) emit(std::integral_constant<int, OUT_F32>{});
    else if (p.out_type == OUT_F8) emit(std::integral_constant<int, OUT_F8>{});
    else emit(std::integral_constant<int, OUT_F16>{});
#endif
}

}  // namespace tg
