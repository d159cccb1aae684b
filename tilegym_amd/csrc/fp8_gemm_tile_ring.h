// Tiles of 32 x 64 to 256 x 128 over a ring of LDS stages: C[m,n] = sum_k A[m,k] * B[n,k], per-tensor or block scales (tiles of
// 64 and 128 columns), for the row counts between decoding and those that fill whole rounds of 256 x 256 tiles.
//
// One workgroup per compute unit: four waves compute (2 x 2, one per SIMD), four waves do nothing but request the next K steps'
// slabs.  A direct global->LDS load holds its wave until the compute unit's address path has room (about 16 clocks per 1 KiB
// load, whoever issues it).  At these tile sizes a step's loads take about as long as its MFMAs (160 x 128: 576 against 640
// clocks), and with every wave loading and computing the two came one after the other: 256 x 4096 x 4096 with 160 x 128 tiles
// took 20.0 us with four such waves, 15.9 with the loads in waves of their own.
//
// Three to twelve stages hold a K step each; a stage is requested again as soon as every computing wave has read it, so
// STAGES - 1 steps are on their way while one is multiplied.  One barrier per step, in front of its last column tiles: behind it
// step k+1 is visible and step k's stage is free, and the fragments of step k+1 are read while those last MFMAs run (activation
// fragments into the registers that a row group's last MFMA releases, weight fragments over three or four rotating sets).
//
// Bound on a full chip by power, that is by bytes moved per MFMA: a 160 x 128 tile of 32 steps takes 38 thousand cycles, 0.53 of them
// with the matrix pipes busy, whether 64 or 240 compute units work; 64 tiles take 18.2 us, 240 tiles of zeros 19.6, 240 of random data
// 22.2 - 22.9 (2.1, 1.94 and 1.69 GHz on average: the counters in profiles/ring_pair_bs320_pmc.txt).  Hence the 192 x 192 tile for larger
// problems, which moves a quarter less.  Measured side by side with the choice among the other kernels (us): 777 x 6144 x 4096 26.9 -> 19.9,
// 1400 x 12288 x 5120 101 -> 78, 1014 x 5120 x 12288 83 -> 61, 512 x 4096 x 4096 17.8 -> 12.8, 185 x 6144 x 4096 16.9 -> 11.8.  A fifth kind
// of wave that touched the lines of steps further ahead to have them in the caches: no faster (23.8 against 25.2 and 54.3 against
// 53.0 us), not kept.
//
// Block scales: a step's products are scaled and added as in fp8_gemm_tile.h.  The loading waves bring the activation scales
// too, in chunks of eight K steps spread over the steps of the chunk before; the scales of step k+1 are read behind the barrier of
// step k.  With the quantizer 485 x 6144 x 4096 30.6 -> 23.6 us, 174 x 3520 x 4992 21.4 -> 18.0,
// 62 x 6144 x 4096 18.4 -> 15.4.
//
// 32 and 64 rows or columns, up to twelve stages: one round of workgroups over 4096 to 12288 weight rows at 24 to 256 rows, bound by
// the bytes a compute unit takes in from its L2 (a 64 x 64 step 0.17 us = 46 bytes a clock, 3.7 us besides, of which 1.9 are the
// launch).  Against the tiles whose four waves split K (fp8_gemm_tile_mid.h) and 64 x 128 tiles with splits: 256 x 4096 x 4096 12.1 -> 9.0
// us, 128 x 6144 x 4096 12.2 -> 8.7, 50 x 12288 x 5120 17.4 -> 12.5, 50 x 4096 x 14336 18.0 -> 15.4, 24 x 12288 x 5120 17.1 -> 12.2.
// 256 x 128: 200 x 28672 x 4096 44 -> 37.
//
// KN: the weight is (K, N); its slab is 128 K rows of BN bytes, staged as they lie and turned on the way out of LDS
// (ds_read_b64_tr_b8), so no (N, K) copy is made.  Bound as above: the lines of a K row tile are whole with 128 columns and halves with
// 64 (1.62 instead of 1.05 million requests to L2 at 256 x 4096 x 4096: 13.6 us, 32 x 128 tiles 12.8, the (N, K) form 9.0; from memory 19.7 and 19.0).  What it measured
// against the copy stands at pick_kn_tile.  Not kept: tiles dealt over the XCDs column by column in other orders (within 5 %
// either way), weights fetched past the first-level cache (30 to 50 % slower).
//
// ONCE, for one row tile over a weight that comes from memory (100 MB and more: three sets of operands do not fit in the caches):
// the weight loads are non-temporal, and workgroup b starts at K step b of its range and goes round -- rows a power of two apart
// would put the requests of one moment on few memory channels.  The same products are added, in a rotated order: not the bits of
// the other forms.  Hence only where the library chooses the tile, or ROW_GROUPS = 1 asks for it.  28672 x 4096,
// us before / after over three sets of operands and over 1 GB of weights, per-tensor: 50 rows 26.1 / 23.4 and 28.6 / 24.4, 90 rows 29.3 / 25.7
// and 31.1 / 26.8, 128 rows 31.0 / 28.6 and 32.8 / 29.2, 256 rows 44.0 / 35.7 and 44.6 / 36.0; block-scaled: 16 rows 26.2 / 25.3 and 26.6 / 26.4,
// 50 rows 29.8 / 26.5 and 31.6 / 26.9.  Either alone 24 - 25.5 at 24 rows, both 22.3.  Smaller weights stay in the caches from one call to
// the next and are up to 1.4 x slower with non-temporal loads; K that is no power of two is 3 - 5 % slower rotated and the same without.
//
// Same slab layout, swizzles, fragment addressing, arithmetic per accumulator and epilogue as
// fp8_gemm_tile_kernel<128, 128, 2, 2, BLOCKSCALE, GROUP_DENSE, SPLIT>: identical results but for ONCE's order over a K that is a power
// of two.
#pragma once

#include "fp8_gemm_tile.h"

namespace tg {

// Place of 16-byte chunk j of K row r of a (K, N) slab: j ^ swz_kn(r).  Two groups of 16 lanes fetch 8 K rows of one chunk each at
// once, rows r ... r + 7 and r + 16 ... r + 23.  128-byte rows: row bit 0 picks a half of the 64 banks, bits 1, 2 and 4 the place in
// it.  64-byte rows: bits 0 and 1 pick a quarter, bits 2 and 4 the place.
template <int BN>
__device__ __forceinline__ int swz_kn(int r) { return BN == 64 ? ((r >> 2) & 1) | ((r >> 3) & 2) : ((r >> 1) & 3) | ((r >> 2) & 4); }

template <int BM, int BN, int STAGES, bool BLOCKSCALE, bool SPLIT, bool KN, bool ONCE>
__global__ void __launch_bounds__(512, 1) fp8_gemm_tile_ring_kernel(const GemmParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int NL = 4, WGN = BN == 32 ? 1 : 2, WGM = 4 / WGN;  // four loading waves, four computing waves
    constexpr int WTN = BN / WGN;
    constexpr int TM = BM / (16 * WGM), TN = WTN / 16;
    constexpr int A_IT = BM / (8 * NL), B_IT = BN / (8 * NL);
    constexpr int STAGE_BYTES = (BM + BN) * kKBlock;
    constexpr int S_GROUPS = BM / 8, S_PHASES = (S_GROUPS + NL - 1) / NL;  // 8-row groups of activation scales; K steps a chunk's loads are spread over
    constexpr int PER_STEP = A_IT + B_IT + (BLOCKSCALE ? 1 : 0);
    constexpr int WS = TN == 6 ? 3 : 4;                 // weight fragment sets
    constexpr int LAST = TN == 4 ? 2 : 1;               // column tiles behind the barrier
    static_assert(BM % (16 * WGM) == 0 && (TN == 2 || TN == 4 || TN == 6) && STAGES >= 3 && STAGES * STAGE_BYTES <= 160 * 1024, "shape");

    static_assert(!KN || ((BN == 128 || BN == 64) && !BLOCKSCALE), "(K, N) weights: a K row of the tile is one 128-byte line or half of one");
    static_assert(!BLOCKSCALE || (128 % BN == 0 && S_PHASES + STAGES - 1 <= kScaleChunk), "one weight scale per tile; a chunk of activation scales lands before its first step");

    __shared__ __align__(1024) uint8_t lds[STAGES * STAGE_BYTES];  // stage s: A slab, then B slab
    // block scales: activation scales of the tile's rows, two chunks of kScaleChunk K steps, laid out as in fp8_gemm_tile.h, and
    // the weight scales of the tile's column block for every K step
    __shared__ __align__(256) float s_as[BLOCKSCALE ? 2 * BM * kScaleChunk : 1];
    __shared__ float s_bs[BLOCKSCALE ? kMaxKBlocks : 1];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = p.K;
    const int tiles_n = (p.N + BN - 1) / BN, tiles_m = (p.M + BM - 1) / BM;
    const int pid = xcd_remap((int)blockIdx.x, tiles_m * tiles_n);
    constexpr int GM = 8;
    const int width = GM * tiles_n;
    const int group = pid / width, first_m = group * GM;
    const int gsz = min(tiles_m - first_m, GM);
    const int m0 = (first_m + (pid % width) % gsz) * BM, n0 = ((pid % width) / gsz) * BN;
    const int rows_valid = min(BM, p.M - m0);
    int ks = 0, ks_end = p.kblocks;
    if constexpr (SPLIT) {
        ks = blockIdx.y * p.ksteps_per_split;
        ks_end = min(ks + p.ksteps_per_split, p.kblocks);
    }
    const int nsteps = ks_end - ks, last = ks_end - 1;
    if (nsteps <= 0) return;
    // ONCE: first K step of this workgroup; step ks + k is the kth behind it, round the end of the range
    const int turn = ONCE && (K & (K - 1)) == 0 ? pid % nsteps : 0;

    constexpr int kPro = (STAGES - 1) * PER_STEP, kLoop = (STAGES - 2) * PER_STEP;  // loads that may stay in flight
    static_assert(kPro < 64, "vmcnt has six bits");
    constexpr int kWaitPro = 0x0F70 | (kPro & 15) | ((kPro >> 4) << 14);
    constexpr int kWaitLoop = 0x0F70 | (kLoop & 15) | ((kLoop >> 4) << 14);
    constexpr int kWaitAll = 0x0F70;
    constexpr int kWaitLds = 0xC07F;
#define TG_FENCE() __builtin_amdgcn_sched_barrier(0)

    if (wave >= 4) {
        // ------------------------------------------------------------ loading waves
        const int lw = wave - 4;
        const int lrow = lane >> 3;
        const int lj = (lane & 7) ^ swz16(lrow);
        const int ljb = (lane & 7) ^ swz_w(((lw & 1) << 3) | lrow);
        uint32_t a_off[A_IT], b_off[B_IT];
#pragma unroll
        for (int i = 0; i < A_IT; ++i) a_off[i] = (uint32_t)(m0 + min((i * NL + lw) * 8 + lrow, rows_valid - 1)) * (uint32_t)K + lj * 16;
#pragma unroll
        for (int i = 0; i < B_IT; ++i) {
            // (KN: K row kr, whose 16-byte place q holds chunk q ^ swz_kn(kr); columns past N repeat the last ones)
            const int kr = (i * NL + lw) * (1024 / BN) + lane / (BN / 16), q = lane % (BN / 16);
            if constexpr (KN) b_off[i] = (uint32_t)kr * (uint32_t)p.N + min(n0 + ((q ^ swz_kn<BN>(kr)) << 4), p.N - 16);
            else b_off[i] = (uint32_t)min(n0 + (i * NL + lw) * 8 + lrow, p.N - 1) * (uint32_t)K + ljb * 16;
        }
        const v4i rsrc_a = make_rsrc(p.A), rsrc_b = make_rsrc(p.B);
        const uint32_t lds0 = lds_address(lds) + lw * 1024;
        const v4i rsrc_s = make_rsrc(p.As ? p.As : kOneScale);
        const int s_kbi = ((lane & 7) - lrow) & 7;    // chunk step this lane fetches
        // row group `ph` of this wave, chunk `chunk` of K steps (a phase past the last group fetches the last one again: every step
        // requests the same number of loads)
        auto issue_s = [&](int chunk, int ph) {
            if constexpr (BLOCKSCALE) {
                const int g = min(ph * NL + lw, S_GROUPS - 1);
                const int row = m0 + min(g * 8 + lrow, rows_valid - 1);
                int kb = ks + chunk * kScaleChunk + s_kbi;
                if constexpr (ONCE) {
                    kb += turn;
                    if (kb > last) kb -= nsteps;
                }
                kb = min(kb, p.kblocks - 1);
                direct_load_b32(rsrc_s, lds_address(s_as) + ((chunk & 1) * BM * kScaleChunk + g * 64) * 4,
                                p.As ? ((uint32_t)row * (uint32_t)p.kblocks + (uint32_t)kb) * 4u : 0u, 0);
            }
        };
        auto issue = [&](int kstep, int stage) {
            if constexpr (ONCE) {
                kstep += turn;
                if (kstep > last) kstep -= nsteps;
            }
            const int k0 = min(kstep, last) * kKBlock;
            const uint32_t dst = lds0 + stage * STAGE_BYTES;
#pragma unroll
            for (int i = 0; i < B_IT; ++i) {
                if constexpr (ONCE) direct_load_b128_nt(rsrc_b, dst + BM * kKBlock + i * NL * 1024, b_off[i], k0);
                else direct_load_b128(rsrc_b, dst + BM * kKBlock + i * NL * 1024, b_off[i], KN ? k0 * p.N : k0);
            }
#pragma unroll
            for (int i = 0; i < A_IT; ++i) direct_load_b128(rsrc_a, dst + i * NL * 1024, a_off[i], k0);
        };
        if constexpr (BLOCKSCALE)
            for (int ph = 0; ph < S_PHASES; ++ph) issue_s(0, ph);
#pragma unroll
        for (int s = 0; s < STAGES; ++s) {
            if (s > 0) issue_s(0, 0);  // (again, for the count: the waits below take every step's requests to be PER_STEP)
            issue(ks + s, s);
        }
        __builtin_amdgcn_s_waitcnt(kWaitPro);
        __builtin_amdgcn_s_barrier();
        int stage = 0;
        for (int k = 0; k < nsteps; ++k) {
            __builtin_amdgcn_s_waitcnt(kWaitLoop);  // step k+1 has landed (steps past the end re-fetch the last one)
            __builtin_amdgcn_s_barrier();           // and every computing wave has read step k
            if constexpr (BLOCKSCALE) issue_s(k / kScaleChunk + 1, k % kScaleChunk);
            issue(ks + k + STAGES, stage);
            stage = stage == STAGES - 1 ? 0 : stage + 1;
        }
        __builtin_amdgcn_s_waitcnt(kWaitAll);  // the re-fetches past the end must land before the workgroup's LDS is released
        return;
    }

    // ---------------------------------------------------------------- computing waves
    TensorScales scales(BLOCKSCALE ? GemmParams{} : p);
    const int wm = wave % WGM, wn = wave / WGM;
    const int li = lane & 15, lg = lane >> 4;
    const uint32_t frag0 = wm * 16 * kKBlock + li * kKBlock + ((lg ^ swz16(li)) << 4), frag1 = frag0 ^ 64;
    const int wrow = ((li >> 2) << 3) | (li & 3);
    const uint32_t wfrag0 = BM * kKBlock + wn * WTN * kKBlock + wrow * kKBlock + ((lg ^ swz_w(wrow)) << 4), wfrag1 = wfrag0 ^ 64;

    v4f acc[TN][TM];
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) acc[tn][tm] = v4f{0.f, 0.f, 0.f, 0.f};

    v8i af[TM], wf[WS];
    auto read_a = [&](int tm, const uint8_t* base) {
        const uint8_t* a = base + tm * (WGM * 16 * kKBlock);
        af[tm] = join(*reinterpret_cast<const v4i*>(a + frag0), *reinterpret_cast<const v4i*>(a + frag1));
    };
    // KN: column li of column tile tn is what 16 lanes turn out of 8 K rows x 16 columns (lane li fetches K row li / 2)
    uint32_t kn_off[KN ? TN : 1];
    if constexpr (KN) {
        const int r = lg * 16 + (li >> 1);
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) kn_off[tn] = BM * kKBlock + r * BN + (((wn * TN + tn) ^ swz_kn<BN>(r)) << 4) + (li & 1) * 8;
    }
    auto read_w = [&](int tn, const uint8_t* base) {
        if constexpr (KN) {
            // K bytes lg * 16 ... + 15 and 64 + lg * 16 ... + 15, eight at a time
            const uint32_t at = lds_address(base) + kn_off[tn];
            const v2i p0 = lds_read_transposed_8x16(at), p1 = lds_read_transposed_8x16(at + 8 * BN);
            const v2i p2 = lds_read_transposed_8x16(at + 64 * BN), p3 = lds_read_transposed_8x16(at + 72 * BN);
            wf[tn % WS] = v8i{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
            return;
        }
        const uint8_t* b = base + ((tn >> 1) * 32 + (tn & 1) * 4) * kKBlock;
        wf[tn % WS] = join(*reinterpret_cast<const v4i*>(b + wfrag0), *reinterpret_cast<const v4i*>(b + wfrag1));
    };
    // block scales of the coming step: activation scale of this lane's row in each row group, weight scale of the wave's columns
    float as_n[BLOCKSCALE ? TM : 1], bs_n = 0.f;
    const int s_rbase = (wm * 2 + (li >> 3)) * 64 + (li & 7) * 8;
    auto read_scales = [&](int k) {
        if constexpr (BLOCKSCALE) {
            const float* cs = s_as + ((k / kScaleChunk) & 1) * (BM * kScaleChunk) + s_rbase + (((k % kScaleChunk) + li) & 7);
#pragma unroll
            for (int tm = 0; tm < TM; ++tm) as_n[tm] = cs[tm * (WGM * 128)];
            k = min(k, nsteps - 1);
            if constexpr (ONCE) {
                k += turn;
                if (k >= nsteps) k -= nsteps;
            }
            bs_n = s_bs[k];
        }
    };
    if constexpr (BLOCKSCALE) {
        for (int kb = tid; kb < nsteps; kb += 256) s_bs[kb] = p.Bs ? p.Bs[(int64_t)(n0 / 128) * p.kblocks + ks + kb] : 1.0f;
        __builtin_amdgcn_s_waitcnt(kWaitLds);
    }
    __builtin_amdgcn_s_barrier();  // step 0 has landed
    scales.arrived();
    read_w(0, lds);
    read_w(1, lds);
    read_scales(0);
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) read_a(tm, lds);
    int stage = 0;
    for (int k = 0; k < nsteps; ++k) {
        const uint8_t* cur = lds + stage * STAGE_BYTES;
        stage = stage == STAGES - 1 ? 0 : stage + 1;
        const uint8_t* nxt = lds + stage * STAGE_BYTES;
        // one MFMA; with block scales into a fresh product, and behind it the scale-and-add of the product issued two MFMAs before
        // (see fp8_gemm_tile.h)
        v4f part[BLOCKSCALE ? 3 : 1];
        float sc[BLOCKSCALE ? TM : 1];
        if constexpr (BLOCKSCALE) {
#pragma unroll
            for (int tm = 0; tm < TM; ++tm) sc[tm] = as_n[tm] * bs_n;
        }
        constexpr int HEAD = (TN - LAST) * TM;  // MFMAs in front of the barrier, column tile by column tile; behind it row group by row group
        auto tn_of = [](int j) constexpr { return j < HEAD ? j / TM : TN - LAST + (j - HEAD) % LAST; };
        auto tm_of = [](int j) constexpr { return j < HEAD ? j % TM : (j - HEAD) / LAST; };
        auto add = [&](int j) __attribute__((always_inline)) {
            if constexpr (BLOCKSCALE) {
                if (j < 0) return;
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[tn_of(j)][tm_of(j)][r] = __builtin_fmaf(part[j % 3][r], sc[tm_of(j)], acc[tn_of(j)][tm_of(j)][r]);
            }
        };
        auto mma = [&](int j) __attribute__((always_inline)) {
            const int tn = tn_of(j), tm = tm_of(j);
            if constexpr (BLOCKSCALE) part[j % 3] = mfma_e4m3(wf[tn % WS], af[tm], v4f{0.f, 0.f, 0.f, 0.f});
            else acc[tn][tm] = mfma_e4m3(wf[tn % WS], af[tm], acc[tn][tm]);
        };
        TG_FENCE();
#pragma unroll
        for (int j = 0; j < HEAD; ++j) {
            mma(j);
            if (tm_of(j) == 0 && tn_of(j) + 2 < TN) read_w(tn_of(j) + 2, cur);
            add(j - 2);
            TG_FENCE();
        }
        __builtin_amdgcn_s_waitcnt(kWaitLds);  // all my reads of step k are done
        __builtin_amdgcn_s_barrier();          // step k+1 is visible
        TG_FENCE();
        read_w(0, nxt);
        if constexpr (TN > 2) read_w(1, nxt);
        read_scales(k + 1);
        TG_FENCE();
#pragma unroll
        for (int j = HEAD; j < TN * TM; ++j) {
            mma(j);
            add(j - 2);
            if (tn_of(j) == TN - 1) {
                TG_FENCE();
                read_a(tm_of(j), nxt);
            }
            TG_FENCE();
        }
        if constexpr (TN == 2) read_w(1, nxt);  // (its registers were the last MFMAs')
        if constexpr (BLOCKSCALE) {
            add(TN * TM - 2);
            add(TN * TM - 1);
            // keep the scale-and-add chain inside this step (see fp8_gemm_tile.h)
#pragma unroll
            for (int tn = 0; tn < TN; ++tn)
#pragma unroll
                for (int tm = 0; tm < TM; ++tm) asm volatile("" : "+v"(acc[tn][tm]));
        }
    }
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) asm volatile("" : : "v"(af[tm]));
    asm volatile("" : : "v"(wf[0]), "v"(wf[1]));
#undef TG_FENCE

    const float scale = BLOCKSCALE ? p.alpha : scales.times(p.alpha);
    const bool vec_ok = p.vec_store != 0 && (p.N % 8) == 0;
    const int64_t MN = (int64_t)p.M * p.N;
    // KN: a lane's four columns of tile t are 16 t + 4 lg ...; what lanes 16 apart hold of a tile pair changes places, so that eight
    // consecutive columns stand in one lane again
    if constexpr (KN) {
#pragma unroll
        for (int tp = 0; tp < TN / 2; ++tp)
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[2 * tp][tm][r]), __float_as_uint(acc[2 * tp + 1][tm][r]), false, false);
                    acc[2 * tp][tm][r] = __uint_as_float(sw[0]);
                    acc[2 * tp + 1][tm][r] = __uint_as_float(sw[1]);
                }
    }
    const int pair_col = KN ? (lg & 1) * 16 + (lg >> 1) * 8 : lg * 8;
    // Whole 16-byte stores without beta: straight code, no test per store (the general form below is forty times as long and its
    // way through the instruction cache takes longer than the stores).
    auto emit_whole = [&](auto type_tag) __attribute__((always_inline)) {
        constexpr int OT = decltype(type_tag)::value;
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
            const int rt = (tm * WGM + wm) * 16 + li;
            if (rt >= rows_valid) continue;
            const int col = n0 + wn * WTN + pair_col;
            const int64_t at = SPLIT ? (int64_t)blockIdx.y * MN + (int64_t)(m0 + rt) * p.N + col : (int64_t)(m0 + rt) * p.ldc + col;
#pragma unroll
            for (int tp = 0; tp < TN / 2; ++tp) {
                if (col + tp * 32 >= p.N) continue;
                if constexpr (SPLIT) put8<OUT_F32>(p.partials, at + tp * 32, acc[2 * tp][tm], acc[2 * tp + 1][tm]);
                else put8<OT>(p.C, at + tp * 32, acc[2 * tp][tm] * scale, acc[2 * tp + 1][tm] * scale);
            }
        }
    };
    if (vec_ok && (SPLIT || p.beta == 0.f)) {
        if (SPLIT || p.out_type == OUT_BF16) emit_whole(std::integral_constant<int, OUT_BF16>{});
        else if (p.out_type == OUT_F32) emit_whole(std::integral_constant<int, OUT_F32>{});
        else if (p.out_type == OUT_F8) emit_whole(std::integral_constant<int, OUT_F8>{});
        else emit_whole(std::integral_constant<int, OUT_F16>{});
        return;
    }
    auto emit = [&](auto type_tag) {
        constexpr int OT = decltype(type_tag)::value;
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
            const int rt = (tm * WGM + wm) * 16 + li;
#pragma unroll
            for (int tp = 0; tp < TN / 2; ++tp) {
                const int col = n0 + wn * WTN + tp * 32 + pair_col;
                if (rt >= rows_valid || col >= p.N) continue;
                if constexpr (SPLIT)
                    store8(p.partials + (int64_t)blockIdx.y * MN, OUT_F32, m0 + rt, col, p.N, p.N, acc[2 * tp][tm], acc[2 * tp + 1][tm], 0.f, vec_ok);
                else
                    store8(p.C, OT, m0 + rt, col, p.N, p.ldc, acc[2 * tp][tm] * scale, acc[2 * tp + 1][tm] * scale, p.beta, vec_ok);
            }
        }
    };
    if (SPLIT || p.out_type == OUT_BF16) emit(std::integral_constant<int, OUT_BF16>{});
    else if (p.out_type == OUT_F32) emit(std::integral_constant<int, OUT_F32>{});
    else if (p.out_type == OUT_F8) emit(std::integral_constant<int, OUT_F8>{});
    else emit(std::integral_constant<int, OUT_F16>{});
#endif
}

template <int BM, int BN, int STAGES, bool BLOCKSCALE, bool KN = false>
inline hipError_t launch_tile_ring(bool split, const GemmParams& p, int gx, int gy, hipStream_t stream) {
    if (split) hipLaunchKernelGGL((fp8_gemm_tile_ring_kernel<BM, BN, STAGES, BLOCKSCALE, true, KN, false>), dim3(gx, gy, 1), dim3(512, 1, 1), 0, stream, p);
    else hipLaunchKernelGGL((fp8_gemm_tile_ring_kernel<BM, BN, STAGES, BLOCKSCALE, false, KN, false>), dim3(gx, gy, 1), dim3(512, 1, 1), 0, stream, p);
    return hipGetLastError();
}

template <int BM, int BN, int STAGES, bool BLOCKSCALE>
inline hipError_t launch_tile_ring_once(const GemmParams& p, int gx, hipStream_t stream) {
    hipLaunchKernelGGL((fp8_gemm_tile_ring_kernel<BM, BN, STAGES, BLOCKSCALE, false, false, true>), dim3(gx, 1, 1), dim3(512, 1, 1), 0, stream, p);
    return hipGetLastError();
}

}  // namespace tg
