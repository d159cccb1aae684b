// Expert-grouped block-scaled GEMMs while the experts' weights stream from memory: tiles of 32, 64 or 128 rows x 128, 192 or 256 weight
// rows, one persistent workgroup per compute unit (ragged segments, token gather, and gather with the SiLU-multiply-quantize
// epilogue).
//
// With up to about a hundred rows per expert a tile's K step multiplies for less time than its weights take to arrive at the
// rate a compute unit gets from memory (25 GB/s: 1.3 us for 256 weight rows x 128 bytes), so what counts is that the requests
// never stop.  The kernels of one workgroup per tile stop them at every tile: 3 to 4 us of set-up (expert, row map, scale table, first
// loads) and the epilogue, and a last round that leaves compute units idle (704 tiles over 512 places).  Here four waves only
// load, as in fp8_gemm_tile_ring.h, and the ring of LDS stages runs on from one tile to the next: the first K steps of the next tile are
// requested while this one's last steps are multiplied and its results are stored.  The computing waves fetch the next tile's
// expert and row map behind their first K step and leave them in LDS, where the loading waves find them STAGES steps before the
// tile's end (so K has at least five steps with 256 columns, eight with 128).  A workgroup's tiles all lie in its XCD's share of the tile sequence.
//
// Activation scales travel with the slabs: a chunk of eight K steps is requested right in front of the slab of its first step, into
// one of three chunk buffers (two would be enough but for last chunks shorter than the ring: the next tile's first chunk is
// then requested while the one before the last is read).  Weight scales are scalar loads, one
// step ahead.  Rows that a tile does not have are requested from beyond the descriptor's range: no memory request.
//
// Eight computing waves for 256 columns (four of 64 x 128 were no faster than the kernels of one workgroup per tile: two waves on a SIMD take
// turns at the scale-and-add), non-temporal weight loads (8 - 11 % over plain ones), 192 columns where 256 would leave a round half empty
// (32 experts of (1536, 4096): 46 us with 256, 43.7 with 192).  Rows that are not spread evenly: a crowded expert's row tiles go over the same
// columns one after the other, and the columns of a tile are chosen on the device.  Over 3900 problems ahead of the kernels of one
// workgroup per tile by 1.12 x with the rows spread evenly, 1.17 on an eighth of the experts, 1.12 with half and 1.19 with all of them on one, 1.11 by
// Zipf's law (without the two 1.13, 1.07, 1.08, 1.02, 1.09); it stays behind where few experts have hundreds of rows each and the mean
// says 30 (120 experts of (2304, 2560), 5032 rows on 15 of them: 96 us, pairs of 128 x 256 tiles 47).  Measured, us before / after (floor at 6.5 TB/s), 64 experts of (2816, 2048)
// top 6: 40 tokens 61.6 / 56.8 (56.0), 200 tokens 65.2 / 61.7 (58.2), 1000 tokens 87.0 / 80.8 (64.0); 128 experts of (1536, 2048) top 8:
// 8 tokens 38.8 / 31.1 (25.0), 1000 tokens 94.1 / 81.8 (68.3); 16 experts of (2048, 2048) top 2: 40 tokens 17.4 / 14.0 (10.4).  A layer of
// the first size (align, quantize, two GEMMs, sum): 200 tokens 122 / 108.
//
// Same slab layout, fragment addressing, arithmetic per accumulator and epilogue as fp8_gemm_tile.h: identical results.
#pragma once

#include "fp8_gemm_tile.h"

namespace tg {

constexpr int kGroupedRingExperts = 256;  // ragged: experts whose tile counts fit in LDS

__device__ __forceinline__ float uniform_f32(const float* p) { return *(const __attribute__((address_space(4))) float*)(uintptr_t)p; }

template <int BM, int BN, int STAGES, int NC, int GROUP>
__global__ void __launch_bounds__(64 * (NC + 4), 1) fp8_gemm_grouped_ring_kernel(const GemmParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr bool ACT = GROUP == GROUP_GATHER_ACT;
    constexpr int WGM = 2, WGN = NC / 2, NL = 4;  // NC computing waves, four loading waves
    constexpr int WTN = BN / WGN;
    constexpr int TM = BM / (16 * WGM), TN = WTN / 16;
    constexpr int A_IT = BM / (8 * NL), B_IT = BN / (8 * NL);
    constexpr int STAGE_BYTES = (BM + BN) * kKBlock;
    constexpr int PER_STEP = A_IT + B_IT;
    constexpr int LAST = 2, HEAD = (TN - LAST) * TM;  // column tiles behind a step's barrier, MFMAs in front of it
    constexpr int CHUNK = BM * kScaleChunk;           // floats of a chunk of activation scales
    static_assert(STAGES + 2 <= (BN == 256 ? 5 : 8), "grouped_ring_steps");
    static_assert((TN == 4 || TN == 8) && (!ACT || BN == 256), "column tiles: four weight fragment sets rotate");

    __shared__ __align__(1024) uint8_t lds[STAGES * STAGE_BYTES];  // stage s: A slab, then B slab
    __shared__ __align__(256) float s_as[3 * CHUNK];
    __shared__ int s_dst[2][BM];                 // of this tile and the next: output row (-1: none)
    __shared__ int s_tile[2][2];                 // expert, first column
    __shared__ int s_end[GROUP == GROUP_RAGGED ? kGroupedRingExperts : 1];  // row tiles of the experts up to and with e
    __shared__ float s_amax[ACT ? WGN * BM : 1];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = p.K, nsteps = p.kblocks;
    // ---- the workgroup's tiles: first, first + stride, ... of its XCD's range.  Columns of a tile: BN, or fewer so that the tiles come out
    // even over the compute units; the weight rows that a tile leaves out are requested from beyond the descriptor's range (no memory request)
    // and not stored.
    int post_pad = 0, total_mt;
    if constexpr (GROUP == GROUP_RAGGED) {
        int base = 0;
        for (int e0 = 0; e0 < p.E; e0 += 64) {
            const int e = e0 + lane;
            int incl = 0;
            if (e < p.E) {
                const int rows = p.m_indptr[e + 1] - p.m_indptr[e];
                incl = rows > 0 ? (rows + BM - 1) / BM : 0;
            }
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int t = __shfl_up(incl, d);
                if (lane >= d) incl += t;
            }
            incl += base;
            if (wave == 0 && e < p.E) s_end[e] = incl;
            base = __shfl(incl, 63);
        }
        total_mt = min(base, p.M / BM + p.E);  // (no more row tiles than M rows in E segments can have, whatever m_indptr holds)
        __syncthreads();
    } else {
        post_pad = min(p.num_post_pad[0], p.em_capacity);
        total_mt = (post_pad + BM - 1) / BM;
    }
    total_mt = __builtin_amdgcn_readfirstlane(total_mt);
    int cols = ACT ? 128 : p.tile_cols;
    if constexpr (BN == 256 && !ACT) {
        // tile_cols 0: by the rounds that the tiles make (a round costs its columns + 16).  Decided here, where the row tiles are known: an
        // expert with more rows than the others is a tile or two more, and those may be a round more.
        if (cols == 0) {
            const float places = __builtin_amdgcn_rcpf((float)gridDim.x);  // (an integer division would delay the first loads by 0.2 us)
            float best = 1e30f;
#pragma unroll
            for (int c = 256; c >= (BM == 128 ? 192 : 128); c -= 64) {
                const float cost = __builtin_ceilf((float)(total_mt * ((p.N + c - 1) / c)) * places - 1e-3f) * (float)(c + 16);
                if (cost < best) { best = cost; cols = c; }
            }
        }
    }
    const int tiles_n = ACT ? p.inter / 128 : (p.N + cols - 1) / cols;
    const int nblk = total_mt * tiles_n;
    const int xcd = blockIdx.x % 8, stride = gridDim.x / 8;  // (the grid is a multiple of eight)
    const int share = nblk / 8, rest = nblk % 8;
    const int first = xcd * share + min(xcd, rest) + (int)blockIdx.x / 8;
    const int end = xcd * share + min(xcd, rest) + share + (xcd < rest ? 1 : 0);
    const int ntiles = first < end ? (end - first - 1) / stride + 1 : 0;
    if (ntiles == 0) return;
    const int total_steps = ntiles * nsteps;

    // ---- a tile's expert, first column and rows.  find() requests what publish() looks at two K steps later: nothing in between waits.
    struct Tile { int expert, n0, lo, hi; };  // lo, hi: ragged, the thread's row and the end of the expert's; gather, the thread's slot
    auto find = [&](int i) {
        const int t = first + i * stride;
        const int tile_m = t / tiles_n;
        int tile_n = t % tiles_n;
        Tile f;
        f.lo = f.hi = 0;
        if constexpr (GROUP == GROUP_RAGGED) {
            int e = 0, before = 0, upto = 0;  // row tiles in front of the expert, and with it
            for (int e0 = 0; e0 < p.E; e0 += 64) {
                const int ends = e0 + lane < p.E ? s_end[e0 + lane] : 0x7FFFFFFF;
                const unsigned long long hit = __ballot(ends > tile_m);
                if (hit) {
                    const int l = __builtin_amdgcn_readfirstlane(__ffsll((long long)hit) - 1);
                    e = e0 + l;
                    upto = __builtin_amdgcn_readlane(ends, l);
                    if (l > 0) before = __builtin_amdgcn_readlane(ends, l - 1);
                    break;
                }
                before = __builtin_amdgcn_readlane(ends, 63);
            }
            // a crowded expert's row tiles one after the other over the same columns: the compute units of an XCD that work on it at one time
            // share its weight in their L2 (with two row tiles the weight is read once more either way, and column by column is 0.8 % ahead)
            const int mine = upto - before;
            int row_tile = tile_m - before;
            if (mine > 2) {
                const int at = t - before * tiles_n;
                tile_n = at / mine;
                row_tile = at - tile_n * mine;
            }
            f.expert = e;
            f.lo = p.m_indptr[e] + row_tile * BM + tid;
            f.hi = p.m_indptr[e + 1];
        } else {
            const int m0 = tile_m * BM;  // position in the sorted slot sequence
            f.expert = p.expert_ids[m0 / p.block_m];
            f.lo = tid < BM && m0 + tid < post_pad ? p.sorted_ids[m0 + tid] : p.num_valid;
        }
        f.n0 = tile_n * cols;
        return f;
    };
    auto publish = [&](Tile& f, int buf) {
        const bool known = f.expert >= 0 && f.expert < p.E;  // (else nothing is stored)
        if (tid < BM) {
            bool ok;
            if constexpr (GROUP == GROUP_RAGGED) ok = f.lo >= 0 && f.lo < min(f.hi, p.M);
            else ok = known && f.lo >= 0 && f.lo < p.num_valid;
            s_dst[buf][tid] = ok ? f.lo : -1;
        }
        if (!known) f.expert = 0;
        if (tid == 0) {
            s_tile[buf][0] = f.expert;
            s_tile[buf][1] = f.n0;
        }
    };

    constexpr int kPro = (STAGES - 1) * PER_STEP, kLoop = (STAGES - 2) * PER_STEP;  // slab loads that may stay in flight
    static_assert(kPro < 64, "vmcnt has six bits");
    constexpr int kWaitPro = 0x0F70 | (kPro & 15) | ((kPro >> 4) << 14);
    constexpr int kWaitLoop = 0x0F70 | (kLoop & 15) | ((kLoop >> 4) << 14);
    constexpr int kWaitAll = 0x0F70;
    constexpr int kWaitLds = 0xC07F;
#define TG_FENCE() __builtin_amdgcn_sched_barrier(0)

    if (wave >= NC) {
        // ------------------------------------------------------------ loading waves
        const int lw = wave - NC;
        const int lrow = lane >> 3;
        const int lj = (lane & 7) ^ swz16(lrow);
        const int ljb = (lane & 7) ^ swz_w(((lw & 1) << 3) | lrow);
        const int s_kbi = ((lane & 7) - lrow) & 7;    // chunk step this lane fetches
        const v4i rsrc_a = make_rsrc(p.A), rsrc_s = make_rsrc(p.As);
        const uint32_t lds0 = lds_address(lds) + lw * 1024, as0 = lds_address(s_as) + lw * 256;
        uint32_t a_off[A_IT], s_off[A_IT], b_off[B_IT];
        v4i rsrc_b;
        auto enter = [&](int buf) {  // the tile whose steps are requested from now on
            const int expert = __builtin_amdgcn_readfirstlane(s_tile[buf][0]), n0 = __builtin_amdgcn_readfirstlane(s_tile[buf][1]);
            rsrc_b = make_rsrc(p.B + (int64_t)expert * p.N * K);
#pragma unroll
            for (int i = 0; i < A_IT; ++i) {
                const int dst = s_dst[buf][(i * NL + lw) * 8 + lrow];
                const int src = GROUP == GROUP_RAGGED ? dst : dst / p.top_k;
                a_off[i] = dst < 0 ? 0x80000000u : (uint32_t)src * (uint32_t)K + lj * 16;
                s_off[i] = dst < 0 ? 0x80000000u : (uint32_t)src * (uint32_t)p.kblocks * 4u;
            }
#pragma unroll
            for (int i = 0; i < B_IT; ++i) {
                const int br = (i * NL + lw) * 8 + lrow;
                const int n = ACT ? ((br % WTN) / (WTN / 2)) * p.inter + n0 + (br / WTN) * (WTN / 2) + br % (WTN / 2) : min(n0 + br, p.N - 1);
                b_off[i] = !ACT && br >= cols ? 0x80000000u : (uint32_t)n * (uint32_t)K + ljb * 16;
            }
        };
        int chunk = 0;  // of three buffers
        auto issue = [&](int kstep, int stage, bool past) {  // past: a step that was requested already
            const int k0 = kstep * kKBlock;
            const uint32_t dst = lds0 + stage * STAGE_BYTES;
            if (kstep % kScaleChunk == 0 && !past) {
                const uint32_t kb = (uint32_t)min(kstep + s_kbi, nsteps - 1) * 4u;
#pragma unroll
                for (int i = 0; i < A_IT; ++i) direct_load_b32(rsrc_s, as0 + chunk * (CHUNK * 4) + i * NL * 256, s_off[i] + kb, 0);
                chunk = chunk == 2 ? 0 : chunk + 1;
            }
#pragma unroll
            for (int i = 0; i < B_IT; ++i) direct_load_b128_nt(rsrc_b, dst + BM * kKBlock + i * NL * 1024, b_off[i], k0);
#pragma unroll
            for (int i = 0; i < A_IT; ++i) direct_load_b128(rsrc_a, dst + i * NL * 1024, a_off[i], k0);
        };
        __builtin_amdgcn_s_barrier();  // the first tile's rows are in LDS
        enter(0);
#pragma unroll
        for (int s = 0; s < STAGES; ++s) issue(s, s, false);
        __builtin_amdgcn_s_waitcnt(kWaitPro);
        __builtin_amdgcn_s_barrier();
        int stage = 0, ahead = STAGES, tile = 0, k = 0;  // `ahead`: the step of the tile entered last that is requested next
        for (int g = 0; g < total_steps; ++g) {
            __builtin_amdgcn_s_waitcnt(kWaitLoop);  // step g+1 has landed
            __builtin_amdgcn_s_barrier();           // and every computing wave has read step g
            if (ahead == nsteps && tile + 1 < ntiles) {
                ahead = 0;
                ++tile;
                enter(tile & 1);
            }
            issue(min(ahead, nsteps - 1), stage, ahead == nsteps);  // (steps past the end re-fetch the last one)
            ahead = min(ahead + 1, nsteps);
            stage = stage == STAGES - 1 ? 0 : stage + 1;
            if constexpr (ACT) {
                if (++k == nsteps) {  // the epilogue's exchange of row maxima
                    k = 0;
                    __builtin_amdgcn_s_barrier();
                }
            }
        }
        __builtin_amdgcn_s_waitcnt(kWaitAll);  // the re-fetches past the end must land before the workgroup's LDS is released
        return;
    }

    // ---------------------------------------------------------------- computing waves
    const int wm = wave % WGM, wn = wave / WGM;
    const int li = lane & 15, lg = lane >> 4;
    const uint32_t frag0 = wm * 16 * kKBlock + li * kKBlock + ((lg ^ swz16(li)) << 4), frag1 = frag0 ^ 64;
    const int wrow = ((li >> 2) << 3) | (li & 3);
    const uint32_t wfrag0 = BM * kKBlock + wn * WTN * kKBlock + wrow * kKBlock + ((lg ^ swz_w(wrow)) << 4), wfrag1 = wfrag0 ^ 64;

    v4f acc[TN][TM];
    v8i af[TM], wf[4];
    auto read_a = [&](int tm, const uint8_t* base) {
        const uint8_t* a = base + tm * (WGM * 16 * kKBlock);
        af[tm] = join(*reinterpret_cast<const v4i*>(a + frag0), *reinterpret_cast<const v4i*>(a + frag1));
    };
    auto read_w = [&](int tn, const uint8_t* base) {
        const uint8_t* b = base + ((tn >> 1) * 32 + (tn & 1) * 4) * kKBlock;
        wf[tn % 4] = join(*reinterpret_cast<const v4i*>(b + wfrag0), *reinterpret_cast<const v4i*>(b + wfrag1));
    };
    // weight scales of a tile: the wave's columns, or gate and up columns
    auto scale_row = [&](int expert, int n0, int up) {
        const int nb = ACT ? (up * p.inter + n0) / 128 : min((n0 + wn * WTN) / 128, p.nblocks - 1);
        return p.Bs + ((int64_t)expert * p.nblocks + nb) * p.kblocks;
    };
    // scales of the coming step
    float as_n[TM], bs_n, bs_up_n = 0.f;
    const int s_rbase = (wm * 2 + (li >> 3)) * 64 + (li & 7) * 8;
    auto read_scales = [&](int k, int chunk) {
        const float* cs = s_as + chunk * CHUNK + s_rbase + (((k % kScaleChunk) + li) & 7);
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) as_n[tm] = cs[tm * (WGM * 128)];
    };

    Tile now = find(0);
    publish(now, 0);
    int expert = __builtin_amdgcn_readfirstlane(now.expert);
    const float *bs = scale_row(expert, now.n0, 0), *bs_up = scale_row(expert, now.n0, 1);
    int n0 = now.n0;
    __builtin_amdgcn_s_waitcnt(kWaitLds);
    __builtin_amdgcn_s_barrier();  // the first tile's rows are in LDS
    bs_n = uniform_f32(bs);
    if constexpr (ACT) bs_up_n = uniform_f32(bs_up);
    __builtin_amdgcn_s_barrier();  // step 0 has landed
    read_w(0, lds);
    read_w(1, lds);
    read_scales(0, 0);
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) read_a(tm, lds);

    int stage = 0, chunk = 0;
    for (int i = 0; i < ntiles; ++i) {
        int dst[TM];
        float rw[TM];
        // (worked out per tile: kept over the loop, the address is the one register too many of the 128 x 256 activation form)
        int here = lane;
        if constexpr (ACT && BM == 128) asm volatile("" : "+v"(here));
        const int row0 = wm * 16 + (here & 15);
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
            dst[tm] = s_dst[i & 1][tm * (WGM * 16) + row0];
            rw[tm] = 1.0f;
            if constexpr (GROUP == GROUP_GATHER)
                if (p.row_weight && dst[tm] >= 0) rw[tm] = p.row_weight[dst[tm]];
        }
        Tile next{0, 0, -1, 0};
        if (i + 1 < ntiles) next = find(i + 1);
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
#pragma unroll
            for (int tm = 0; tm < TM; ++tm) acc[tn][tm] = v4f{0.f, 0.f, 0.f, 0.f};
        const float *bs_next = bs, *bs_up_next = bs_up;
        int k = 0;
        for (int part = 0; part < 2; ++part) {
            for (const int stop = part == 0 ? 2 : nsteps; k < stop; ++k) {
                const uint8_t* cur = lds + stage * STAGE_BYTES;
                stage = stage == STAGES - 1 ? 0 : stage + 1;
                const uint8_t* nxt = lds + stage * STAGE_BYTES;
                // one MFMA into a fresh product, and behind it the scale-and-add of the product issued two MFMAs before (see
                // fp8_gemm_tile.h)
                v4f part_sum[3];
                float sc[TM], sc_up[ACT ? TM : 1];
#pragma unroll
                for (int tm = 0; tm < TM; ++tm) {
                    sc[tm] = as_n[tm] * bs_n;
                    if constexpr (ACT) sc_up[tm] = as_n[tm] * bs_up_n;
                }
                auto tn_of = [](int j) constexpr { return j < HEAD ? j / TM : TN - LAST + (j - HEAD) % LAST; };
                auto tm_of = [](int j) constexpr { return j < HEAD ? j % TM : (j - HEAD) / LAST; };
                auto add = [&](int j) __attribute__((always_inline)) {
                    if (j < 0) return;
                    float s;
                    if constexpr (ACT) s = tn_of(j) >= TN / 2 ? sc_up[tm_of(j)] : sc[tm_of(j)];
                    else s = sc[tm_of(j)];
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[tn_of(j)][tm_of(j)][r] = __builtin_fmaf(part_sum[j % 3][r], s, acc[tn_of(j)][tm_of(j)][r]);
                };
                auto mma = [&](int j) __attribute__((always_inline)) {
                    part_sum[j % 3] = mfma_e4m3(wf[tn_of(j) % 4], af[tm_of(j)], v4f{0.f, 0.f, 0.f, 0.f});
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
                const bool over = k + 1 == nsteps;     // the coming step is the next tile's first
                const int kn = over ? 0 : k + 1;
                if (kn % kScaleChunk == 0) chunk = chunk == 2 ? 0 : chunk + 1;
                read_w(0, nxt);
                read_w(1, nxt);
                read_scales(kn, chunk);
                bs_n = uniform_f32(over ? bs_next : bs + kn);
                if constexpr (ACT) bs_up_n = uniform_f32(over ? bs_up_next : bs_up + kn);
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
                add(TN * TM - 2);
                add(TN * TM - 1);
                // keep the scale-and-add chain inside this step (see fp8_gemm_tile.h)
#pragma unroll
                for (int tn = 0; tn < TN; ++tn)
#pragma unroll
                    for (int tm = 0; tm < TM; ++tm) asm volatile("" : "+v"(acc[tn][tm]));
            }
            if (part == 0 && i + 1 < ntiles) {
                // the next tile's rows have arrived; the loading waves read them behind a later barrier
                publish(next, (i + 1) & 1);
                expert = __builtin_amdgcn_readfirstlane(next.expert);
                bs_next = scale_row(expert, next.n0, 0);
                bs_up_next = scale_row(expert, next.n0, 1);
            }
        }

        // ---- results
        if constexpr (ACT) {
            // gate columns in column tiles 0 ... TN/2 - 1, the matching up columns in the others: as in fp8_gemm_tile.h
            float actv[TM][TN / 4][8];
            auto activate = [&](auto type_tag) {
                using T = decltype(type_tag);
#pragma unroll
                for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                    for (int tp = 0; tp < TN / 4; ++tp)
#pragma unroll
                        for (int q = 0; q < 8; ++q) {
                            const float ga = acc[2 * tp + (q >> 2)][tm][q & 3], ua = acc[TN / 2 + 2 * tp + (q >> 2)][tm][q & 3];
                            actv[tm][tp][q] = silu_mul_round<T>((float)(T)ga, (float)(T)ua);
                        }
            };
            if (p.act_is_bf16) activate(__bf16{});
            else activate(_Float16{});
#pragma unroll
            for (int tm = 0; tm < TM; ++tm) {
                float amax = 0.f;
#pragma unroll
                for (int tp = 0; tp < TN / 4; ++tp)
#pragma unroll
                    for (int q = 0; q < 8; ++q) amax = fmaxf(amax, fabsf(actv[tm][tp][q]));
                amax = fmaxf(amax, __shfl_xor(amax, 16));
                amax = fmaxf(amax, __shfl_xor(amax, 32));
                if (lg == 0) s_amax[wn * BM + (tm * WGM + wm) * 16 + li] = amax;
            }
            __builtin_amdgcn_s_waitcnt(kWaitLds);
            __builtin_amdgcn_s_barrier();
            uint8_t* const qout = reinterpret_cast<uint8_t*>(p.C);
#pragma unroll
            for (int tm = 0; tm < TM; ++tm) {
                const int rt = (tm * WGM + wm) * 16 + li;
                float amax = s_amax[rt];
#pragma unroll
                for (int w = 1; w < WGN; ++w) amax = fmaxf(amax, s_amax[w * BM + rt]);
                const float sc1 = amax == 0.f ? 1.0f : amax / 448.0f;
                if (dst[tm] < 0) continue;
                const ScaleDivider div(sc1);
                if (div.fast) {
#pragma unroll
                    for (int tp = 0; tp < TN / 4; ++tp)
#pragma unroll
                        for (int q = 0; q < 8; ++q) actv[tm][tp][q] = div.quotient(actv[tm][tp][q]);
                } else {
#pragma unroll
                    for (int tp = 0; tp < TN / 4; ++tp)
#pragma unroll
                        for (int q = 0; q < 8; ++q) actv[tm][tp][q] = actv[tm][tp][q] / sc1;
                }
#pragma unroll
                for (int tp = 0; tp < TN / 4; ++tp) {
                    int packed[2];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        float c[4];
#pragma unroll
                        for (int q = 0; q < 4; ++q) c[q] = fminf(fmaxf(actv[tm][tp][4 * h + q], -448.0f), 448.0f);
                        int w = 0;
                        w = __builtin_amdgcn_cvt_pk_fp8_f32(c[0], c[1], w, false);
                        w = __builtin_amdgcn_cvt_pk_fp8_f32(c[2], c[3], w, true);
                        packed[h] = w;
                    }
                    *reinterpret_cast<v2i*>(qout + (int64_t)dst[tm] * p.inter + n0 + wn * (WTN / 2) + tp * 32 + lg * 8) = v2i{packed[0], packed[1]};
                }
                if (wn == 0 && lg == 0) p.act_scales[(int64_t)dst[tm] * (p.inter / 128) + n0 / 128] = sc1;
            }
        } else {
            const bool vec_ok = p.vec_store != 0 && (p.N % 8) == 0;
            const int n_end = min(n0 + cols, p.N);
            auto emit = [&](auto type_tag, auto whole_tag) __attribute__((always_inline)) {
                constexpr int OT = decltype(type_tag)::value;
#pragma unroll
                for (int tm = 0; tm < TM; ++tm) {
                    if (dst[tm] < 0) continue;
#pragma unroll
                    for (int tp = 0; tp < TN / 2; ++tp) {
                        const int col = n0 + wn * WTN + tp * 32 + lg * 8;
                        if (col >= n_end) continue;
                        const v4f lo = acc[2 * tp][tm] * rw[tm], hi = acc[2 * tp + 1][tm] * rw[tm];
                        if constexpr (decltype(whole_tag)::value) put8<OT>(p.C, (int64_t)dst[tm] * p.ldc + col, lo, hi);
                        else store8(p.C, OT, dst[tm], col, n_end, p.ldc, lo, hi, 0.f, false);
                    }
                }
            };
            auto emit_type = [&](auto whole_tag) {
                if (p.out_type == OUT_BF16) emit(std::integral_constant<int, OUT_BF16>{}, whole_tag);
                else if (p.out_type == OUT_F32) emit(std::integral_constant<int, OUT_F32>{}, whole_tag);
                else if (p.out_type == OUT_F8) emit(std::integral_constant<int, OUT_F8>{}, whole_tag);
                else emit(std::integral_constant<int, OUT_F16>{}, whole_tag);
            };
            if (vec_ok) emit_type(std::integral_constant<bool, true>{});
            else emit_type(std::integral_constant<bool, false>{});
        }
        n0 = next.n0;
        bs = bs_next;
        bs_up = bs_up_next;
    }
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) asm volatile("" : : "v"(af[tm]));
    asm volatile("" : : "v"(wf[0]), "v"(wf[1]));
#undef TG_FENCE
#endif
}

template <int BM, int BN, int STAGES, int NC, int GROUP>
inline hipError_t launch_grouped_ring(const GemmParams& p, int grid, hipStream_t stream) {
    hipLaunchKernelGGL((fp8_gemm_grouped_ring_kernel<BM, BN, STAGES, NC, GROUP>), dim3(grid, 1, 1), dim3(64 * (NC + 4), 1, 1), 0, stream, p);
    return hipGetLastError();
}

}  // namespace tg
