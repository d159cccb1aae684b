// The FP8 MoE layer for a handful of rows per expert (decoding): two or three launches that stream the weights of the
// experts that have rows once each.
//
//   moe_decode_kernel<.., true>    x (16-bit) -> quantize 1 x 128 -> w1 -> T(silu(gate) * up), stored as 16-bit values
//   moe_decode_kernel<.., false>   those -> quantize 1 x 128 -> w2 -> x routed weight, one row per (token, slot)
//   moe_decode_sum_kernel          the same and the sum over a token's slots in one launch, for very few slots
//
// Bound by the experts' weights out of HBM, 5.8 + 2.9 MB per expert at (hidden, inter) = (2048, 1408), and at one or two
// tokens by the latency of the launches in a row.  Whole layer, 64 experts, top 6 (row-tiled form in brackets): 1 token 16.1 us
// (35.0), 16 tokens 75 (114), 40 tokens 95 (122), 64 tokens 99 (124); at 40 tokens the first GEMM reads its weights at
// 6.0 TB/s.  The row-tiled form of the layer pads every expert to 128 rows, needs
// moe_align and the quantizer in front and a sum behind, and leaves half of the chip without weights in flight.  Here:
//   * No alignment launch.  The routing is a few hundred ids: every workgroup reads them all, counts the rows of every
//     expert in LDS and takes an equal share of (expert, pass, group of columns) units -- contiguous, so that a workgroup
//     meets one or two experts.  A pass is as many rows as are held at a time; an expert with more is streamed once per
//     pass, and the passes are dealt like experts.  Every compute unit then takes in the same number of weight bytes whatever
//     the routing is, which is what bounds the launch (24 bytes per nanosecond and compute unit at 40 tokens).
//   * No quantizer launch.  Four waves of a workgroup quantize the rows of its expert (a few rows; they come out of the L2)
//     into LDS, in MFMA order, with the scales beside them, while the first weights are on their way to the others.
//     The arithmetic is the quantizer's: the same bits.
//   * A streaming wave owns 16 weight rows at a time over the whole K and a private ring of pieces (16 rows x 512 bytes of K), all in
//     flight: it waits for its own loads only, reads a piece's fragments, requests the next piece into the same place
//     and multiplies.  No barrier in the loop; the ring runs on from one group of rows to the next.
//   * In the first GEMM the 16 rows are 8 gate rows and the 8 up rows of the same columns, dealt so that a lane's four
//     results are two gate / up pairs.
// K blocks are added in ascending order with one fused multiply-add each, as in the row-tiled kernels: identical bits.
//
// Weight rows of an expert: N * K < 2^31 (32-bit offsets); K % 128 == 0.
#pragma once

#include "fp8_gemm_tile.h"
#include "tg_host.h"

namespace tg {

constexpr int kDecodePiece = 512;                  // bytes of K of one row in a piece: four K steps
constexpr int kDecodeSteps = kDecodePiece / kKBlock;
constexpr int kDecodeBuf = 16 * kDecodePiece;      // 8 KiB
constexpr uint32_t kDecodeOutOfRange = 0x80000000u;  // >= the descriptors' 2^31 - 1 bytes: no request, zeros

// 16 bytes per lane from a buffer into registers.  The caller orders its use behind a vmcnt wait by hand, so that the
// direct loads requested after it may stay in flight (the compiler's own wait would drain them).
__device__ __forceinline__ v4i buffer_load_b128_raw(v4i rsrc, uint32_t voffset) {
    v4i r;
    asm volatile("s_nop 4\n\tbuffer_load_dwordx4 %0, %1, %2, 0 offen" : "=v"(r) : "v"(voffset), "s"(rsrc) : "memory");
    return r;
}
__device__ __forceinline__ float buffer_load_f32_raw(v4i rsrc, uint32_t voffset) {
    float r;
    asm volatile("s_nop 4\n\tbuffer_load_dword %0, %1, %2, 0 offen" : "=v"(r) : "v"(voffset), "s"(rsrc) : "memory");
    return r;
}
// Every wave's LDS accesses are done, direct loads stay in flight.
__device__ __forceinline__ void decode_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt field");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// Maximum over the 16 lanes of a DPP row, in every one of them (four rotations; a shuffle would go through the LDS crossbar).
__device__ __forceinline__ float row16_max(float x) {
    x = fmaxf(x, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x128, 0xF, 0xF, false)));  // row_ror:8
    x = fmaxf(x, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x124, 0xF, 0xF, false)));
    x = fmaxf(x, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x122, 0xF, 0xF, false)));
    x = fmaxf(x, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x121, 0xF, 0xF, false)));
    return x;
}

// Eight values of one 128-element group (16 lanes hold one) -> their e4m3 codes and the group's scale: scale = amax / 448,
// 1 for an all-zero group, codes = e4m3(x / scale): act_quant_group_kernel's rule 0.
template <typename T>
__device__ __forceinline__ v2i quantize_lane(v4i raw, float* scale_out) {
    typedef T vecT __attribute__((ext_vector_type(8)));
    typedef float vecF __attribute__((ext_vector_type(8)));
    const vecF v = __builtin_convertvector(__builtin_bit_cast(vecT, raw), vecF);
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(v[i]));
    amax = row16_max(amax);
    const float s = amax == 0.f ? 1.0f : amax / 448.0f;
    const ScaleDivider div(s);
    float c[8];
    if (div.fast) {
#pragma unroll
        for (int i = 0; i < 8; ++i) c[i] = div.quotient(v[i]);
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) c[i] = v[i] / s;
    }
    int packed[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        float q[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) q[i] = fminf(fmaxf(c[4 * h + i], -448.0f), 448.0f);
        int w = 0;
        w = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], w, false);
        w = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], w, true);
        packed[h] = w;
    }
    *scale_out = s;
    return v2i{packed[0], packed[1]};
}

__device__ __forceinline__ int decode_expert_id(const MoeDecodeParams& p, int slot) {
    // (ids past the int32 range are no experts either way)
    if (p.ids_are_i64) {
        const long long id = reinterpret_cast<const long long*>(p.ids)[slot];
        return id >= 0 && id < p.E ? (int)id : -1;
    }
    const int id = reinterpret_cast<const int*>(p.ids)[slot];
    return id >= 0 && id < p.E ? id : -1;
}

// Waves of a workgroup: those that stream the weights, with the pieces in flight of each, and those that prepare the
// activations.  (Pieces in flight, 80 KiB per compute unit, cover the latency of HBM at its full rate; one token, first
// GEMM: 12.4 / 11.6 / 10.7 us with 4 waves x 3 pieces, 4 x 2 and 5 x 2 -- a workgroup's share is five groups there, one per
// wave; 40 tokens: 59.4 / 60.1 / 60.2.)
constexpr int kDecodeWaves = 5, kDecodeStages = 2, kDecodeQuantWaves = 4;

// LDS of a compute unit.  The kernels below have no static LDS: a static variable in front of the 1024-byte aligned dynamic
// array would take 1 KiB of it, whatever its size (the build check holds them to that).
constexpr int kLdsBytes = 160 * 1024;

// Dynamic LDS of moe_decode_kernel, in this order.
struct MoeDecodeLds {
    int ring, codes, scales, wscales, ids, list, weight, count, rows, total;  // byte offsets
    __host__ __device__ static MoeDecodeLds of(const MoeDecodeParams& p) {
        MoeDecodeLds l{};
        l.ring = 0;
        l.codes = kDecodeWaves * kDecodeStages * kDecodeBuf;
        l.scales = l.codes + p.row_cap * p.K;
        l.wscales = l.scales + (p.row_cap * p.kblocks * 4 + 255) / 256 * 256;
        l.ids = l.wscales + p.wscale_cap * 4;
        l.list = l.ids + p.slots * 2;
        l.weight = l.list + p.slots * 2;
        l.count = l.weight + p.slots * 4;
        l.rows = l.count + (p.E + 1) / 2 * 4;
        l.total = l.rows + 4;
        return l;
    }
};

template <typename T, bool UP>
__global__ void __launch_bounds__(64 * (kDecodeWaves + kDecodeQuantWaves)) moe_decode_kernel(const MoeDecodeParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int NW = kDecodeWaves, STAGES = kDecodeStages, NT = 64 * (NW + kDecodeQuantWaves), NTQ = 64 * kDecodeQuantWaves;
    constexpr int COLS = UP ? 8 : 16;           // output columns of a group of 16 weight rows
    constexpr int LOADS = kDecodeBuf / 1024;    // direct loads of a piece
    extern __shared__ __align__(1024) uint8_t lds[];
    const MoeDecodeLds at = MoeDecodeLds::of(p);
    uint8_t* const s_codes = lds + at.codes;    // [K step][row][128 bytes], chunk j of row r at j ^ (r % 8)
    float* const s_scale = reinterpret_cast<float*>(lds + at.scales);      // [K step][row]
    float* const s_wscale = reinterpret_cast<float*>(lds + at.wscales);    // [block row of the segment][gate, up][K step]
    int16_t* const s_ids = reinterpret_cast<int16_t*>(lds + at.ids);
    uint16_t* const s_list = reinterpret_cast<uint16_t*>(lds + at.list);   // the slots of the segment's expert
    float* const s_weight = reinterpret_cast<float*>(lds + at.weight);     // second GEMM: routed weight of every slot
    uint16_t* const s_src = reinterpret_cast<uint16_t*>(lds + at.weight);  // first GEMM: the listed slots' rows of x
    uint32_t* const s_count = reinterpret_cast<uint32_t*>(lds + at.count); // rows of every expert, two 16-bit counts a word
    int* const s_rows = reinterpret_cast<int*>(lds + at.rows);             // rows of the segment's expert

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = p.K, kblocks = p.kblocks, slots = p.slots, cap = p.row_cap;
    const int groups = (UP ? p.inter : p.N) / COLS;

    // ---- the experts' rows
    if (tid < (p.E + 1) / 2) s_count[tid] = 0;  // (at most 256 words)
    __syncthreads();
    for (int i = tid; i < slots; i += NT) {
        const int e = decode_expert_id(p, i);
        s_ids[i] = (int16_t)e;
        if constexpr (!UP) s_weight[i] = p.topk_weights[i];
        if (e >= 0) atomicAdd(&s_count[e >> 1], 1u << ((e & 1) * 16));   // (at most 2048 slots: no carry into the other half)
    }
    __syncthreads();
    auto rows_of = [&](int e) { return e < p.E ? (int)reinterpret_cast<const uint16_t*>(s_count)[e] : 0; };
    const int cap_log2 = __builtin_ctz(cap);
    int total_passes = 0;                       // one per expert that has rows; more for those with more than are held, if any
    bool hot = false;
#pragma unroll 1
    for (int base = 0; base < p.E; base += 64) {
        const int c = rows_of(base + lane);
        total_passes += __popcll(__ballot(c > 0));
        hot |= __ballot(c > cap) != 0;
    }
    if (__builtin_expect(hot, 0)) {
        total_passes = 0;
        for (int base = 0; base < p.E; base += 64) total_passes += (rows_of(base + lane) + cap - 1) >> cap_log2;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) total_passes += __shfl_xor(total_passes, d);
        total_passes = __builtin_amdgcn_readfirstlane(total_passes);
    }

    // ---- this workgroup's share of the total_passes * groups units, in segments of one pass each.  Either a pass's groups are
    // dealt over workgroups of its own (one token, six experts: 42 of 256 for each), or the units are dealt over all of them
    // and a workgroup may meet two passes or more: an equal share, but a second pass's preparation costs as much as streaming
    // pass_groups groups, two and 40 K steps (about 3 us).  One expert in every token, 32 experts of (2048, 512), top 4, 48 tokens (33
    // passes): 41.6 -> 32.7 us with 7 workgroups to each pass; 64 of (1024, 512), top 8, 56 tokens, half alike: 40.7 -> 35.6.
    const int grid = (int)gridDim.x, bid = (int)blockIdx.x;
    // x / d from inv = 1 / d: two roundings move (x + 0.5) / d, which is 0.5 / d or more away from an integer, by less than
    // (x + 0.5) / d * 2^-22, so exact for x < 2^21 (below: groups <= 8192 times fewer than 256 workgroups)
    auto small_div = [](int x, float inv) { return (int)(((float)x + 0.5f) * inv); };
    int u_begin, u_end;
    const int per = total_passes > 0 ? small_div(grid, 1.0f / (float)total_passes) : 0;  // workgroups per pass
    if (per > 0 && groups * grid <= per * (total_passes * groups + p.pass_groups * grid)) {
        const float inv_per = 1.0f / (float)per;
        const int idx = small_div(bid, inv_per), part = bid - idx * per;
        u_begin = idx * groups + small_div(groups * part, inv_per);
        u_end = part == per - 1 ? (idx + 1) * groups : idx * groups + small_div(groups * (part + 1), inv_per);
        if (idx >= total_passes) u_begin = u_end = 0;
    } else {
        // units * bid / grid by quotient and remainder of units / grid: 32 bits suffice
        const uint32_t units = (uint32_t)(total_passes * groups), q = units / (uint32_t)grid, r = units - q * (uint32_t)grid;
        u_begin = (int)(q * (uint32_t)bid + r * (uint32_t)bid / (uint32_t)grid);
        u_end = (int)(q * (uint32_t)(bid + 1) + r * (uint32_t)(bid + 1) / (uint32_t)grid);
    }
    u_begin = __builtin_amdgcn_readfirstlane(u_begin);
    u_end = __builtin_amdgcn_readfirstlane(u_end);
    // unit u -> its expert, the first of its rows and the groups [g0, g1) of the pass that are this workgroup's
    auto segment = [&](int u, int* e, int* r0, int* g0, int* g1) {
        const int idx = __builtin_amdgcn_readfirstlane(u / groups);
        *g0 = u - idx * groups;
        *g1 = min(groups, *g0 + u_end - u);
        int left = idx;
        *e = 0;
        *r0 = 0;
        if (__builtin_expect(!hot, 1)) {
            // the left-th expert that has rows
#pragma unroll 1
            for (int base = 0; base < p.E; base += 64) {
                const int c = rows_of(base + lane);
                const unsigned long long any = __ballot(c > 0);
                if (left < __popcll(any)) {
                    const int rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(any >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)any, 0));
                    *e = base + __builtin_ctzll(__ballot(c > 0 && rank == left));
                    break;
                }
                left -= __popcll(any);
            }
            return;
        }
        for (int base = 0; base < p.E; base += 64) {
            const int mine = (rows_of(base + lane) + cap - 1) >> cap_log2;
            int incl = mine;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int below = __shfl_up(incl, d);
                if (lane >= d) incl += below;
            }
            const unsigned long long past = __ballot(incl > left);
            if (past != 0) {
                const int at_lane = __builtin_ctzll(past);
                *e = base + at_lane;
                *r0 = (left - __builtin_amdgcn_readlane(incl - mine, at_lane)) * cap;
                break;
            }
            left -= __builtin_amdgcn_readlane(incl, 63);
        }
    };

    if (wave >= NW) {
        // ================================================================ the waves that prepare the activations
        const int qt = tid - 64 * NW;
        const float inv_kblocks = 1.0f / (float)kblocks, inv_top_k = 1.0f / (float)p.top_k;
        for (int u = u_begin; u < u_end;) {
            int e, r0, g0, g1;
            segment(u, &e, &r0, &g0, &g1);
            u += g1 - g0;
            // the expert's slots, in ascending order (every one of these waves writes the same list)
            int rows = 0;
            for (int base = 0; base < slots; base += 64) {
                const bool mine = base + lane < slots && s_ids[base + lane] == e;
                const unsigned long long m = __ballot(mine);
                if (mine) {
                    const int at_row = rows + __popcll(m & ((1ull << lane) - 1ull));
                    s_list[at_row] = (uint16_t)(base + lane);
                    if constexpr (UP) s_src[at_row] = (uint16_t)small_div(base + lane, inv_top_k);
                }
                rows += __popcll(m);
            }
            if (qt == 0) *s_rows = rows;
            // weight scales of the segment's block rows (UP: of the gate and of the up rows)
            const float* const ws = p.ws + (int64_t)e * p.nblocks * kblocks;
            const int nb0 = g0 * COLS / 128, nbs = (g1 * COLS - 1) / 128 - nb0 + 1;
            const int n_ws = nbs * (UP ? 2 : 1) * kblocks;
            for (int i = qt; i < n_ws; i += NTQ) {
                const int row = small_div(i, inv_kblocks), kb = i - row * kblocks;
                const int nb = UP ? nb0 + (row >> 1) + ((row & 1) ? p.inter / 128 : 0) : nb0 + row;
                s_wscale[i] = ws[nb * kblocks + kb];
            }
            const int rows_a = min(cap, rows - r0);
            const int n_x = rows_a * kblocks * 16;   // 16-byte pieces of activations: 16 to a group of 128
            constexpr int BATCH = 8;
            for (int first = qt; first - qt < n_x; first += BATCH * NTQ) {
                v4i raw[BATCH];
#pragma unroll
                for (int j = 0; j < BATCH; ++j) {
                    const int task = min(first + j * NTQ, n_x - 16 + (lane & 15)), group = task >> 4;
                    const int row = small_div(group, inv_kblocks), kb = group - row * kblocks;
                    const int src = (UP ? s_src : s_list)[r0 + row];
                    raw[j] = *reinterpret_cast<const v4i*>(reinterpret_cast<const T*>(p.x) + ((int64_t)src * K + kb * 128 + (task & 15) * 8));
                }
                // the first activations are requested before the weights: the compute unit takes its requests in order
                if (first == qt) decode_barrier();
#pragma unroll
                for (int j = 0; j < BATCH; ++j) {
                    const int task = first + j * NTQ, group = task >> 4, sub = task & 15;
                    const int row = small_div(group, inv_kblocks), kb = group - row * kblocks;
                    float sc;
                    const v2i codes = quantize_lane<T>(raw[j], &sc);
                    if (task < n_x) {
                        *reinterpret_cast<v2i*>(s_codes + (kb * cap + row) * kKBlock + (((sub >> 1) ^ swz16(row)) << 4) + (sub & 1) * 8) = codes;
                        if (sub == 0) s_scale[kb * cap + row] = sc;
                    }
                }
            }
            decode_barrier();   // the tile is ready
            decode_barrier();   // ... and done with
        }
        return;
    }

    // ==================================================================== the waves that stream the weights
    const int li = lane & 15, lg = lane >> 4;
    const int npieces = (K + kDecodePiece - 1) / kDecodePiece;
    const int tail_steps = (K % kDecodePiece) / kKBlock;  // 0: every piece is whole
    // a lane's place in a load: row 2i + lane / 32 of the piece, LDS position lane % 32 of the row's 32 chunks, which holds
    // logical chunk (lane % 32) ^ row.  Row r of a group: UP: column 2 (r / 4) + r % 2, gate for r % 4 < 2, else up.
    const int half = lane >> 5, pos = lane & 31;
    uint32_t w_off[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int r = 2 * i + half;
        const uint32_t n = UP ? (uint32_t)((r >> 2) * 2 + (r & 1) + ((r & 2) ? p.inter : 0)) : (uint32_t)r;
        w_off[i] = n * (uint32_t)K + ((pos ^ r) << 4);
    }
    const uint32_t my_lds = lds_address(lds) + wave * STAGES * kDecodeBuf;
    const uint8_t* const my_ring = lds + wave * STAGES * kDecodeBuf;
    const int arow = li & (cap - 1);            // (columns past the rows of a tile repeat rows; they are not stored)
    const uint32_t frag0 = arow * kKBlock + ((lg ^ swz16(arow)) << 4), frag1 = frag0 ^ 64;

    for (int u = u_begin; u < u_end;) {
        int e, r0, g0, g1;
        segment(u, &e, &r0, &g0, &g1);
        u += g1 - g0;
        const v4i rsrc_w = make_rsrc(p.w + (int64_t)e * p.N * K);
        const int nb0 = g0 * COLS / 128;
        const int total = max(0, (g1 - g0 - wave + NW - 1) / NW) * npieces;   // pieces of this wave
        // ---- the ring: as many pieces as it holds, before the activations are waited for
        int gi = g0 + wave, ci = 0;
        auto issue = [&](int stage) {
            const int k0 = gi * (COLS * K) + ci * kDecodePiece;
            const int valid = (tail_steps != 0 && ci == npieces - 1) ? tail_steps * 8 : 32;
#pragma unroll
            for (int i = 0; i < LOADS; ++i)
                direct_load_b128_nt(rsrc_w, my_lds + stage * kDecodeBuf + i * 1024, (pos ^ (2 * i + half)) < valid ? w_off[i] : kDecodeOutOfRange, k0);
            if (++ci == npieces) { ci = 0; gi += NW; }
        };
        decode_barrier();
        for (int s = 0; s < STAGES && s < total; ++s) issue(s);
        decode_barrier();
        const int rows_a = min(cap, __builtin_amdgcn_readfirstlane(*s_rows) - r0);

        // ---- this wave's groups
        int gc = g0 + wave, cc = 0;
        v4f acc = v4f{0.f, 0.f, 0.f, 0.f};
        int stage = 0;
        for (int i = 0; i < total; ++i) {
            if (i + STAGES <= total) wait_vmcnt<(STAGES - 1) * LOADS>();
            else wait_vmcnt<0>();
            // Everything the piece needs is read at once: one LDS round trip per piece.  K steps past the end of K multiply
            // zeros (their weight loads are out of range) with the last step's activations, under scales of zero (the last step's
            // may be infinite).
            const uint8_t* wb = my_ring + stage * kDecodeBuf + li * kDecodePiece;
            const float* ws = s_wscale + ((gc * COLS >> 7) - nb0) * (UP ? 2 : 1) * kblocks;
            v8i wf[kDecodeSteps], af[kDecodeSteps];
            float as[kDecodeSteps], bg[kDecodeSteps], bu[kDecodeSteps];
#pragma unroll
            for (int s = 0; s < kDecodeSteps; ++s) {
                const int kb = min(cc * kDecodeSteps + s, kblocks - 1);
                const uint8_t* ab = s_codes + kb * cap * kKBlock;
                wf[s] = join(*reinterpret_cast<const v4i*>(wb + (((s * 8 + lg) ^ li) << 4)), *reinterpret_cast<const v4i*>(wb + (((s * 8 + 4 + lg) ^ li) << 4)));
                af[s] = join(*reinterpret_cast<const v4i*>(ab + frag0), *reinterpret_cast<const v4i*>(ab + frag1));
                as[s] = s_scale[kb * cap + arow];
                bg[s] = ws[kb];
                bu[s] = UP ? ws[kblocks + kb] : 0.f;
            }
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the fragments are in registers, the stage is free
#pragma unroll
            for (int s = 0; s < kDecodeSteps; ++s) asm volatile("" : "+v"(wf[s]), "+v"(af[s]), "+v"(as[s]), "+v"(bg[s]), "+v"(bu[s]));
            if (i + STAGES < total) issue(stage);
            stage = stage + 1 == STAGES ? 0 : stage + 1;
            if (tail_steps != 0 && cc == npieces - 1) {
#pragma unroll
                for (int s = 1; s < kDecodeSteps; ++s) {
                    const bool past = s >= tail_steps;
                    as[s] = past ? 0.f : as[s];
                    bg[s] = past ? 0.f : bg[s];
                    bu[s] = past ? 0.f : bu[s];
                }
            }
            v4f part[kDecodeSteps];
#pragma unroll
            for (int s = 0; s < kDecodeSteps; ++s) part[s] = mfma_e4m3(wf[s], af[s], v4f{0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int s = 0; s < kDecodeSteps; ++s) {
                const float lo = as[s] * bg[s], hi = UP ? as[s] * bu[s] : lo;
                acc += part[s] * v4f{lo, lo, hi, hi};
            }
            if (++cc == npieces) {
                if (li < rows_a) {
                    const int slot = s_list[r0 + li];
                    if constexpr (UP) {
                        typedef T vec2 __attribute__((ext_vector_type(2)));
                        vec2 v;
                        v[0] = (T)silu_mul_round<T>((float)(T)acc[0], (float)(T)acc[2]);
                        v[1] = (T)silu_mul_round<T>((float)(T)acc[1], (float)(T)acc[3]);
                        *reinterpret_cast<vec2*>(reinterpret_cast<T*>(p.out) + (int64_t)slot * p.inter + gc * COLS + lg * 2) = v;
                    } else {
                        typedef T vec4 __attribute__((ext_vector_type(4)));
                        *reinterpret_cast<vec4*>(reinterpret_cast<T*>(p.out) + (int64_t)slot * p.N + gc * COLS + lg * 4) =
                            __builtin_convertvector(acc * s_weight[slot], vec4);
                    }
                }
                acc = v4f{0.f, 0.f, 0.f, 0.f};
                cc = 0;
                gc += NW;
            }
        }
        decode_barrier();
    }
#endif
}

// The second GEMM and the sum over a token's slots: one workgroup per token and R output columns, one wave per slot.  A wave
// streams its slot's expert's R weight rows (weights shared by two tokens are read twice, mostly out of the caches: for a
// few tokens that costs less than the sum's launch), all of a short K in flight at once, and the slots' results, rounded
// to the 16-bit type as the row-per-slot form stores them, are added through LDS in slot order.
constexpr int kDecodeSumRows = 8;
constexpr int kDecodeSumStages = 3;
// Dynamic LDS of moe_decode_sum_kernel: every wave's ring (in the end its slot's results), every wave's codes and scales.
// (the scales of a piece's four K steps are read whole: three zeros behind the last one)
__host__ __device__ inline int moe_decode_sum_codes(int K) { return (K + K / 32 + 12 + 255) / 256 * 256; }
inline int moe_decode_sum_lds(int top_k, int K) {
    return top_k * (kDecodeSumStages * kDecodeSumRows * kDecodePiece + moe_decode_sum_codes(K));
}

template <typename T>
__global__ void __launch_bounds__(512) moe_decode_sum_kernel(const MoeDecodeParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int R = kDecodeSumRows, STAGES = kDecodeSumStages, BUF = R * kDecodePiece, LOADS = BUF / 1024, X_LOADS = 4;
    extern __shared__ __align__(1024) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const int K = p.K, kblocks = p.kblocks;
    const int slot = (int)blockIdx.y * p.top_k + wave, n0 = (int)blockIdx.x * R;
    const int npieces = (K + kDecodePiece - 1) / kDecodePiece;
    const int tail_steps = (K % kDecodePiece) / kKBlock;
    uint8_t* const my_ring = lds + wave * STAGES * BUF;
    const int codes_bytes = moe_decode_sum_codes(K);
    uint8_t* const my_codes = lds + p.top_k * STAGES * BUF + wave * codes_bytes;  // [K step][128 bytes]
    float* const my_scale = reinterpret_cast<float*>(my_codes + K);               // [K step]
    const int e = __builtin_amdgcn_readfirstlane(decode_expert_id(p, slot));
    const float weight = p.topk_weights[slot];
    v4f acc = v4f{0.f, 0.f, 0.f, 0.f};
    if (e >= 0) {
        const v4i rsrc_x = make_rsrc(reinterpret_cast<const T*>(p.x) + (int64_t)slot * K);
        const v4i rsrc_w = make_rsrc(p.w + (int64_t)e * p.N * K);
        const v4i rsrc_ws = make_rsrc(p.ws + ((int64_t)e * p.nblocks + n0 / 128) * kblocks);
        float wsc = buffer_load_f32_raw(rsrc_ws, lane < kblocks ? lane * 4u : kDecodeOutOfRange);  // lane kb: the scale of K step kb
        v4i raw[X_LOADS];
#pragma unroll
        for (int j = 0; j < X_LOADS; ++j) {
            const int task = lane + j * 64;
            raw[j] = buffer_load_b128_raw(rsrc_x, task < kblocks * 16 ? task * 16u : kDecodeOutOfRange);
        }
        const int half = lane >> 5, pos = lane & 31;
        uint32_t w_off[LOADS];
#pragma unroll
        for (int i = 0; i < LOADS; ++i) w_off[i] = (uint32_t)(n0 + 2 * i + half) * (uint32_t)K + ((pos ^ (2 * i + half)) << 4);
        const uint32_t my_lds = lds_address(my_ring);
        auto issue = [&](int c, int stage) {
            const int valid = c >= npieces ? 0 : (tail_steps != 0 && c == npieces - 1) ? tail_steps * 8 : 32;
#pragma unroll
            for (int i = 0; i < LOADS; ++i)
                direct_load_b128_nt(rsrc_w, my_lds + stage * BUF + i * 1024, (pos ^ (2 * i + half)) < valid ? w_off[i] : kDecodeOutOfRange, c * kDecodePiece);
        };
#pragma unroll
        for (int s = 0; s < STAGES; ++s) issue(s, s);  // (pieces past the end request nothing)
        wait_vmcnt<STAGES * LOADS>();
        asm volatile("" : "+v"(wsc));
#pragma unroll
        for (int j = 0; j < X_LOADS; ++j) asm volatile("" : "+v"(raw[j]));
        auto put = [&](int task, v4i v) {
            float s;
            const v2i codes = quantize_lane<T>(v, &s);
            if (task < kblocks * 16) {
                *reinterpret_cast<v2i*>(my_codes + task * 8) = codes;
                if ((task & 15) == 0) my_scale[task >> 4] = s;
            }
        };
#pragma unroll
        for (int j = 0; j < X_LOADS; ++j)
            if (j * 4 < kblocks) put(lane + j * 64, raw[j]);
        if (lane < 3) my_scale[kblocks + lane] = 0.f;   // K steps past the end add nothing: both of their scales are zero
        for (int task = lane + X_LOADS * 64; task - lane < kblocks * 16; task += 64) {
            v4i v = v4i{0, 0, 0, 0};
            if (task < kblocks * 16) v = *reinterpret_cast<const v4i*>(reinterpret_cast<const uint8_t*>(p.x) + ((int64_t)slot * K + task * 8) * 2);
            put(task, v);
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);
        int stage = 0;
        for (int c = 0; c < npieces; ++c) {
            if (c + STAGES <= npieces) wait_vmcnt<(STAGES - 1) * LOADS>();
            else wait_vmcnt<0>();
            const int r = li & (R - 1);
            const uint8_t* wb = my_ring + stage * BUF + r * kDecodePiece;
            v8i wf[kDecodeSteps], af[kDecodeSteps];
            float sc[kDecodeSteps];
#pragma unroll
            for (int s = 0; s < kDecodeSteps; ++s) {
                const int kb = min(c * kDecodeSteps + s, kblocks - 1);
                const uint8_t* ab = my_codes + kb * kKBlock + lg * 16;   // (one row: the same in every column)
                wf[s] = join(*reinterpret_cast<const v4i*>(wb + (((s * 8 + lg) ^ r) << 4)), *reinterpret_cast<const v4i*>(wb + (((s * 8 + 4 + lg) ^ r) << 4)));
                af[s] = join(*reinterpret_cast<const v4i*>(ab), *reinterpret_cast<const v4i*>(ab + 64));
                sc[s] = my_scale[c * kDecodeSteps + s];
            }
            __builtin_amdgcn_s_waitcnt(0xC07F);
#pragma unroll
            for (int s = 0; s < kDecodeSteps; ++s) asm volatile("" : "+v"(wf[s]), "+v"(af[s]), "+v"(sc[s]));
            if (c + STAGES < npieces) issue(c + STAGES, stage);
            stage = stage + 1 == STAGES ? 0 : stage + 1;
            v4f part[kDecodeSteps];
#pragma unroll
            for (int s = 0; s < kDecodeSteps; ++s) part[s] = mfma_e4m3(wf[s], af[s], v4f{0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int s = 0; s < kDecodeSteps; ++s) {
                // (at most 64 K steps; lanes past the last one hold zero)
                acc += part[s] * (sc[s] * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wsc), c * kDecodeSteps + s)));
            }
        }
    }
    if (li == 0 && lg * 4 < R) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float v = e >= 0 ? acc[q] * weight : 0.f;   // (a slot without an expert adds nothing, whatever its weight)
            asm("" : "+v"(v));  // (the product is rounded on its own before the conversion, as the stored form is)
            reinterpret_cast<float*>(my_ring)[lg * 4 + q] = (float)(T)v;   // (the ring has been read to its end)
        }
    }
    __syncthreads();
    if (tid < R) {
        auto slot_result = [&](int w) { return reinterpret_cast<const float*>(lds + w * STAGES * BUF)[tid]; };
        float sum = slot_result(0);
        for (int w = 1; w < p.top_k; ++w) sum += slot_result(w);
        reinterpret_cast<T*>(p.out)[(int64_t)blockIdx.y * p.N + n0 + tid] = (T)sum;
    }
#endif
}

}  // namespace tg
