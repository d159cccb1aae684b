"""Parity of the HIP FP8 GEMM path (through the C ABI) with the CPU oracle.

Tolerance (stated by the task): |out - ref| <= 2e-2 * sigma_ref + 2e-2 * |ref| with
sigma_ref = std of the oracle output ("relative to output scale").  Kernel and oracle consume
the same quantized bytes, so the real error is fp32 re-association plus one output rounding;
TIGHT below is the much smaller bound we additionally expect (and flag when exceeded).
"""

import math

import pytest
import torch

import tilegym_amd
from oracle import reference as R
from tilegym_amd import _lib, workloads as W
from tilegym_amd.ops import group_gemm, matmul, moe_align_block_size
from tilegym_amd.ops.moe_interface import invoke_fused_moe_kernel
from tilegym_amd.suites.flashinfer.ops import gemm_alpha_beta, ragged_block_scaled_bmm
from tilegym_amd.suites.unsloth.ops import w8a8_block_fp8_matmul

pytestmark = pytest.mark.gpu
FP8 = torch.float8_e4m3fn
RTOL = ATOL = 2e-2
TIGHT = 8.5e-3  # one bf16 ulp is at most 2^-7 = 7.8e-3 relative (a rounding tie may flip one ulp)


def _g(seed):
    return torch.Generator().manual_seed(seed)


def check(out, ref, tight=TIGHT, what=""):
    ok, rep = R.compare_to_oracle(out, ref, RTOL, ATOL)
    assert ok, f"{what}: outside tolerance: {rep}"
    ok2, rep2 = R.compare_to_oracle(out, ref, tight, tight)
    assert ok2, f"{what}: inside the stated tolerance but worse than expected: {rep2}"


def fp8_randn(shape, g, std=1.0):
    return (torch.randn(shape, generator=g) * std).clamp(-448, 448).to(FP8)


def used(kernel_name):
    cfg = _lib.last_config()
    assert cfg["KERNEL_NAME"] == kernel_name, f"expected the {kernel_name} kernel, library chose {cfg}"
    return cfg


# ----------------------------------------------------------------------------- per-tensor, tiled
@pytest.mark.parametrize("bm,bn", [(256, 256), (128, 128), (128, 256), (64, 128)])
@pytest.mark.parametrize("M,N,K", [(256, 512, 1024), (200, 328, 384), (77, 130, 128), (513, 1000, 256)])
def test_per_tensor_tiled_configs(device, bm, bn, M, N, K):
    g = _g(M + N + K)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.5)
    sa, sb = torch.tensor([0.37]), torch.tensor([1.9])
    ref = R.ref_gemm_per_tensor(a, b, sa, sb, trans_b=True)
    out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=sa.to(device), scale_b=sb.to(device),
                 out_dtype=torch.bfloat16, kernel_configs={"KERNEL": "tiled", "BLOCK_M": bm, "BLOCK_N": bn, "SPLIT_K": 1})
    cfg = used("tiled")
    assert (cfg["BLOCK_M"], cfg["BLOCK_N"]) == (bm, bn)
    assert out.dtype == torch.bfloat16 and out.shape == (M, N)
    check(out, ref, what=f"tiled {bm}x{bn} {M}x{N}x{K}")


@pytest.mark.parametrize("split", [2, 3, 8])
def test_per_tensor_tiled_split_k(device, split):
    g = _g(split)
    M, N, K = 200, 264, 2048
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g)
    ref = R.ref_gemm_per_tensor(a, b, 0.01, 0.5, trans_b=True)
    kc = {"KERNEL": "tiled", "BLOCK_M": 128, "BLOCK_N": 128, "SPLIT_K": split}
    out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=0.01, scale_b=0.5, out_dtype=torch.bfloat16, kernel_configs=kc)
    assert used("tiled")["SPLIT_K"] > 1
    check(out, ref, what=f"split-K {split}")
    # the reduction order is fixed: reruns are bit-identical, and the counters were left at zero
    for _ in range(3):
        again = matmul(a.to(device), b.to(device), trans_b=True, scale_a=0.01, scale_b=0.5, out_dtype=torch.bfloat16, kernel_configs=kc)
        assert torch.equal(again, out)


# ----------------------------------------------------------------------------- per-tensor, persistent hand-ordered 256x256 tile
@pytest.mark.parametrize("waves", [-1, 8])
@pytest.mark.parametrize("M,N,K", [(256, 256, 128), (300, 520, 384), (257, 255, 512), (1024, 768, 1280), (40, 1000, 256), (512, 252, 640)])
def test_per_tensor_ordered_256(device, M, N, K, waves):
    """The 256x256 tile in its persistent hand-ordered form (default from two K steps up) and in the generic form
    (WAVES = 8): K = 128 (one step: always the generic form), odd numbers of steps, ragged M and N, N not a multiple of 8
    (scalar store path); bf16, f16, f32 outputs and beta; the two forms agree bit for bit."""
    g = _g(M + 3 * N + K)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.02)
    sa, sb = torch.tensor([0.013]), torch.tensor([0.0004])
    kc = {"KERNEL": "tiled", "BLOCK_M": 256, "BLOCK_N": 256, "SPLIT_K": 1, "WAVES": waves}
    ref = R.ref_gemm_per_tensor(a, b, sa, sb, trans_b=True)
    res = matmul(a.to(device), b.to(device), trans_b=True, scale_a=sa.to(device), scale_b=sb.to(device),
                 out_dtype=torch.bfloat16, kernel_configs=kc)
    cfg = used("tiled")
    assert (cfg["BLOCK_M"], cfg["BLOCK_N"]) == (256, 256)
    check(res, ref, what=f"256x256 M={M} N={N} K={K} waves={waves}")
    other = matmul(a.to(device), b.to(device), trans_b=True, scale_a=sa.to(device), scale_b=sb.to(device),
                   out_dtype=torch.bfloat16, kernel_configs=dict(kc, WAVES=8 if waves != 8 else -1))
    assert torch.equal(res, other), "ordered and generic 256x256 kernels differ"
    one = torch.tensor([1.0])  # keep the f16 outputs in the normal range
    ref16 = R.ref_gemm_per_tensor(a, b, one, one, trans_b=True, out_dtype=torch.float16)
    res16 = matmul(a.to(device), b.to(device), trans_b=True, scale_a=one.to(device), scale_b=one.to(device),
                   out_dtype=torch.float16, kernel_configs=kc)
    check(res16, ref16, what=f"256x256 f16 M={M} N={N} K={K}")
    ref32 = R.ref_gemm_per_tensor(a, b, sa, sb, trans_b=True, out_dtype=torch.float32)
    res32 = matmul(a.to(device), b.to(device), trans_b=True, scale_a=sa.to(device), scale_b=sb.to(device),
                   out_dtype=torch.float32, kernel_configs=kc)
    check(res32, ref32, what=f"256x256 f32 M={M} N={N} K={K}")


@pytest.mark.parametrize("M,N,K,out_dtype", [(4352, 4352, 384, torch.bfloat16), (4300, 4360, 256, torch.bfloat16),
                                             (4200, 4507, 640, torch.float16), (2100, 9000, 256, torch.float32)])
def test_persistent_256_walks_several_tiles_per_workgroup(device, M, N, K, out_dtype):
    """More 256x256 tiles than the device has compute units: workgroups of the persistent kernel compute two or more
    tiles, with the operand rings running on from one tile into the next.  Full tiles only; ragged last tile rows and
    columns (a partial tile in the middle of a workgroup's sequence); N not a multiple of 8 (scalar stores); two K steps
    (the switch to the next tile's addresses happens in a tile's first step).  Bit-equal to the generic eight-wave
    kernel, which computes one tile per workgroup, and sampled rows against the oracle."""
    assert math.ceil(M / 256) * math.ceil(N / 256) > torch.cuda.get_device_properties(device).multi_processor_count
    g = _g(M + N + K)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.02)
    sa, sb = torch.tensor([0.021]), torch.tensor([0.0007])
    kc = {"KERNEL": "tiled", "BLOCK_M": 256, "BLOCK_N": 256, "SPLIT_K": 1}
    args = dict(trans_b=True, scale_a=sa.to(device), scale_b=sb.to(device), out_dtype=out_dtype)
    res = matmul(a.to(device), b.to(device), kernel_configs=kc, **args)
    cfg = used("tiled")
    assert (cfg["BLOCK_M"], cfg["BLOCK_N"]) == (256, 256)
    other = matmul(a.to(device), b.to(device), kernel_configs=dict(kc, WAVES=8), **args)
    assert torch.equal(res, other), "persistent and generic 256x256 kernels differ"
    rows = torch.cat([torch.arange(0, 4), torch.arange(255, 258), torch.randint(0, M, (24,), generator=g), torch.arange(M - 3, M)])
    ref = R.ref_gemm_per_tensor(a[rows], b, sa, sb, trans_b=True, out_dtype=out_dtype)
    check(res[rows.to(device)], ref, what=f"persistent 256x256 M={M} N={N} K={K}")


@pytest.mark.parametrize("bm,bn", [(32, 64), (64, 64), (32, 128)])
@pytest.mark.parametrize("dm,N,K,split", [(0, 256, 128, 1), (-1, 120, 1024, 1), (1, 136, 1152, 2), (17, 257, 2176, 1), (-15, 384, 2304, 2), (0, 192, 4096, 1)])
def test_ring_tiles_block_scaled_narrow(device, bm, bn, dm, N, K, split):
    """The tiles of 64 columns (half of a block of weight scales) and 32 rows, over the same edges and four chunks of scales: same bits
    as the 128 x 128 tile kernel, with either scale tensor missing too, and the oracle's result; beta in the epilogue."""
    M = 2 * bm + dm
    g = _g(bm + bn + N + K)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.5)
    sa, sb = torch.rand(M, K // 128, generator=g) * 0.1 + 0.01, torch.rand((N + 127) // 128, K // 128, generator=g) * 0.1 + 0.01
    ad, bd, sad, sbd = a.to(device), b.to(device), sa.to(device), sb.to(device)
    c0 = torch.randn(M, N, generator=g)
    for s1, s2, dtype, beta in ((sad, sbd, torch.bfloat16, 0.0), (None, sbd, torch.float32, 0.0), (sad, None, torch.float16, 0.0), (sad, sbd, torch.float32, 0.5)):
        out, base = c0.to(device).to(dtype), c0.to(device).to(dtype)
        _lib.fp8_gemm(out, ad, bd, s1, s2, False, True, 1.0, beta, {"KERNEL": "tiled", "BLOCK_M": bm, "BLOCK_N": bn, "SPLIT_K": split, "WAVES": 8})
        cfg = used("tiled")
        assert (cfg["BLOCK_M"], cfg["BLOCK_N"], cfg["WAVES"]) == (bm, bn, 8), cfg
        _lib.fp8_gemm(base, ad, bd, s1, s2, False, True, 1.0, beta, {"KERNEL": "tiled", "BLOCK_M": 128, "BLOCK_N": 128, "SPLIT_K": cfg["SPLIT_K"]})
        assert torch.equal(out, base)
        if dtype is torch.bfloat16:
            check(out, R.ref_w8a8_block_fp8_matmul(a, b, sa, sb, None, torch.bfloat16), what=f"block ring {bm}x{bn} M={M} N={N} K={K}")


@pytest.mark.parametrize("bm,bn", [(32, 32), (64, 32), (64, 64)])
@pytest.mark.parametrize("M,N,K", [(64, 512, 1024), (40, 200, 384), (17, 1000, 2560), (130, 72, 128), (33, 264, 256), (96, 4096, 4096)])
def test_per_tensor_mid_tiles(device, bm, bn, M, N, K):
    """The narrow tiles whose four waves split K inside the workgroup: fewer K steps than waves (K = 128, 256: waves
    without a step), K steps that do not divide by four, ragged M (also across row tiles) and N, N not a multiple of 8;
    bf16 and f32 outputs with alpha and beta; reruns are bit-identical (fixed reduction order)."""
    g = _g(M + 5 * N + K + bm + bn)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.02)
    sa, sb = torch.tensor([0.013]), torch.tensor([0.0004])
    kc = {"KERNEL": "tiled", "BLOCK_M": bm, "BLOCK_N": bn}
    ref = R.ref_gemm_per_tensor(a, b, sa, sb, trans_b=True)
    out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=sa.to(device), scale_b=sb.to(device), out_dtype=torch.bfloat16, kernel_configs=kc)
    cfg = used("tiled")
    assert (cfg["BLOCK_M"], cfg["BLOCK_N"], cfg["SPLIT_K"]) == (bm, bn, 1)
    check(out, ref, what=f"mid {bm}x{bn} M={M} N={N} K={K}")
    again = matmul(a.to(device), b.to(device), trans_b=True, scale_a=sa.to(device), scale_b=sb.to(device), out_dtype=torch.bfloat16, kernel_configs=kc)
    assert torch.equal(out, again)
    c0 = torch.randn(M, N, generator=g)
    c = c0.clone().to(device)
    _lib.fp8_gemm(c, a.to(device), b.to(device), sa.to(device), sb.to(device), False, True, 1.5, 0.5, kernel_configs=kc)
    ref32 = 1.5 * R.ref_gemm_per_tensor(a, b, sa, sb, trans_b=True, out_dtype=torch.float32) + 0.5 * c0
    check(c, ref32, what=f"mid {bm}x{bn} f32 alpha/beta M={M} N={N} K={K}")


def test_mid_tiles_are_the_default_for_small_weights(device):
    g = _g(8)
    b = fp8_randn((4096, 4096), g, 0.02)
    for M, want in ((32, (32, 32)), (64, (32, 32)), (128, (64, 32)), (192, (64, 64)), (256, (64, 64))):
        a = fp8_randn((M, 4096), g)
        out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=0.01, scale_b=0.02, out_dtype=torch.bfloat16)
        cfg = used("tiled")
        assert (cfg["BLOCK_M"], cfg["BLOCK_N"]) == want, (M, cfg)
        check(out, R.ref_gemm_per_tensor(a, b, 0.01, 0.02, trans_b=True), what=f"M={M} default")


@pytest.mark.parametrize("N,K", [(4096, 4096), (2048, 4096), (2048, 8192), (3072, 4096)])
def test_a_full_last_row_tile_changes_no_schedule(device, N, K):
    """319 and 320 rows are five row tiles of 64 either way (four of 96, three of 128, two of 160 and 192): the same kernel runs, and the
    first 319 rows get the same bits."""
    g = _g(320)
    a, b = fp8_randn((320, K), g), fp8_randn((N, K), g, 0.02)
    outs, cfgs = [], []
    for M in (319, 320):
        outs.append(matmul(a[:M].to(device), b.to(device), trans_b=True, scale_a=0.01, scale_b=0.02, out_dtype=torch.bfloat16))
        cfgs.append(used("tiled"))
    assert cfgs[0] == cfgs[1]
    assert torch.equal(outs[0], outs[1][:319])
    check(outs[1], R.ref_gemm_per_tensor(a, b, 0.01, 0.02, trans_b=True), what=f"320 x {N} x {K}")


def test_weights_of_2_gib_and_more_run_in_column_chunks(device):
    """A (N, K) weight of 2 GiB or more cannot be indexed with 32-bit byte offsets: the columns of C are computed in
    chunks of weight rows on the fast kernels (streaming for M = 8, tiled for M = 40), not on the software-decode
    fallback.  Checked against the oracle on sampled columns, among them both sides of the chunk boundary and the
    last column, with per-tensor and with block scales."""
    K = 16384
    N = (1 << 31) // K + 520          # 2 GiB + 8.1 MiB of weights; N is a multiple of 8, not of 128
    chunk = ((1 << 31) - 1) // K // 256 * 256
    g = _g(77)
    codes = torch.randint(0, 256, (N, K), dtype=torch.uint8, device=device)
    codes[(codes & 0x7F) == 0x7F] = 0x38          # no NaN codes
    codes &= 0xBF                                  # |value| < 2: sums stay well inside bf16's range
    b_dev = codes.view(torch.float8_e4m3fn)
    cols = torch.tensor(sorted({0, 1, 127, 128, chunk - 1, chunk, chunk + 1, chunk + 255, N - 129, N - 2, N - 1}
                               | set(torch.randint(0, N, (64,), generator=g).tolist())))
    b_cols = b_dev[cols.to(device)].cpu()
    for M, kernel in ((8, "stream"), (40, "tiled")):
        a = fp8_randn((M, K), g)
        sa, sb = torch.tensor([0.02]), torch.tensor([0.01])
        out = matmul(a.to(device), b_dev, trans_b=True, scale_a=sa.to(device), scale_b=sb.to(device), out_dtype=torch.bfloat16)
        used(kernel)
        ref = R.ref_gemm_per_tensor(a, b_cols, sa, sb, trans_b=True)
        check(out[:, cols.to(device)], ref, what=f"2 GiB weight, per-tensor, M={M}")
        # block scales: (M, K/128) and (ceil(N/128), K/128)
        As = torch.rand(M, K // 128, generator=g) * 0.02 + 0.01
        Bs = torch.rand((N + 127) // 128, K // 128, generator=g) * 0.02 + 0.01
        out = w8a8_block_fp8_matmul(a.to(device), b_dev, As.to(device), Bs.to(device), [128, 128], torch.bfloat16)
        used(kernel)
        a_deq = a.float().view(M, K // 128, 128) * As[:, :, None]
        b_deq = b_cols.float().view(len(cols), K // 128, 128) * Bs[cols // 128][:, :, None]
        ref = (a_deq.reshape(M, K).double() @ b_deq.reshape(len(cols), K).double().T).to(torch.bfloat16)
        check(out[:, cols.to(device)], ref, what=f"2 GiB weight, block scales, M={M}")
        assert _lib.last_config()["PIECES"] == 2
    del codes, b_dev


def test_column_piece_with_more_than_one_row_chunk(device):
    """Both chunkings at once: M = 16384, N = 1280, K = 131072 is 320 tiles of 256 x 256 (1.25 rounds), so columns
    0 .. 1023 and 1024 .. 1279 run as two pieces of a C that is 1280 wide, and the activations are 2 GiB, so every piece
    walks its rows in two chunks (32-bit byte offsets).  The second row chunk of a piece must land at row stride 1280, not
    at the piece's own width: rows either side of the chunk boundary, in both column pieces, against the oracle."""
    M, N, K = 16384, 1280, 131072
    g = _g(5)
    codes = torch.randint(0, 256, (M, K), dtype=torch.uint8, device=device)
    codes[(codes & 0x7F) == 0x7F] = 0x38
    codes &= 0xBF
    a_dev = codes.view(FP8)
    b = fp8_randn((N, K), g, 0.5)
    sa, sb = torch.tensor([0.02]), torch.tensor([0.01])
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=device)
    _lib.fp8_gemm(out, a_dev, b.to(device), sa.to(device), sb.to(device), False, True, 1.0, 0.0, None)
    cfg = _lib.last_config()
    assert cfg["KERNEL_NAME"] == "tiled" and cfg["PIECES"] == 2, cfg
    boundary = ((1 << 31) - 1) // K // 256 * 256     # first row of the second row chunk
    rows = torch.tensor([0, 1, 255, boundary - 1, boundary, boundary + 1, boundary + 200, M - 1])
    ref = R.ref_gemm_per_tensor(a_dev[rows.to(device)].cpu(), b, sa, sb, trans_b=True)
    check(out[rows.to(device)], ref, what="column pieces x row chunks")
    assert not torch.isnan(out.float()).any()
    del codes, a_dev, out


@pytest.mark.parametrize("block_size", [[64, 64], [64, 128], [256, 32], [128, 256], [48, 80], [256, 128], [256, 256], [384, 512]])
@pytest.mark.parametrize("M,N,K", [(128, 128, 128), (256, 256, 256), (33, 200, 328), (16, 1000, 1536), (700, 520, 1024)])
def test_block_scaled_quantization_blocks_other_than_128(device, block_size, M, N, K):
    """w8a8_block_fp8_matmul with the reference's block_size=[block_n, block_k] argument
    (src/tilegym/suites/unsloth/cutile/fp8.py:388-446) for blocks other than 128 x 128, ragged at both edges.  Blocks that
    are multiples of 128 x 128 run on the MFMA kernels (their scales are written out per 128 x 128 block first), the others
    on the software-decode kernel; all must match the oracle like every other form."""
    bn, bk = block_size
    g = _g(M + N + K + bn * 3 + bk)
    A, B = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.5)
    As = torch.rand(M, -(-K // bk), generator=g) * 0.05 + 0.01
    Bs = torch.rand(-(-N // bn), -(-K // bk), generator=g) * 0.05 + 0.01
    ref = R.ref_w8a8_block_fp8_matmul(A, B, As, Bs, block_size, torch.bfloat16)
    out = w8a8_block_fp8_matmul(A.to(device), B.to(device), As.to(device), Bs.to(device), block_size, torch.bfloat16)
    cfg = _lib.last_config()
    if bn % 128 == 0 and bk % 128 == 0:   # (K = 328 runs zero-padded to 384)
        assert cfg["KERNEL_NAME"] in ("tiled", "stream", "skinny") and (cfg["QUANT_BLOCK_N"], cfg["QUANT_BLOCK_K"]) == (bn, bk), cfg
    else:
        assert cfg["KERNEL_NAME"] == "fallback", cfg
    check(out, ref, what=f"block_size={block_size} M={M} N={N} K={K}")
    # the same problem described with 128 x 128 scales has other shapes: the library must refuse the mismatch
    if (As.shape[1], Bs.shape) != (-(-K // 128), (-(-N // 128), -(-K // 128))):
        with pytest.raises(RuntimeError):
            _lib.fp8_gemm(out, A.to(device), B.to(device), As.to(device), Bs.to(device), False, True, 1.0, 0.0, None)


@pytest.mark.parametrize("bn,bk", [(64, 64), (128, 64), (256, 32)])
def test_ragged_quantization_blocks_other_than_128(device, bn, bk):
    """ragged_block_scaled_bmm derives the quantization block from the scale tensor's shape, as the reference does
    (src/tilegym/suites/flashinfer/cutile/gemm/ragged_block_scaled_bmm.py:535-537): blocks other than 128 x 128 run on the
    software-decode kernel and match the oracle, empty experts included."""
    g = _g(900 + bn + bk)
    Q, N, K = 5, 256, 384
    sizes = [37, 0, 130, 1, 64]
    ptr = torch.tensor([0] + list(torch.tensor(sizes).cumsum(0)), dtype=torch.int32)
    total = int(ptr[-1])
    a, b = fp8_randn((total, K), g), fp8_randn((Q, N, K), g, 0.5)
    a_s = torch.rand(total, K // bk, generator=g) * 0.05 + 0.01
    b_s = torch.rand(Q, N // bn, K // bk, generator=g) * 0.05 + 0.01
    ref = R.ref_ragged_block_scaled_bmm(a, b, a_s, b_s, ptr, block_n=bn, block_k=bk)
    out = ragged_block_scaled_bmm(a.to(device), b.to(device), a_s.to(device), b_s.to(device), ptr.to(device), max(sizes))
    used("fallback")
    check(out, ref, what=f"ragged, blocks {bn}x{bk}")


@pytest.mark.parametrize("block_scaled", [False, True])
def test_columns_split_where_256_tiles_leave_the_last_round_mostly_empty(device, block_scaled):
    """M = 1024, N = 16896: 4 x 66 = 264 tiles of 256 x 256 are 1.03 rounds of the chip.  The library computes the 64
    column tiles that fill one round with 256 x 256 tiles and the remaining 512 columns as a problem of its own
    (C's row stride stays N).  Same bits as one schedule for everything, and the oracle on sampled rows."""
    M, N, K = 1024, 16896, 256
    g = _g(4242 + block_scaled)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.5)
    if block_scaled:
        sa = torch.rand(M, K // 128, generator=g) * 0.05 + 0.01
        sb = torch.rand(N // 128, K // 128, generator=g) * 0.05 + 0.01
    else:
        sa, sb = torch.tensor([0.03]), torch.tensor([0.02])
    ad, bd, sad, sbd = a.to(device), b.to(device), sa.to(device), sb.to(device)
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=device)
    _lib.fp8_gemm(out, ad, bd, sad, sbd, False, True, 1.0, 0.0, None)
    cfg = _lib.last_config()          # the schedule of the first piece (the columns that fill whole rounds) and the piece count
    assert cfg["KERNEL_NAME"] == "tiled" and (cfg["BLOCK_M"], cfg["BLOCK_N"], cfg["PIECES"]) == (256, 256, 2), cfg
    one = torch.empty_like(out)
    _lib.fp8_gemm(one, ad, bd, sad, sbd, False, True, 1.0, 0.0, {"KERNEL": "tiled", "BLOCK_M": 256, "BLOCK_N": 256})
    assert torch.equal(out, one)
    rows = _rows_stratified(M, 8, seed=17)
    if block_scaled:
        ref = R.ref_w8a8_block_fp8_matmul(a[rows], b, sa[rows], sb, [128, 128], torch.bfloat16)
    else:
        ref = R.ref_gemm_per_tensor(a[rows], b, sa, sb, trans_b=True)
    check(out[rows.to(device)], ref, what=f"column split, block_scaled={block_scaled}")
    # beta != 0 reads each piece's own part of C
    c0 = torch.randn(M, N, generator=g).to(torch.bfloat16)
    c = c0.clone().to(device)
    if not block_scaled:
        _lib.fp8_gemm(c, ad, bd, sad, sbd, False, True, 1.0, 1.0, None)
        ref2 = (R.ref_gemm_per_tensor(a[rows], b, sa, sb, trans_b=True, out_dtype=torch.float32) + c0[rows].float()).to(torch.bfloat16)
        check(c[rows.to(device)], ref2, what="column split, beta = 1")


@pytest.mark.parametrize("block_scaled", [False, True])
def test_rows_split_where_256_tiles_leave_the_last_round_mostly_empty(device, block_scaled):
    """M = 5120, N = 4096: 20 x 16 = 320 tiles of 256 x 256; no whole number of column tiles fills a round, sixteen row
    tiles do: rows 0 .. 4095 run with 256 x 256 tiles, the last 1024 rows as a problem of their own."""
    M, N, K = 5120, 4096, 128
    g = _g(4343 + block_scaled)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.5)
    if block_scaled:
        sa = torch.rand(M, 1, generator=g) * 0.05 + 0.01
        sb = torch.rand(N // 128, 1, generator=g) * 0.05 + 0.01
    else:
        sa, sb = torch.tensor([0.03]), torch.tensor([0.02])
    ad, bd, sad, sbd = a.to(device), b.to(device), sa.to(device), sb.to(device)
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=device)
    _lib.fp8_gemm(out, ad, bd, sad, sbd, False, True, 1.0, 0.0, None)
    cfg = _lib.last_config()
    assert cfg["KERNEL_NAME"] == "tiled" and (cfg["BLOCK_M"], cfg["BLOCK_N"], cfg["PIECES"]) == (256, 256, 2), cfg
    one = torch.empty_like(out)
    _lib.fp8_gemm(one, ad, bd, sad, sbd, False, True, 1.0, 0.0, {"KERNEL": "tiled", "BLOCK_M": 256, "BLOCK_N": 256})
    assert torch.equal(out, one)
    rows = _rows_stratified(M, 4, seed=18)
    if block_scaled:
        ref = R.ref_w8a8_block_fp8_matmul(a[rows], b, sa[rows], sb, [128, 128], torch.bfloat16)
    else:
        ref = R.ref_gemm_per_tensor(a[rows], b, sa, sb, trans_b=True)
    check(out[rows.to(device)], ref, what=f"row split, block_scaled={block_scaled}")


def test_fallback_kernel_takes_more_rows_than_one_grid_dimension_holds(device):
    """The software-decode kernel walks rows grid-stride: 300 000 rows (above 4 x 65 535)."""
    M, N, K = 300_000, 8, 24
    g = _g(78)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.5)
    out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=0.5, scale_b=0.25, out_dtype=torch.bfloat16,
                 kernel_configs={"KERNEL": "fallback"})
    used("fallback")
    rows = torch.tensor([0, 1, 262139, 262140, 262143, 262144, 299_999] + torch.randint(0, M, (200,), generator=g).tolist())
    check(out[rows.to(device)], R.ref_gemm_per_tensor(a[rows], b, 0.5, 0.25, trans_b=True), what="fallback, 300000 rows")


# ----------------------------------------------------------------------------- skinny
@pytest.mark.parametrize("M", [1, 3, 8, 16, 17, 33, 64])
@pytest.mark.parametrize("N,K,rg,split,waves", [(1000, 512, 1, 1, 4), (4096, 1024, 2, 2, 8), (520, 2064, 4, 4, 16), (256, 128, 1, 1, 16)])
def test_per_tensor_skinny(device, M, N, K, rg, split, waves):
    g = _g(M * 7 + N)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.02)
    sa, sb = torch.tensor([0.011]), torch.tensor([0.0003])
    ref = R.ref_gemm_per_tensor(a, b, sa, sb, trans_b=True)
    out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=sa.to(device), scale_b=sb.to(device),
                 out_dtype=torch.bfloat16, kernel_configs={"KERNEL": "skinny", "ROW_GROUPS": rg, "SPLIT_K": split, "WAVES": waves})
    cfg = used("skinny")
    assert cfg["WAVES"] == waves
    check(out, ref, what=f"skinny M={M} N={N} K={K} rg={rg} split={split} waves={waves}")


@pytest.mark.parametrize("M", [1, 5, 16, 17, 40, 64])
@pytest.mark.parametrize("N,K,split", [(1000, 1024, 1), (520, 4096, 1), (264, 2064, 1), (256, 9216, 1), (128, 16384, 4), (72, 512, 1)])
def test_per_tensor_stream(device, M, N, K, split):
    """Weight streaming through LDS: K tails inside a 1 KiB piece, ragged N, single and double buffering, split-K."""
    g = _g(M * 11 + N + K)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.02)
    sa, sb = torch.tensor([0.011]), torch.tensor([0.0003])
    ref = R.ref_gemm_per_tensor(a, b, sa, sb, trans_b=True)
    out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=sa.to(device), scale_b=sb.to(device),
                 out_dtype=torch.bfloat16, kernel_configs={"KERNEL": "stream", "SPLIT_K": split})
    cfg = used("stream")
    assert cfg["SPLIT_K"] == split
    check(out, ref, what=f"stream M={M} N={N} K={K} split={split}")


@pytest.mark.parametrize("M", [1, 5, 8, 16])
@pytest.mark.parametrize("N,K", [(1000, 1024), (520, 14336), (264, 2064), (256, 9216), (72, 512)])
def test_per_tensor_stream_eight_waves(device, M, N, K):
    """The streaming kernel with eight waves per workgroup splitting K (long K over few weight rows, one launch):
    more waves than 1 KiB pieces, K tails inside a piece, ragged N."""
    g = _g(M * 17 + N + K)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.02)
    sa, sb = torch.tensor([0.011]), torch.tensor([0.0003])
    ref = R.ref_gemm_per_tensor(a, b, sa, sb, trans_b=True)
    out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=sa.to(device), scale_b=sb.to(device),
                 out_dtype=torch.bfloat16, kernel_configs={"KERNEL": "stream", "WAVES": 8})
    cfg = used("stream")
    assert cfg["WAVES"] == 8 and cfg["SPLIT_K"] == 1
    check(out, ref, what=f"stream 8 waves M={M} N={N} K={K}")


def test_stream_eight_waves_is_the_default_for_long_k_one_or_two_rows(device):
    g = _g(5)
    a, b = fp8_randn((2, 14336), g), fp8_randn((4096, 14336), g, 0.02)
    ref = R.ref_gemm_per_tensor(a, b, 0.01, 0.02, trans_b=True)
    out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=0.01, scale_b=0.02, out_dtype=torch.bfloat16)
    cfg = used("stream")
    assert cfg["WAVES"] == 8 and cfg["SPLIT_K"] == 1, cfg
    check(out, ref, what="down projection, M=2")


@pytest.mark.parametrize("M", [4, 16])
def test_stream_wide_with_one_workgroup_per_compute_unit_is_the_default_for_long_k(device, M):
    """4096 x 14336: 64 row blocks, four K splits = 256 workgroups."""
    g = _g(6 + M)
    a, b = fp8_randn((M, 14336), g), fp8_randn((4096, 14336), g, 0.02)
    ref = R.ref_gemm_per_tensor(a, b, 0.01, 0.02, trans_b=True)
    out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=0.01, scale_b=0.02, out_dtype=torch.bfloat16)
    cfg = used("stream")
    assert cfg["ROW_GROUPS"] == 4 and cfg["SPLIT_K"] == 4 and cfg["WAVES"] == 4, cfg
    check(out, ref, what=f"down projection, M={M}")


def _wide_form(K, in_flight):
    """WAVES as tg_last_config reports it for the wide form: 4 = two half pieces per wave in flight (K % 128 == 0 only),
    1 = one 1 KiB piece."""
    return 4 if in_flight == 2 and K % 128 == 0 else 1


@pytest.mark.parametrize("in_flight", [2, 1])
@pytest.mark.parametrize("M", [1, 3, 8, 16])
@pytest.mark.parametrize("N,K,split", [(1000, 1024, 1), (520, 4096, 1), (264, 2064, 1), (128, 16384, 4), (72, 512, 1), (4096, 3072, 2),
                                       (200, 1408, 1), (136, 128, 1), (520, 2432, 2), (264, 11008, 3)])
def test_per_tensor_stream_wide(device, M, N, K, split, in_flight):
    """64 weight rows per workgroup with the activation piece shared through LDS: ragged N (also inside a
    workgroup's 64 rows), K tails inside a 1 KiB piece, split-K, every M up to 16; both forms of the piece pipeline."""
    g = _g(M * 13 + N + K)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.02)
    sa, sb = torch.tensor([0.011]), torch.tensor([0.0003])
    ref = R.ref_gemm_per_tensor(a, b, sa, sb, trans_b=True)
    kc = {"KERNEL": "stream", "ROW_GROUPS": 4, "SPLIT_K": split}
    if in_flight == 1:
        kc["WAVES"] = 1
    out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=sa.to(device), scale_b=sb.to(device),
                 out_dtype=torch.bfloat16, kernel_configs=kc)
    cfg = used("stream")
    assert cfg["ROW_GROUPS"] == 4 and cfg["SPLIT_K"] == split and cfg["WAVES"] == _wide_form(K, in_flight), cfg
    check(out, ref, what=f"stream wide M={M} N={N} K={K} split={split}")


@pytest.mark.parametrize("in_flight", [2, 1])
@pytest.mark.parametrize("M", [1, 7, 16])
@pytest.mark.parametrize("N,K,split", [(640, 1024, 1), (264, 2304, 1), (1152, 5120, 2), (128, 12288, 6), (1000, 512, 1),
                                       (200, 1408, 1), (136, 128, 1), (520, 2432, 2), (264, 11008, 3)])
def test_block_scaled_stream_wide(device, M, N, K, split, in_flight):
    case = W.block_scaled_case(M, N, K, seed=M + N)
    ref = R.ref_w8a8_block_fp8_matmul(case.a, case.b, case.scale_a, case.scale_b, None, torch.bfloat16)
    d = case.to(device)
    kc = {"KERNEL": "stream", "ROW_GROUPS": 4, "SPLIT_K": split}
    if in_flight == 1:
        kc["WAVES"] = 1
    out = w8a8_block_fp8_matmul(d.a, d.b, d.scale_a, d.scale_b, None, torch.bfloat16, kernel_configs=kc)
    cfg = used("stream")
    assert cfg["ROW_GROUPS"] == 4 and cfg["SPLIT_K"] == split and cfg["WAVES"] == _wide_form(K, in_flight), cfg
    check(out, ref, what=f"block-scaled stream wide M={M} N={N} K={K} split={split}")


@pytest.mark.parametrize("M", [17, 24, 32])
@pytest.mark.parametrize("N,K,split", [(1000, 1024, 1), (520, 4096, 2), (72, 512, 1), (4096, 3072, 3), (200, 1408, 1), (264, 2432, 2)])
def test_stream_wide_two_row_tiles(device, M, N, K, split):
    """17 .. 32 activation rows: two tiles of 16 in the wide form's activation piece (per-tensor and block-scaled)."""
    g = _g(M * 7 + N + K)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.02)
    sa, sb = torch.tensor([0.011]), torch.tensor([0.0003])
    kc = {"KERNEL": "stream", "ROW_GROUPS": 4, "SPLIT_K": split}
    out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=sa.to(device), scale_b=sb.to(device),
                 out_dtype=torch.bfloat16, kernel_configs=kc)
    cfg = used("stream")
    assert cfg["ROW_GROUPS"] == 4 and cfg["SPLIT_K"] == split and cfg["WAVES"] == 4, cfg
    check(out, R.ref_gemm_per_tensor(a, b, sa, sb, trans_b=True), what=f"stream wide, two row tiles M={M} N={N} K={K}")
    case = W.block_scaled_case(M, N, K, seed=M + N)
    d = case.to(device)
    out = w8a8_block_fp8_matmul(d.a, d.b, d.scale_a, d.scale_b, None, torch.bfloat16, kernel_configs=kc)
    cfg = used("stream")
    assert cfg["ROW_GROUPS"] == 4 and cfg["SPLIT_K"] == split, cfg
    check(out, R.ref_w8a8_block_fp8_matmul(case.a, case.b, case.scale_a, case.scale_b, None, torch.bfloat16),
          what=f"block-scaled stream wide, two row tiles M={M} N={N} K={K}")


@pytest.mark.parametrize("bn", [56, 48, 40, 24, 12])
@pytest.mark.parametrize("M,N,K,split", [(5, 1000, 1024, 1), (16, 1000, 1152, 1), (30, 520, 2048, 2), (16, 4096, 640, 1)])
def test_stream_wide_with_fewer_rows_per_workgroup(device, bn, M, N, K, split):
    """BLOCK_N of the wide streaming form: 4 x the weight rows a wave owns (64 by default).  Rows a wave does not own are
    neither loaded nor stored; with block scales a wave's rows may lie on both sides of a 128-row boundary of the weight
    scales (bn = 56, 48, 40, 24: rows 112 .. 139 etc.) and every output takes the scale of its own block.  N that is no
    multiple of bn, one and two tiles of activation rows, a short last piece, split-K."""
    g = _g(bn * 11 + M + N + K)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.02)
    sa, sb = torch.tensor([0.011]), torch.tensor([0.0003])
    kc = {"KERNEL": "stream", "ROW_GROUPS": 4, "SPLIT_K": split, "BLOCK_N": bn}
    out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=sa.to(device), scale_b=sb.to(device),
                 out_dtype=torch.bfloat16, kernel_configs=kc)
    cfg = used("stream")
    assert (cfg["ROW_GROUPS"], cfg["SPLIT_K"], cfg["WAVES"], cfg["BLOCK_N"]) == (4, split, 4, bn), cfg
    check(out, R.ref_gemm_per_tensor(a, b, sa, sb, trans_b=True), what=f"stream wide, {bn} rows per workgroup, M={M} N={N} K={K}")
    case = W.block_scaled_case(M, N, K, seed=M + N + bn)
    d = case.to(device)
    out = w8a8_block_fp8_matmul(d.a, d.b, d.scale_a, d.scale_b, None, torch.bfloat16, kernel_configs=kc)
    cfg = used("stream")
    assert (cfg["ROW_GROUPS"], cfg["SPLIT_K"], cfg["BLOCK_N"]) == (4, split, bn), cfg
    check(out, R.ref_w8a8_block_fp8_matmul(case.a, case.b, case.scale_a, case.scale_b, None, torch.bfloat16),
          what=f"block-scaled stream wide, {bn} rows per workgroup, M={M} N={N} K={K}")


def test_stream_wide_picks_its_rows_per_workgroup(device):
    """12288 weight rows in workgroups of 48 are one workgroup per compute unit (64: 192 workgroups, a quarter of the chip
    idle); 8192 x 8192 takes 32 rows per workgroup in one launch instead of 64 and two K splits."""
    g = _g(4848)
    for N, K, bn in [(12288, 1024, 48), (8192, 8192, 32)]:
        a, b = fp8_randn((16, K), g), fp8_randn((N, K), g, 0.02)
        out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=0.01, scale_b=0.02, out_dtype=torch.bfloat16)
        cfg = used("stream")
        assert (cfg["ROW_GROUPS"], cfg["SPLIT_K"], cfg["BLOCK_N"]) == (4, 1, bn), cfg
        rows = torch.arange(0, N, 37)
        check(out[:, rows.to(device)], R.ref_gemm_per_tensor(a, b[rows], 0.01, 0.02, trans_b=True), what=f"{N} x {K}, rows per workgroup")


@pytest.mark.parametrize("bn", [72, 96, 112, 120])
@pytest.mark.parametrize("M,N,K,split", [(64, 1000, 1024, 1), (40, 2304, 512, 1), (130, 520, 2048, 2), (17, 4096, 640, 1)])
def test_deep_tile_kernel_over_fewer_weight_rows_per_tile(device, bn, M, N, K, split):
    """BLOCK_N = 72 .. 120 with BLOCK_M = 64: the 64 x 128 tile kernel with tiles that cover fewer weight rows (the rest of
    the weight slab is neither loaded nor stored).  N that is no multiple of the tile, several row tiles, split-K."""
    g = _g(bn * 13 + M + N + K)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.02)
    kc = {"KERNEL": "tiled", "BLOCK_M": 64, "BLOCK_N": bn, "SPLIT_K": split}
    out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=0.011, scale_b=0.0003, out_dtype=torch.bfloat16, kernel_configs=kc)
    cfg = used("tiled")
    assert (cfg["BLOCK_M"], cfg["BLOCK_N"], cfg["SPLIT_K"]) == (64, bn, split), cfg
    check(out, R.ref_gemm_per_tensor(a, b, 0.011, 0.0003, trans_b=True), what=f"64 x {bn} tiles, M={M} N={N} K={K}")
    full = matmul(a.to(device), b.to(device), trans_b=True, scale_a=0.011, scale_b=0.0003, out_dtype=torch.bfloat16,
                  kernel_configs={"KERNEL": "tiled", "BLOCK_M": 64, "BLOCK_N": 128, "SPLIT_K": split})
    assert torch.equal(out, full)     # the same products in the same order, whatever the tile's width


@pytest.mark.parametrize("bm,bn", [(64, 128), (96, 128), (128, 128), (160, 128), (160, 192), (192, 192)])
@pytest.mark.parametrize("dm,dn,K,split", [(0, 0, 128, 1), (-1, -8, 256, 1), (1, 8, 384, 2), (17, -3, 640, 1), (-33, 72, 2176, 3)])
def test_ring_tiles(device, bm, bn, dm, dn, K, split):
    """The tiles with waves of their own for the loads: rows and columns that end inside a tile, fewer K steps than stages,
    split K.  Same bits as the 128 x 128 tile kernel (the same products in the same order), and the oracle's result."""
    M, N = 2 * bm + dm, bn + dn
    g = _g(bm + bn + K)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.5)
    ad, bd = a.to(device), b.to(device)
    kc = {"KERNEL": "tiled", "BLOCK_M": bm, "BLOCK_N": bn, "SPLIT_K": split, "WAVES": 8}
    for dtype in (torch.bfloat16, torch.float32, torch.float8_e4m3fn):
        out = matmul(ad, bd, trans_b=True, scale_a=0.37, scale_b=0.5, out_dtype=dtype, kernel_configs=kc)
        cfg = used("tiled")
        assert (cfg["BLOCK_M"], cfg["BLOCK_N"], cfg["WAVES"]) == (bm, bn, 8), cfg
        base = matmul(ad, bd, trans_b=True, scale_a=0.37, scale_b=0.5, out_dtype=dtype,
                      kernel_configs={"KERNEL": "tiled", "BLOCK_M": 128, "BLOCK_N": 128, "SPLIT_K": cfg["SPLIT_K"]})
        assert _lib.last_config()["WAVES"] != 8
        assert torch.equal(out.view(torch.uint8), base.view(torch.uint8))
        if dtype == torch.bfloat16:
            check(out, R.ref_gemm_per_tensor(a, b, 0.37, 0.5, trans_b=True), what=f"ring {bm}x{bn} M={M} N={N} K={K}")


@pytest.mark.parametrize("bm,bn", [(64, 32), (32, 64), (64, 64), (32, 128), (256, 128)])
@pytest.mark.parametrize("dm,dn,K,split", [(0, 0, 128, 1), (-1, -8, 1664, 1), (1, 8, 384, 2), (17, -3, 640, 1), (-15, 72, 2176, 3)])
def test_ring_tiles_narrow_and_tall(device, bm, bn, dm, dn, K, split):
    """The same for the tiles of 32 and 64 columns, 32 rows and 256 rows (13 K steps: one more than the twelve stages; one wave
    column, one or two column tiles per wave)."""
    test_ring_tiles(device, bm, bn, dm, dn, K, split)


@pytest.mark.parametrize("M,N,K,want", [(24, 12288, 1280, (32, 64)), (33, 12288, 1280, (64, 64)), (256, 4096, 1280, (64, 64)), (128, 4096, 1408, (64, 32)),
                                        (256, 28672, 1280, (256, 128))])
def test_narrow_and_tall_ring_tiles_are_chosen(device, M, N, K, want):
    g = _g(M + K)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.02)
    out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=0.01, scale_b=0.02, out_dtype=torch.float16)
    cfg = used("tiled")
    assert (cfg["BLOCK_M"], cfg["BLOCK_N"], cfg["WAVES"]) == want + (8,), cfg
    cols = torch.arange(0, N, 13)
    check(out[:, cols.to(device)], R.ref_gemm_per_tensor(a, b[cols], 0.01, 0.02, trans_b=True, out_dtype=torch.float16), what=f"M={M} N={N} K={K}")


@pytest.mark.parametrize("kind,M,N,K,ring", [
    ("nk", 88, 1520, 5248, False), ("nk", 90, 4096, 4096, True), ("nk", 128, 4096, 4096, False), ("nk", 256, 4096, 4096, True), ("nk", 482, 9216, 3072, False),
    ("block", 100, 1120, 8320, False),
    ("kn", 16, 1024, 1920, False), ("kn", 16, 10240, 1920, True), ("kn", 256, 4096, 4096, False), ("kn", 16, 4096, 4096, True),
    ("nk", 24, 12288, 5120, True), ("nk", 30, 17072, 5120, False), ("nk", 40, 12288, 5120, True), ("nk", 64, 12288, 5120, False), ("nk", 64, 6144, 4096, False),
    ("nk", 50, 4096, 14336, True), ("nk", 50, 2048, 5120, False), ("nk", 24, 22032, 2560, False),
    ("block", 24, 12288, 5120, True), ("block", 20, 18576, 2944, False), ("block", 28, 3520, 4864, False), ("block", 17, 1520, 2304, False), ("block", 17, 8192, 8192, False), ("block", 21, 5120, 5120, False)])
def test_narrow_ring_tiles_are_chosen_where_they_hold_from_memory(device, kind, M, N, K, ring):
    """Either side of the lines between the narrow ring tiles (and 256 x 128), and the kernels that are ahead of them when the weight is not in the caches."""
    zeros = lambda *shape: torch.zeros(*shape, dtype=torch.uint8, device=device).view(FP8)  # noqa: E731
    c = torch.empty(M, N, dtype=torch.bfloat16, device=device)
    one = torch.ones(1, device=device)
    sa, sb = (torch.ones(M, K // 128, device=device), torch.ones(-(-N // 128), K // 128, device=device)) if kind == "block" else (one, one)
    _lib.fp8_gemm(c, zeros(M, K), zeros(K, N) if kind == "kn" else zeros(N, K), sa, sb, trans_b=kind != "kn")
    cfg = _lib.last_config()
    narrow = cfg["WAVES"] == 8 and (cfg["BLOCK_N"] <= 64 or cfg["BLOCK_M"] in (32, 256))
    assert (cfg["KERNEL_NAME"] == "tiled" and narrow) == ring, cfg


@pytest.mark.parametrize("block_scaled", [False, True])
@pytest.mark.parametrize("M,N,K,want", [(16, 25616, 4096, (32, 128)), (17, 25616, 4096, (32, 128)), (33, 32768, 4096, (64, 128)), (64, 25604, 4096, (64, 128)),
                                        (16, 16360, 8192, (32, 64)), (50, 14728, 8192, (64, 64)), (65, 25616, 4096, (96, 128)), (128, 25616, 4096, (128, 128)),
                                        (160, 25616, 4096, (160, 128)), (256, 25616, 4096, (256, 128)), (250, 20112, 5120, (256, 128))])
def test_ring_tiles_over_weights_from_memory(device, block_scaled, M, N, K, want):
    """Weights of 100 MB and more on one row tile: workgroups start at different K steps and go round, over chunks of activation scales
    that end inside the round; N that ends inside a tile, first and last row counts of the tiles.  Small integers and scales
    that are powers of two: every sum is exact in fp32, whatever its order."""
    if block_scaled and M > 160:
        pytest.skip("per-tensor tiles")
    g = torch.Generator(device=device).manual_seed(M + N)
    a, b = (torch.randint(-2, 3, s, generator=g, device=device).float() for s in ((M, K), (N, K)))
    a8, b8 = a.to(FP8), b.to(FP8)
    if block_scaled:
        sa, sb = (2.0 ** torch.randint(-1, 2, s, generator=g, device=device).float() for s in ((M, K // 128), ((N + 127) // 128, K // 128)))
        a *= sa.repeat_interleave(128, 1)
        b *= sb.repeat_interleave(128, 0)[:N].repeat_interleave(128, 1)
    else:
        sa = sb = torch.full((1,), 0.5, device=device)
    out = torch.full((M, N), float("nan"), device=device)
    cfg = {"KERNEL": "tiled", "BLOCK_M": want[0], "BLOCK_N": want[1], "SPLIT_K": 1, "WAVES": 8, "ROW_GROUPS": 1}
    if block_scaled or 17 <= M <= 64:  # (the library's own choice there)
        cfg = None
    _lib.fp8_gemm(out, a8, b8, sa, sb, False, True, 1.0, 0.0, cfg)
    got = used("tiled")
    assert (got["BLOCK_M"], got["BLOCK_N"], got["WAVES"], got["SPLIT_K"], got["ROW_GROUPS"]) == want + (8, 1, 1), got
    assert torch.equal(out, (a @ b.t()) * (1.0 if block_scaled else 0.25))


@pytest.mark.parametrize("block_scaled", [False, True])
@pytest.mark.parametrize("M,bm,bn,K", [(30, 32, 128, 4096), (61, 64, 64, 8192), (150, 160, 128, 4096)])
def test_rotated_sums_are_asked_for_and_named(device, block_scaled, M, bm, bn, K):
    """A tile asked for by name alone sums in the order of every other kernel (the bits of 128 x 128 tiles), with ROW_GROUPS = 1 in the
    rotated one; either within the oracle's tolerance on operands of ordinary values, with either scale tensor missing and with beta."""
    N = 100000000 // K // 128 * 128 + 128
    g = torch.Generator(device=device).manual_seed(M + K)
    a, b = torch.randn(M, K, generator=g, device=device).to(FP8), (torch.randn(N, K, generator=g, device=device) * 0.5).to(FP8)
    if block_scaled:
        sa, sb = torch.rand(M, K // 128, generator=g, device=device) * 0.1 + 0.01, torch.rand(N // 128, K // 128, generator=g, device=device) * 0.1 + 0.01
    else:
        sa, sb = torch.full((1,), 0.5, device=device), torch.full((1,), 0.25, device=device)
    kc = {"KERNEL": "tiled", "BLOCK_M": bm, "BLOCK_N": bn, "SPLIT_K": 1, "WAVES": 8}
    blocks = torch.arange(0, N // 128, 97)
    cols = (blocks[:, None] * 128 + torch.arange(128)).flatten()
    c0 = torch.randn(M, N, generator=g, device=device)
    for s1, s2, dtype, beta in ((sa, sb, torch.bfloat16, 0.0), (None, sb, torch.float32, 0.0), (sa, None, torch.float16, 0.0), (sa, sb, torch.float32, 0.5)):
        plain, turned, base = (c0.to(dtype, copy=True) for _ in range(3))
        _lib.fp8_gemm(plain, a, b, s1, s2, False, True, 1.0, beta, kc)
        assert _lib.last_config()["ROW_GROUPS"] != 1 and _lib.last_config()["BLOCK_M"] == bm
        _lib.fp8_gemm(base, a, b, s1, s2, False, True, 1.0, beta, {"KERNEL": "tiled", "BLOCK_M": 128, "BLOCK_N": 128, "SPLIT_K": 1})
        assert torch.equal(plain, base)
        _lib.fp8_gemm(turned, a, b, s1, s2, False, True, 1.0, beta, {**kc, "ROW_GROUPS": 1})
        assert _lib.last_config()["ROW_GROUPS"] == 1 and _lib.last_config()["BLOCK_M"] == bm
        f = lambda t, scale: t.cpu().double() if scale is None else t.cpu().double() * (scale.cpu().double() if scale.numel() == 1 else scale.cpu().double().repeat_interleave(128, 1))  # noqa: E731
        bs = s2 if s2 is None or not block_scaled else s2[blocks.to(device)].repeat_interleave(128, 0)
        ref = f(a.float(), s1) @ f(b[cols.to(device)].float(), bs).t() + beta * c0[:, cols.to(device)].cpu().double()
        err = (turned[:, cols.to(device)].cpu().double() - ref).norm() / ref.norm()
        # about twice what is measured: f32 sums of the matrix unit 2.8e-5, the outputs' rounding 1.7e-3 (bf16) and 2.1e-4 (f16)
        assert err < {torch.float32: 6e-5, torch.float16: 6e-4, torch.bfloat16: 4e-3}[dtype], err


@pytest.mark.parametrize("block_scaled", [False, True])
@pytest.mark.parametrize("M,N,K,form", [(1, 8208, 1024, 4), (8, 8208, 1152, 4), (3, 8192, 1024, 1), (3, 6160, 9344, 1), (1, 4096, 9344, 1)])
def test_decode_streams_narrow_or_wide(device, block_scaled, M, N, K, form):
    """Either side of 512 workgroups of 16 weight rows (from there on the wide form); over ten pieces of K with more workgroups than
    compute units (one buffer per wave) and as many (eight waves)."""
    g = _g(N + K)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.2)
    rows = torch.arange(128 * 3)
    if block_scaled:
        sa, sb = torch.rand(M, K // 128, generator=g) * 0.1 + 0.01, torch.rand((N + 127) // 128, K // 128, generator=g) * 0.1 + 0.01
        out = w8a8_block_fp8_matmul(a.to(device), b.to(device), sa.to(device), sb.to(device), None, torch.bfloat16)
        ref = [R.ref_w8a8_block_fp8_matmul(a, b[:384], sa, sb[:3], None, torch.bfloat16)]
    else:
        out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=0.01, scale_b=0.02, out_dtype=torch.bfloat16)
        ref = [R.ref_gemm_per_tensor(a, r, 0.01, 0.02, trans_b=True, out_dtype=torch.bfloat16) for r in (b[:384], b[-40:])]
    cfg = used("stream")
    assert (cfg["ROW_GROUPS"] == 4) == (form == 4), cfg
    check(out[:, rows.to(device)], ref[0], what=f"M={M} N={N} K={K}")
    if not block_scaled:
        check(out[:, -40:], ref[1], what=f"M={M} N={N} K={K}, last rows")


def test_block_scaled_skinny_to_sixteen_rows(device):
    for M, N, K, want in ((8, 4096, 1280, "skinny"), (9, 2048, 1280, "skinny"), (16, 2048, 1536, "skinny"), (8, 1024, 2176, "stream"), (9, 4096, 1024, "stream")):
        g = _g(M + N)
        a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.2)
        sa, sb = torch.rand(M, K // 128, generator=g) * 0.1 + 0.01, torch.rand(N // 128, K // 128, generator=g) * 0.1 + 0.01
        out = w8a8_block_fp8_matmul(a.to(device), b.to(device), sa.to(device), sb.to(device), None, torch.bfloat16)
        used(want)
        check(out, R.ref_w8a8_block_fp8_matmul(a, b, sa, sb, None, torch.bfloat16), what=f"M={M} N={N} K={K}")


@pytest.mark.parametrize("M,N,K,want", [(8, 10240, 5120, (32, 64)), (9, 6144, 4096, (32, 64)), (16, 20480, 2048, (32, 128)), (16, 11008, 4096, None),
                                        (8, 6144, 4096, None), (16, 6400, 3072, None), (12, 7168, 3584, None), (4, 20864, 4096, None), (2, 5504, 6912, None), (9, 12288, 5120, None), (16, 8192, 8192, None)])  # None: streaming
def test_block_scaled_decode_on_ring_tiles(device, M, N, K, want):
    g = _g(M + N)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.5)
    sa, sb = torch.rand(M, K // 128, generator=g) * 0.1 + 0.01, torch.rand(N // 128, K // 128, generator=g) * 0.1 + 0.01
    out = w8a8_block_fp8_matmul(a.to(device), b.to(device), sa.to(device), sb.to(device), None, torch.bfloat16)
    cfg = used("tiled" if want else "stream")
    assert not want or (cfg["BLOCK_M"], cfg["BLOCK_N"], cfg["WAVES"]) == want + (8,), cfg
    rows = torch.arange(0, N, 128 * 5)[:, None].add(torch.arange(128)).flatten()  # (whole scale blocks)
    rows = rows[rows < N]
    check(out[:, rows.to(device)], R.ref_w8a8_block_fp8_matmul(a, b[rows], sa, sb[::5], None, torch.bfloat16), what=f"M={M} N={N} K={K}")


@pytest.mark.parametrize("bm", [64, 96, 128, 160, 192])
@pytest.mark.parametrize("dm,N,K,split", [(0, 256, 128, 1), (-1, 120, 1024, 1), (1, 136, 1152, 2), (17, 257, 2176, 1), (-33, 384, 2304, 2)])
def test_ring_tiles_block_scaled(device, bm, dm, N, K, split):
    """Chunks of activation scales that end inside a K range (8 K steps per chunk: 1, 8, 9, 17 and 2 x 9 steps), rows and
    columns that end inside a tile.  Same bits as the 128 x 128 tile kernel, with either scale tensor missing too."""
    M = 2 * bm + dm
    g = _g(bm + N + K)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.5)
    sa, sb = torch.rand(M, K // 128, generator=g) * 0.1 + 0.01, torch.rand((N + 127) // 128, K // 128, generator=g) * 0.1 + 0.01
    ad, bd, sad, sbd = a.to(device), b.to(device), sa.to(device), sb.to(device)
    kc = {"KERNEL": "tiled", "BLOCK_M": bm, "BLOCK_N": 128, "SPLIT_K": split, "WAVES": 8}
    out, base = (torch.empty(M, N, dtype=torch.bfloat16, device=device) for _ in range(2))
    for s1, s2 in ((sad, sbd), (None, sbd), (sad, None)):
        _lib.fp8_gemm(out, ad, bd, s1, s2, False, True, 1.0, 0.0, kc)
        cfg = used("tiled")
        assert (cfg["BLOCK_M"], cfg["BLOCK_N"], cfg["WAVES"]) == (bm, 128, 8), cfg
        _lib.fp8_gemm(base, ad, bd, s1, s2, False, True, 1.0, 0.0, {"KERNEL": "tiled", "BLOCK_M": 128, "BLOCK_N": 128, "SPLIT_K": cfg["SPLIT_K"]})
        assert _lib.last_config()["WAVES"] != 8
        assert torch.equal(out, base)
        if s1 is not None and s2 is not None:
            check(out, R.ref_w8a8_block_fp8_matmul(a, b, sa, sb, None, torch.bfloat16), what=f"block ring {bm} M={M} N={N} K={K}")


@pytest.mark.parametrize("M,N,K", [(256, 320, 128), (257, 352, 256), (300, 672, 1152), (511, 1024, 384), (700, 960, 2176)])
def test_block_scaled_256_x_320_tile(device, M, N, K):
    """The smallest problem of one tile, last row and column tiles that are moved back over their neighbours (by every distance
    between a column block's edge and a tile's), odd numbers of K steps, chunks of scales that end inside K; beta reads the
    output that a moved tile's neighbour writes.  Same bits as the 256 x 256 tile.  Narrower problems and N that is no
    multiple of 32 take another tile."""
    g = _g(M + N + K)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.5)
    sa, sb = torch.rand(M, K // 128, generator=g) * 0.1 + 0.01, torch.rand((N + 127) // 128, K // 128, generator=g) * 0.1 + 0.01
    args = [t.to(device) for t in (a, b, sa, sb)]
    old = torch.randn(M, N, generator=g).to(torch.bfloat16).to(device)
    for beta in (0.0, 1.0):
        out, base = old.clone(), old.clone()
        _lib.fp8_gemm(out, *args, False, True, 0.7, beta, {"KERNEL": "tiled", "BLOCK_M": 256, "BLOCK_N": 320, "SPLIT_K": 1})
        cfg = used("tiled")
        assert (cfg["BLOCK_M"], cfg["BLOCK_N"]) == (256, 320), cfg
        _lib.fp8_gemm(base, *args, False, True, 0.7, beta, {"KERNEL": "tiled", "BLOCK_M": 256, "BLOCK_N": 256, "SPLIT_K": 1})
        assert torch.equal(out, base)
    check(w8a8_block_fp8_matmul(*args, None, torch.bfloat16, kernel_configs={"KERNEL": "tiled", "BLOCK_M": 256, "BLOCK_N": 320}),
          R.ref_w8a8_block_fp8_matmul(a, b, sa, sb, None, torch.bfloat16), what=f"256 x 320, M={M} N={N} K={K}")
    for m, n in ((255, N), (M, 312), (M, N - 8)):
        few = [args[0][:m], args[1][:n], args[2][:m], args[3][:(n + 127) // 128]]
        out = w8a8_block_fp8_matmul(*[t.contiguous() for t in few], None, torch.bfloat16, kernel_configs={"KERNEL": "tiled", "BLOCK_M": 256, "BLOCK_N": 320})
        assert used("tiled")["BLOCK_N"] != 320
        check(out, R.ref_w8a8_block_fp8_matmul(a[:m], b[:n], sa[:m], sb[:(n + 127) // 128], None, torch.bfloat16))


def test_deep_tile_is_narrowed_to_fill_the_chip(device):
    """28672 weight rows at M = 64: 224 tiles of 128 columns would leave an eighth of the compute units idle; 256 tiles of 112 run."""
    g = _g(112)
    a, b = fp8_randn((64, 512), g), fp8_randn((28672, 512), g, 0.02)
    out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=0.01, scale_b=0.02, out_dtype=torch.bfloat16)
    cfg = _lib.last_config()
    if cfg["KERNEL_NAME"] == "tiled" and cfg["BLOCK_M"] == 64 and cfg["BLOCK_N"] > 64:
        assert cfg["BLOCK_N"] == 112, cfg
    rows = torch.arange(0, 28672, 61)
    check(out[:, rows.to(device)], R.ref_gemm_per_tensor(a, b[rows], 0.01, 0.02, trans_b=True), what="28672 x 512 at M = 64")


@pytest.mark.parametrize("rows", [14, 12, 8, 5])
@pytest.mark.parametrize("M,N,K", [(1, 1000, 1024), (8, 520, 4096), (16, 2050, 1152)])
def test_narrow_stream_form_with_fewer_rows_per_workgroup(device, rows, M, N, K):
    """BLOCK_N of the narrow streaming form: the weight rows a workgroup owns (16 by default).  Same bits as with 16."""
    g = _g(rows * 17 + M + N + K)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.02)
    kc = {"KERNEL": "stream", "ROW_GROUPS": 1, "WAVES": 4, "SPLIT_K": 1, "BLOCK_N": rows}
    out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=0.011, scale_b=0.0003, out_dtype=torch.bfloat16, kernel_configs=kc)
    cfg = used("stream")
    assert (cfg["ROW_GROUPS"], cfg["BLOCK_N"]) == (1, rows), cfg
    check(out, R.ref_gemm_per_tensor(a, b, 0.011, 0.0003, trans_b=True), what=f"narrow stream, {rows} rows per workgroup, M={M} N={N} K={K}")
    kc["BLOCK_N"] = 16
    full = matmul(a.to(device), b.to(device), trans_b=True, scale_a=0.011, scale_b=0.0003, out_dtype=torch.bfloat16, kernel_configs=kc)
    assert torch.equal(out, full)
    if rows == 8:   # block-scaled: a workgroup's rows share one weight scale, so only divisors of 128
        case = W.block_scaled_case(M, N, K, seed=M + N)
        d = case.to(device)
        out = w8a8_block_fp8_matmul(d.a, d.b, d.scale_a, d.scale_b, None, torch.bfloat16, kernel_configs=kc | {"BLOCK_N": 8})
        assert used("stream")["BLOCK_N"] == 8
        check(out, R.ref_w8a8_block_fp8_matmul(case.a, case.b, case.scale_a, case.scale_b, None, torch.bfloat16), what="block-scaled narrow stream, 8 rows")


def _random_shapes(count, seed):
    """Seeded shapes across the regimes of the automatic choice: rows log-uniform in 1 .. 700, weight rows multiples of 16
    up to 6000, K a multiple of 128 (three in four) or of 16; the CPU oracle's work is capped at 2 GFLOP per shape."""
    g = _g(seed)
    out = []
    while len(out) < count:
        M = int(round(math.exp(float(torch.rand(1, generator=g)) * math.log(700.0))))
        N = 16 * int(torch.randint(1, 376, (1,), generator=g))
        K = 128 * int(torch.randint(1, 72, (1,), generator=g)) if float(torch.rand(1, generator=g)) < 0.75 else 16 * int(torch.randint(8, 500, (1,), generator=g))
        if M * N * K <= 1_000_000_000:
            out.append((M, N, K))
    return out


@pytest.mark.parametrize("block_scaled", [False, True])
def test_automatic_schedules_on_random_shapes(device, block_scaled):
    """Whatever kernel, tile and split the library picks by itself (fixed rules to 16 rows, cost models above), the whole
    output matches the oracle: 70 seeded shapes per scaling, and every kind of kernel must have been met on the way."""
    seen = set()
    for M, N, K in _random_shapes(70, 2024 + block_scaled):
        g = _g(M * 31 + N * 7 + K)
        a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.5)
        if block_scaled:
            sa = torch.rand(M, -(-K // 128), generator=g) * 0.05 + 0.01
            sb = torch.rand(-(-N // 128), -(-K // 128), generator=g) * 0.05 + 0.01
            ref = R.ref_w8a8_block_fp8_matmul(a, b, sa, sb, [128, 128], torch.bfloat16)
            out = w8a8_block_fp8_matmul(a.to(device), b.to(device), sa.to(device), sb.to(device), [128, 128], torch.bfloat16)
        else:
            ref = R.ref_gemm_per_tensor(a, b, 0.03, 0.02, trans_b=True)
            out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=0.03, scale_b=0.02, out_dtype=torch.bfloat16)
        cfg = _lib.last_config()
        seen.add((cfg["KERNEL_NAME"], cfg["BLOCK_M"], cfg["BLOCK_N"], cfg["SPLIT_K"] > 1, cfg["ROW_GROUPS"], cfg["WAVES"]))
        assert cfg["KERNEL_NAME"] != "fallback", (M, N, K, cfg)   # (a K tail runs zero-padded through the workspace)
        check(out, ref, what=f"automatic schedule {cfg} for {M}x{N}x{K} block_scaled={block_scaled}")
    kernels = {k[0] for k in seen}
    assert {"tiled", "stream", "skinny"} <= kernels, seen
    assert len({k[1:3] for k in seen if k[0] == "tiled"}) >= (2 if block_scaled else 3) and any(k[3] for k in seen), seen


def test_kernel_choice_at_32_rows_follows_the_cost_model(device):
    """17 .. 64 rows: the cheapest of tile kernels, wide streaming form and skinny kernel by the fitted cost model.
    16384 x 1024 at M = 32 streams (256 workgroups, one 1 KiB piece each); 4096 x 14336 takes 64 x 128 tiles with eight
    splits (16.7 us against 18.1 for the streaming form with four); 6144 x 4096 takes tiles that split K inside the workgroup."""
    g = _g(41)
    a, b = fp8_randn((32, 1024), g), fp8_randn((16384, 1024), g, 0.02)
    out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=0.01, scale_b=0.02, out_dtype=torch.bfloat16)
    cfg = used("stream")
    assert cfg["ROW_GROUPS"] == 4 and cfg["SPLIT_K"] == 1, cfg
    check(out, R.ref_gemm_per_tensor(a, b, 0.01, 0.02, trans_b=True), what="16384 x 1024, M=32")
    a, b = fp8_randn((32, 14336), g), fp8_randn((4096, 14336), g, 0.02)
    out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=0.01, scale_b=0.02, out_dtype=torch.bfloat16)
    cfg = used("tiled")
    assert (cfg["BLOCK_M"], cfg["BLOCK_N"], cfg["SPLIT_K"]) == (64, 128, 8), cfg
    check(out, R.ref_gemm_per_tensor(a, b, 0.01, 0.02, trans_b=True), what="down projection, M=32")
    a, b = fp8_randn((32, 4096), g), fp8_randn((6144, 4096), g, 0.02)
    out = matmul(a.to(device), b.to(device), trans_b=True, scale_a=0.01, scale_b=0.02, out_dtype=torch.bfloat16)
    cfg = used("tiled")
    assert (cfg["BLOCK_M"], cfg["BLOCK_N"]) in ((32, 32), (64, 32)), cfg
    check(out, R.ref_gemm_per_tensor(a, b, 0.01, 0.02, trans_b=True), what="qkv projection, M=32")


def test_stream_wide_staggered_start_adds_the_same_products(device):
    """The two-piece form starts every workgroup at another K piece and wraps around; with integer-valued operands the
    sums are exact in fp32, so the rotated order must give the bits of the in-order form."""
    g = _g(77)
    M, N, K = 16, 1024, 8192
    a = torch.randint(-2, 3, (M, K), generator=g).float().to(torch.float8_e4m3fn)
    b = torch.randint(-2, 3, (N, K), generator=g).float().to(torch.float8_e4m3fn)
    outs = []
    for kc in ({"KERNEL": "stream", "ROW_GROUPS": 4}, {"KERNEL": "stream", "ROW_GROUPS": 4, "WAVES": 1}):
        outs.append(matmul(a.to(device), b.to(device), trans_b=True, out_dtype=torch.float32, kernel_configs=kc))
    assert torch.equal(outs[0], outs[1])
    assert torch.equal(outs[0].cpu(), a.float() @ b.float().t())


def test_decode_auto_schedule_and_determinism(device):
    case = W.llama_decode_case(16, "o")
    ref = R.ref_gemm_per_tensor(case.a, case.b, case.scale_a, case.scale_b, trans_b=True)
    d = case.to(device)
    outs = [matmul(d.a, d.b, trans_b=True, scale_a=d.scale_a, scale_b=d.scale_b, out_dtype=torch.bfloat16) for _ in range(4)]
    used("stream")
    check(outs[0], ref, what="decode o M=16")
    assert all(torch.equal(outs[0], o) for o in outs[1:])


# ----------------------------------------------------------------------------- layouts / fallbacks / dtypes
def test_all_four_layouts_agree_with_the_oracle(device):
    g = _g(21)
    M, N, K = 96, 136, 256
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g)
    at = a.view(torch.uint8).t().contiguous().view(FP8)
    bt = b.view(torch.uint8).t().contiguous().view(FP8)
    ref = R.ref_gemm_per_tensor(a, b, trans_b=True)
    for (x, y, ta, tb) in [(a, b, False, True), (a, bt, False, False), (at, bt, True, False), (at, b, True, True)]:
        out = matmul(x.to(device), y.to(device), trans_a=ta, trans_b=tb, out_dtype=torch.bfloat16)
        check(out, ref, what=f"layout ta={ta} tb={tb}")
    # (K,N) weights go through a K-contiguous copy in the workspace and then the MFMA kernels
    matmul(a.to(device), bt.to(device), out_dtype=torch.bfloat16)
    assert _lib.last_config()["KERNEL_NAME"] in ("tiled", "skinny")
    matmul(at.to(device), b.to(device), trans_a=True, trans_b=True, out_dtype=torch.bfloat16)
    used("fallback")


@pytest.mark.parametrize("trans_b", [True, False])
@pytest.mark.parametrize("M,N,K", [(32, 64, 1023), (130, 70, 200), (5, 33, 17), (300, 520, 1040), (200, 264, 4104), (16, 4096, 1000)])
def test_any_k_runs_on_the_mfma_kernels_through_zero_padded_copies(device, M, N, K, trans_b):
    """K = 1023 is the case the reference skips (tests/ops/test_matmul.py:130-131).  A K that is no multiple of 16, or no
    multiple of 128 above 64 rows, is padded with zeros into the workspace -- (K, N) weights transposed on the way -- and
    runs on the MFMA kernels; without a workspace the software-decode kernel takes it.  Same oracle either way."""
    g = _g(K)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g)
    ref = R.ref_gemm_per_tensor(a, b, 0.5, 2.0, trans_b=True)
    bd = b.to(device) if trans_b else b.view(torch.uint8).t().contiguous().view(FP8).to(device)
    out = matmul(a.to(device), bd, trans_b=trans_b, scale_a=0.5, scale_b=2.0, out_dtype=torch.bfloat16)
    assert _lib.last_config()["KERNEL_NAME"] in ("tiled", "stream", "skinny"), _lib.last_config()
    check(out, ref, what=f"padded K={K}")
    sa, sb = torch.tensor([0.5], device=device), torch.tensor([2.0], device=device)
    plain = torch.empty_like(out)
    _lib.fp8_gemm(plain, a.to(device), bd, sa, sb, False, trans_b, 1.0, 0.0, None, use_workspace=False)
    used("fallback")
    check(plain, ref, what=f"fallback K={K}")


def test_block_scaled_k_tail_above_64_rows_runs_padded(device):
    """Block-scaled, M = 200, K = 1000: the last K block holds 104 values; padded to 1024 the scales keep their shape."""
    M, N, K = 200, 392, 1000
    g = _g(1000)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.5)
    sa = torch.rand(M, 8, generator=g) * 0.05 + 0.01
    sb = torch.rand(4, 8, generator=g) * 0.05 + 0.01
    ref = R.ref_w8a8_block_fp8_matmul(a, b, sa, sb, [128, 128], torch.bfloat16)
    out = w8a8_block_fp8_matmul(a.to(device), b.to(device), sa.to(device), sb.to(device), [128, 128], torch.bfloat16)
    used("tiled")
    check(out, ref, what="block-scaled, K = 1000")


def test_k_tail_multiple_of_16_skinny(device):
    g = _g(33)
    M, N, K = 8, 256, 1040
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g)
    ref = R.ref_gemm_per_tensor(a, b, trans_b=True)
    out = matmul(a.to(device), b.to(device), trans_b=True, out_dtype=torch.bfloat16)
    used("stream")
    check(out, ref)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_output_dtypes(device, dtype):
    g = _g(4)
    a, b = fp8_randn((150, 256), g, 0.1), fp8_randn((264, 256), g, 0.1)
    for kernel in ("tiled", "fallback"):
        out = matmul(a.to(device), b.to(device), trans_b=True, out_dtype=dtype, kernel_configs={"KERNEL": kernel})
        assert out.dtype == dtype
        ref = R.ref_gemm_per_tensor(a, b, trans_b=True, out_dtype=dtype)
        check(out, ref, what=f"{kernel} {dtype}")
    out = matmul(a[:9].contiguous().to(device), b.to(device), trans_b=True, out_dtype=dtype)
    used("skinny")  # K = 256: too short for 1 KiB pieces
    check(out, R.ref_gemm_per_tensor(a[:9], b, trans_b=True, out_dtype=dtype))


def test_reference_default_returns_input_dtype(device):
    """Without keywords the op returns a.dtype like the reference (src/tilegym/ops/cutile/matmul.py:446);
    oracle as in tests/ops/test_matmul.py:231-236 (matmul then cast to fp8), tolerance 1 there."""
    g = _g(5)
    a = (torch.randn(128, 256, generator=g) * 0.3).to(FP8)
    b = (torch.randn(256, 192, generator=g) * 0.3).to(FP8)
    out = matmul(a.to(device), b.to(device))
    assert out.dtype == FP8 and out.shape == (128, 192)
    ref = R.ref_gemm_per_tensor(a, b, out_dtype=torch.float32).to(FP8)
    assert torch.allclose(out.float().cpu(), ref.float(), atol=1.0, rtol=1.0)
    ok, rep = R.compare_to_oracle(out.float(), ref.float(), 0.13, 0.02)  # one e4m3 ulp
    assert ok, rep


@pytest.mark.parametrize("kc", [None, {"KERNEL": "tiled", "BLOCK_M": 256, "BLOCK_N": 256}, {"KERNEL": "tiled", "BLOCK_M": 128, "BLOCK_N": 128, "SPLIT_K": 2},
                                {"KERNEL": "tiled", "BLOCK_M": 64, "BLOCK_N": 128}, {"KERNEL": "stream"}, {"KERNEL": "skinny"}, {"KERNEL": "fallback"}],
                         ids=lambda k: "auto" if k is None else "-".join(str(v) for v in k.values()))
def test_e4m3_output_is_cast_in_the_epilogue(device, kc):
    """c of dtype float8_e4m3fn through the C ABI: every kernel family rounds its fp32 result to e4m3 (nearest even)
    in its own epilogue and saturates at +-448 (the torch cast would give NaN from 465 up).  Integer-valued operands
    make the fp32 result exact, so the expected codes are known bit for bit, ragged N included (scalar store path)."""
    g = _g(77)
    M, N, K = 40, 202, 256
    a = torch.randint(-3, 4, (M, K), generator=g).float()
    b = torch.randint(-2, 3, (N, K), generator=g).float()
    exact = a @ b.t()
    for scale in (1.0, 16.0):  # 16: most results lie beyond +-448
        want = R.cast_output(exact * scale, FP8)  # the oracle's stated rule: saturating
        c = torch.empty(M, N, dtype=FP8, device=device)
        _lib.fp8_gemm(c, a.to(FP8).to(device), b.to(FP8).to(device), None, None, False, True, scale, 0.0, kernel_configs=kc)
        got = c.cpu()
        assert torch.equal(got.view(torch.uint8), want.view(torch.uint8)), f"scale {scale}: {(got.float() != want.float()).sum().item()} codes differ"
        if scale == 16.0:
            assert (want.float().abs() == 448).float().mean() > 0.3 and not torch.isnan(got.float()).any()


def test_power_of_two_scales_are_exact(device):
    g = _g(6)
    a, b = fp8_randn((64, 512), g), fp8_randn((256, 512), g)
    base = matmul(a.to(device), b.to(device), trans_b=True, out_dtype=torch.bfloat16)
    scaled = matmul(a.to(device), b.to(device), trans_b=True, scale_a=4.0, scale_b=torch.tensor([0.125], device=device), out_dtype=torch.bfloat16)
    assert torch.equal(scaled.float(), base.float() * 0.5)


# ----------------------------------------------------------------------------- alpha / beta
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (1.5, 2.0)])
@pytest.mark.parametrize("M,N,K,kernel", [(512, 512, 512, None), (16, 520, 256, None), (100, 72, 136, "fallback")])
def test_gemm_alpha_beta(device, alpha, beta, M, N, K, kernel):
    """Data recipe of tests/suites/flashinfer/test_flashinfer_gemm_alpha_beta.py:24-43 (rand in [0,1))."""
    g = _g(7)
    a = torch.rand(M, K, generator=g).to(torch.float16).to(FP8)
    b = torch.rand(N, K, generator=g).to(torch.float16).to(FP8)
    c0 = torch.rand(M, N, generator=g).to(torch.bfloat16)
    ref = R.ref_gemm_alpha_beta(a, b, c0.clone(), False, True, alpha, beta)
    c = c0.clone().to(device)
    kw = {"kernel_configs": {"KERNEL": kernel}} if kernel else {}
    out = tilegym_amd.backend._REGISTRY["flashinfer.gemm.gemm_alpha_beta"]["hip"](a.to(device), b.to(device), c, False, True, alpha, beta, **kw)
    assert out.data_ptr() == c.data_ptr()
    check(c, ref, what=f"alpha={alpha} beta={beta}")
    c2 = c0.clone().to(device)
    gemm_alpha_beta(a.to(device), b.to(device), c2, False, True, alpha, beta)
    if kernel is None:
        assert torch.equal(c2, c)


@pytest.mark.parametrize("m,n,k", [(1024, 1024, 1024), (1024, 1024, 1023), (8192, 8192, 8192), (8, 8, 8), (3072, 6144, 2720)])
def test_matmul_reference_test_shapes(device, m, n, k):
    """Shapes and layout (a (m,k), b (k,n), no transposes) of Test_Matmul.test_op (tests/ops/test_matmul.py:15-21),
    e4m3 operands drawn as there (N(0, 0.3), :64-66), per-tensor scales, bf16 out; K = 1023, 8 and 2720 take the
    paths for K % 128 != 0.  The oracle is evaluated on at most 128 sampled rows."""
    g = _g(m + k)
    a, b = fp8_randn((m, k), g, 0.3), fp8_randn((k, n), g, 0.3)
    sa, sb = torch.tensor(0.75), torch.tensor(1.5)
    out = matmul(a.to(device), b.to(device), scale_a=sa.to(device), scale_b=sb.to(device), out_dtype=torch.bfloat16)
    assert out.shape == (m, n) and out.dtype == torch.bfloat16
    rows = _rows_subset(m, 128)
    ref = R.ref_gemm_per_tensor(a[rows], b, sa, sb)
    check(out[rows.to(device)], ref, what=f"matmul {m}x{n}x{k}")
    assert torch.isfinite(out.float()).all()
    plain = matmul(a.to(device), b.to(device))              # the reference's own call: output typed like a
    assert plain.dtype == FP8 and plain.shape == (m, n)


@pytest.mark.parametrize("transpose_b", [True, False])
@pytest.mark.parametrize("group_k", [[1024, 512, 256, 128], [128, 128, 128, 128]])
@pytest.mark.parametrize("group_n", [[1024, 512, 256, 128], [128, 128, 128, 128]])
@pytest.mark.parametrize("group_m", [[1024, 512, 256, 128], [256, 256, 256, 256]])
def test_group_gemm_reference_test_shapes(device, group_m, group_n, group_k, transpose_b):
    """The group shapes of Test_GroupGemm.test_op (tests/ops/test_group_gemm.py:32-53), operands drawn as there
    (rand in [0,1), :81-88) and cast to e4m3, bf16 out."""
    g = _g(sum(group_m) + sum(group_n) + sum(group_k) + transpose_b)
    As = [torch.rand(M, K, generator=g).to(torch.float16).to(FP8) for M, K in zip(group_m, group_k)]
    Bs = [torch.rand((N, K) if transpose_b else (K, N), generator=g).to(torch.float16).to(FP8) for N, K in zip(group_n, group_k)]
    outs = group_gemm([x.to(device) for x in As], [x.to(device) for x in Bs], transpose_b=transpose_b, out_dtype=torch.bfloat16)
    refs = R.ref_group_gemm(As, Bs, transpose_b=transpose_b, out_dtype=torch.bfloat16)
    assert len(outs) == len(refs) == 4
    for i, (o, r) in enumerate(zip(outs, refs)):
        assert o.shape == (group_m[i], group_n[i])
        check(o, r, what=f"group {i}")


@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (1.5, 2.0)])
@pytest.mark.parametrize("size", [4096, 8192])
def test_gemm_alpha_beta_reference_test_sizes(device, size, alpha, beta):
    """m = n = k = 4096 and 8192 as in tests/suites/flashinfer/test_flashinfer_gemm_alpha_beta.py:45-55 (fp8 in,
    bf16 out); the oracle is evaluated on 128 sampled rows (a row of the output depends on its own rows of a and c)."""
    g = _g(size)
    a = torch.rand(size, size, generator=g).to(torch.float16).to(FP8)
    b = torch.rand(size, size, generator=g).to(torch.float16).to(FP8)
    c0 = torch.rand(size, size, generator=g).to(torch.bfloat16)
    c = c0.clone().to(device)
    out = gemm_alpha_beta(a.to(device), b.to(device), c, False, True, alpha, beta)
    assert out.data_ptr() == c.data_ptr()
    rows = torch.randperm(size, generator=g)[:128].sort().values
    rows[0], rows[-1] = 0, size - 1
    ref = R.ref_gemm_alpha_beta(a[rows], b, c0[rows].clone(), False, True, alpha, beta)
    check(c[rows.to(device)], ref, what=f"{size}^3 alpha={alpha} beta={beta}")
    assert torch.isfinite(c.float()).all()


# ----------------------------------------------------------------------------- block scaled
@pytest.mark.parametrize("M,N,K", [(128, 128, 128), (256, 256, 256), (512, 1024, 512), (1024, 2048, 1024)])
def test_block_scaled_reference_test_shapes(device, M, N, K):
    """Shapes, data recipe and tolerance of Test_Unsloth_W8A8_FP8_Matmul (tests/suites/unsloth/test_fp8.py:193-231)."""
    g = _g(42)
    A = (torch.randn(M, K, generator=g) * 0.1).to(FP8)
    B = (torch.randn(N, K, generator=g) * 0.1).to(FP8)
    As = torch.rand(M, K // 128, generator=g) + 0.1
    Bs = torch.rand(N // 128, K // 128, generator=g) + 0.1
    ref = R.ref_w8a8_block_fp8_matmul(A, B, As, Bs, [128, 128])
    out = w8a8_block_fp8_matmul(A.to(device), B.to(device), As.to(device), Bs.to(device), [128, 128])
    used("tiled")
    assert out.dtype == torch.float32
    assert torch.allclose(out.cpu(), ref, rtol=5e-2, atol=5e-2)
    check(out, ref, tight=1e-4, what="block-scaled f32")


@pytest.mark.parametrize("bm,bn", [(256, 256), (128, 128), (128, 256), (64, 128)])
@pytest.mark.parametrize("M,N,K", [(300, 640, 384), (129, 136, 256)])
def test_block_scaled_tiled_configs_and_edges(device, bm, bn, M, N, K):
    case = W.block_scaled_case(M, N, K, seed=M)
    ref = R.ref_w8a8_block_fp8_matmul(case.a, case.b, case.scale_a, case.scale_b, output_dtype=torch.bfloat16)
    d = case.to(device)
    out = tilegym_amd.backend._REGISTRY["unsloth.w8a8_block_fp8_matmul"]["hip"](
        d.a, d.b, d.scale_a, d.scale_b, None, torch.bfloat16, kernel_configs={"KERNEL": "tiled", "BLOCK_M": bm, "BLOCK_N": bn})
    cfg = used("tiled")
    assert (cfg["BLOCK_M"], cfg["BLOCK_N"]) == (bm, bn)
    check(out, ref, what=f"block-scaled {bm}x{bn}")


@pytest.mark.parametrize("M,N,K", [(256, 256, 256), (300, 520, 1280), (1000, 1000, 384), (2048, 1024, 1408), (768, 256, 768),
                                   (520, 300, 896), (700, 512, 1024), (256, 512, 5120), (512, 768, 512)])
def test_block_scaled_persistent_256(device, M, N, K):
    """The persistent form of the block-scaled 256x256 tile (ROW_GROUPS = 1): three weight slabs, scales in registers in
    chunks of four K steps.  K steps that are a multiple of four and not (the last chunk holds 2 or 3 steps), a single
    chunk, ten chunks; ragged M and N; bf16 and f32 outputs.  Against the oracle, and bit for bit against the kernel of
    one workgroup per tile (WAVES = 8)."""
    case = W.block_scaled_case(M, N, K, seed=M + N + K)
    d = case.to(device)
    kc = {"KERNEL": "tiled", "BLOCK_M": 256, "BLOCK_N": 256, "SPLIT_K": 1, "ROW_GROUPS": 1}
    for dtype in (torch.bfloat16, torch.float32):
        ref = R.ref_w8a8_block_fp8_matmul(case.a, case.b, case.scale_a, case.scale_b, None, dtype)
        out = w8a8_block_fp8_matmul(d.a, d.b, d.scale_a, d.scale_b, None, dtype, kernel_configs=kc)
        cfg = used("tiled")
        assert (cfg["BLOCK_M"], cfg["BLOCK_N"], cfg["ROW_GROUPS"]) == (256, 256, 1), cfg
        check(out, ref, what=f"persistent block-scaled M={M} N={N} K={K} {dtype}")
        other = w8a8_block_fp8_matmul(d.a, d.b, d.scale_a, d.scale_b, None, dtype, kernel_configs=dict(kc, ROW_GROUPS=-1, WAVES=8))
        assert _lib.last_config()["ROW_GROUPS"] != 1
        assert torch.equal(out, other), "persistent and one-workgroup-per-tile block-scaled kernels differ"


def test_block_scaled_persistent_256_refuses_a_single_step_last_chunk(device):
    """K % 512 == 128 (a last chunk of scales of one step) stays with the kernel of one workgroup per tile, also when the
    persistent form is asked for."""
    case = W.block_scaled_case(300, 256, 640, seed=9)
    d = case.to(device)
    out = w8a8_block_fp8_matmul(d.a, d.b, d.scale_a, d.scale_b, None, torch.bfloat16,
                                kernel_configs={"KERNEL": "tiled", "BLOCK_M": 256, "BLOCK_N": 256, "ROW_GROUPS": 1})
    assert used("tiled")["ROW_GROUPS"] != 1
    check(out, R.ref_w8a8_block_fp8_matmul(case.a, case.b, case.scale_a, case.scale_b, None, torch.bfloat16))


def test_block_scaled_persistent_256_walks_several_tiles_per_workgroup(device):
    """More tiles than compute units: workgroups compute two tiles, the operand rings and the scale chunks run on from one
    tile into the next (K = 768: the first tile's last chunk is partial); a partial row tile and a partial column tile."""
    M, N, K = 4300, 4360, 768
    assert math.ceil(M / 256) * math.ceil(N / 256) > torch.cuda.get_device_properties(device).multi_processor_count
    case = W.block_scaled_case(M, N, K, seed=4)
    d = case.to(device)
    kc = {"KERNEL": "tiled", "BLOCK_M": 256, "BLOCK_N": 256, "SPLIT_K": 1, "ROW_GROUPS": 1}
    out = w8a8_block_fp8_matmul(d.a, d.b, d.scale_a, d.scale_b, None, torch.bfloat16, kernel_configs=kc)
    assert used("tiled")["ROW_GROUPS"] == 1
    other = w8a8_block_fp8_matmul(d.a, d.b, d.scale_a, d.scale_b, None, torch.bfloat16, kernel_configs=dict(kc, ROW_GROUPS=-1, WAVES=8))
    assert torch.equal(out, other)
    rows = torch.cat([torch.arange(0, 3), torch.arange(254, 259), torch.randint(0, M, (24,), generator=_g(1)), torch.arange(M - 3, M)])
    ref = R.ref_w8a8_block_fp8_matmul(case.a[rows], case.b, case.scale_a[rows], case.scale_b, None, torch.bfloat16)
    check(out[rows.to(device)], ref, what="persistent block-scaled, several tiles per workgroup")


@pytest.mark.parametrize("N,K", [(392, 256), (512, 768), (300, 1408), (256, 2048)])
def test_ragged_persistent_256(device, N, K):
    """The persistent block-scaled kernel over ragged expert segments (ROW_GROUPS = 1; the default for K <= 1536): empty,
    tiny, unaligned and multi-tile experts, rows of no segment untouched; against the oracle and bit for bit against the
    kernel of one workgroup per tile; more than 64 experts."""
    sizes = [5, 0, 131, 64, 0, 0, 600, 1, 77, 256, 300]
    a, b, a_s, b_s, ptr = _ragged_inputs(sizes, N, K, 17 + K, total_extra=6)
    ref = R.ref_ragged_block_scaled_bmm(a, b, a_s, b_s, ptr)
    impl = tilegym_amd.backend._REGISTRY["flashinfer.gemm.ragged_block_scaled_bmm"]["hip"]
    kc = {"BLOCK_M": 256, "BLOCK_N": 256, "ROW_GROUPS": 1}
    out = impl(a.to(device), b.to(device), a_s.to(device), b_s.to(device), ptr.to(device), max(sizes), kernel_configs=kc, zero_init=True)
    cfg = used("tiled")
    assert (cfg["BLOCK_M"], cfg["BLOCK_N"], cfg["ROW_GROUPS"]) == (256, 256, 1), cfg
    check(out, ref, what=f"ragged persistent N={N} K={K}")
    assert torch.equal(out[sum(sizes):].cpu().float(), torch.zeros(6, N))
    other = impl(a.to(device), b.to(device), a_s.to(device), b_s.to(device), ptr.to(device), max(sizes),
                 kernel_configs={"BLOCK_M": 256, "BLOCK_N": 256, "WAVES": 8}, zero_init=True)
    assert _lib.last_config()["ROW_GROUPS"] != 1
    assert torch.equal(out, other), "persistent and one-workgroup-per-tile ragged kernels differ"
    sizes2 = torch.randint(0, 40, (150,), generator=_g(K)).tolist()
    a, b, a_s, b_s, ptr = _ragged_inputs(sizes2, 256, K, 5)
    out = impl(a.to(device), b.to(device), a_s.to(device), b_s.to(device), ptr.to(device), max(sizes2), kernel_configs=kc)
    check(out, R.ref_ragged_block_scaled_bmm(a, b, a_s, b_s, ptr), what="ragged persistent, 150 experts")


def test_ragged_persistent_256_is_the_default_for_short_k(device):
    a, b, a_s, b_s, ptr = _ragged_inputs([300] * 8, 512, 1408, 3)
    dev = [t.to(device) for t in (a, b, a_s, b_s, ptr)]
    ragged_block_scaled_bmm(*dev, 300)
    cfg = used("tiled")
    assert (cfg["BLOCK_M"], cfg["BLOCK_N"], cfg["ROW_GROUPS"]) == (256, 256, 1), cfg
    a, b, a_s, b_s, ptr = _ragged_inputs([300] * 8, 512, 2048, 3)
    ragged_block_scaled_bmm(*[t.to(device) for t in (a, b, a_s, b_s, ptr)], 300)
    assert used("tiled")["ROW_GROUPS"] != 1


@pytest.mark.parametrize("M", [1, 16, 40, 64])
@pytest.mark.parametrize("split", [1, 4])
@pytest.mark.parametrize("kernel,K", [("skinny", 1024), ("stream", 1024), ("stream", 4224)])
def test_block_scaled_skinny(device, M, split, kernel, K):
    case = W.block_scaled_case(M, 640, K, seed=M)
    ref = R.ref_w8a8_block_fp8_matmul(case.a, case.b, case.scale_a, case.scale_b, output_dtype=torch.bfloat16)
    d = case.to(device)
    out = tilegym_amd.backend._REGISTRY["unsloth.w8a8_block_fp8_matmul"]["hip"](
        d.a, d.b, d.scale_a, d.scale_b, None, torch.bfloat16, kernel_configs={"KERNEL": kernel, "SPLIT_K": split})
    used(kernel)
    check(out, ref, what=f"block-scaled {kernel} M={M} K={K}")


def test_block_scaled_batched_leading_dims_and_invariants(device):
    g = _g(9)
    A = fp8_randn((2, 3, 256), g)
    B = fp8_randn((128, 256), g)
    As = torch.rand(2, 3, 2, generator=g) + 0.5
    Bs = torch.rand(1, 2, generator=g) + 0.5
    out = w8a8_block_fp8_matmul(A.to(device), B.to(device), As.to(device), Bs.to(device), None, torch.bfloat16)
    assert out.shape == (2, 3, 128)
    check(out, R.ref_w8a8_block_fp8_matmul(A, B, As, Bs, None, torch.bfloat16))
    # all-equal block scales == per-tensor scales (bit-exact)
    A2, B2 = fp8_randn((200, 512), g), fp8_randn((256, 512), g)
    blk = w8a8_block_fp8_matmul(A2.to(device), B2.to(device), torch.full((200, 4), 0.25, device=device),
                                torch.full((2, 4), 2.0, device=device), None, torch.float32)
    pt = matmul(A2.to(device), B2.to(device), trans_b=True, scale_a=0.25, scale_b=2.0, out_dtype=torch.float32,
                kernel_configs={"KERNEL": "tiled", "BLOCK_M": 128, "BLOCK_N": 128})
    check(blk, pt.cpu(), tight=1e-5)
    # doubling every activation scale doubles the result exactly
    case = W.block_scaled_case(130, 256, 512, seed=3).to(device)
    o1 = w8a8_block_fp8_matmul(case.a, case.b, case.scale_a, case.scale_b, None, torch.bfloat16)
    o2 = w8a8_block_fp8_matmul(case.a, case.b, case.scale_a * 2, case.scale_b, None, torch.bfloat16)
    assert torch.equal(o2.float(), o1.float() * 2)


# ----------------------------------------------------------------------------- grouped (ragged)
def _ragged_inputs(sizes, N, K, seed, total_extra=0):
    g = _g(seed)
    Q = len(sizes)
    total = sum(sizes) + total_extra
    ptr = torch.zeros(Q + 1, dtype=torch.int32)
    ptr[1:] = torch.cumsum(torch.tensor(sizes), 0)
    a = fp8_randn((total, K), g)
    b = fp8_randn((Q, N, K), g, 0.5)
    a_s = torch.rand(total, K // 128, generator=g) * 1e-2 + 1e-3
    b_s = torch.rand(Q, -(-N // 128), K // 128, generator=g) * 1e-2 + 1e-3
    return a, b, a_s, b_s, ptr


@pytest.mark.parametrize("groups,m", [(4, 128), (16, 128), (4, 512), (16, 512)])
@pytest.mark.parametrize("n,k", [(2048, 2048), (4096, 4096)])
def test_ragged_reference_test_shapes(device, groups, m, n, k):
    """Group counts / segment sizes of Test_FlashInfer_RaggedBlockScaledBMM
    (tests/suites/flashinfer/test_flashinfer_ragged_block_scaled_bmm.py:216-223); that test allows atol=rtol=1."""
    a, b, a_s, b_s, ptr = _ragged_inputs([m] * groups, n, k, groups + m)
    ref = R.ref_ragged_block_scaled_bmm(a, b, a_s, b_s, ptr)
    out = ragged_block_scaled_bmm(a.to(device), b.to(device), a_s.to(device), b_s.to(device), ptr.to(device), m)
    used("tiled")
    assert out.dtype == torch.bfloat16
    assert torch.allclose(out.float().cpu(), ref.float(), atol=1.0, rtol=1.0)
    check(out, ref, what="ragged aligned")


@pytest.mark.parametrize("bm,bn", [(256, 256), (128, 128), (128, 256), (64, 128)])
def test_ragged_unaligned_empty_and_single_experts(device, bm, bn):
    sizes = [5, 0, 131, 64, 0, 0, 257, 1, 77]
    a, b, a_s, b_s, ptr = _ragged_inputs(sizes, 392, 256, 17, total_extra=6)
    ref = R.ref_ragged_block_scaled_bmm(a, b, a_s, b_s, ptr)
    impl = tilegym_amd.backend._REGISTRY["flashinfer.gemm.ragged_block_scaled_bmm"]["hip"]
    out = impl(a.to(device), b.to(device), a_s.to(device), b_s.to(device), ptr.to(device), max(sizes),
               kernel_configs={"BLOCK_M": bm, "BLOCK_N": bn}, zero_init=True)
    cfg = used("tiled")
    assert (cfg["BLOCK_M"], cfg["BLOCK_N"]) == (bm, bn)
    check(out, ref, what=f"ragged unaligned {bm}x{bn}")
    assert torch.equal(out[sum(sizes):].cpu().float(), torch.zeros(6, 392))  # rows of no segment untouched
    # single expert == dense
    a1, b1, as1, bs1, p1 = _ragged_inputs([150], 256, 384, 3)
    o1 = impl(a1.to(device), b1.to(device), as1.to(device), bs1.to(device), p1.to(device), 150, kernel_configs={"BLOCK_M": bm, "BLOCK_N": bn})
    dense = w8a8_block_fp8_matmul(a1.to(device), b1[0].to(device), as1.to(device), bs1[0].to(device), None, torch.bfloat16)
    check(o1, dense.cpu(), tight=1e-5)
    # no activation scales
    o2 = impl(a.to(device), b.to(device), None, b_s.to(device), ptr.to(device), max(sizes), zero_init=True)
    check(o2, R.ref_ragged_block_scaled_bmm(a, b, None, b_s, ptr))


@pytest.mark.parametrize("K", [128, 256, 384, 1024, 1152, 2176])
def test_ragged_tiles_of_two_workgroups_per_compute_unit(device, K):
    """128 x 256 tiles: a ring of half weight slabs (1, 2, 3 K steps), chunks of scales that end inside K (8, 9, 17 steps), no
    row, one row, whole and partly filled row groups per expert.  Same bits as 128 x 128 tiles."""
    impl = tilegym_amd.backend._REGISTRY["flashinfer.gemm.ragged_block_scaled_bmm"]["hip"]
    sizes = [0, 1, 128, 129, 77, 300, 0, 16]
    a, b, a_s, b_s, ptr = _ragged_inputs(sizes, 392, K, K)
    args = [t.to(device) for t in (a, b, a_s, b_s, ptr)] + [max(sizes)]
    out = impl(*args, kernel_configs={"BLOCK_M": 128, "BLOCK_N": 256})
    cfg = used("tiled")
    assert (cfg["BLOCK_M"], cfg["BLOCK_N"]) == (128, 256)
    assert torch.equal(out, impl(*args, kernel_configs={"BLOCK_M": 128, "BLOCK_N": 128}))
    check(out, R.ref_ragged_block_scaled_bmm(a, b, a_s, b_s, ptr), what=f"pair tiles, K={K}")


@pytest.mark.parametrize("crowded", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_moe_layer_same_bits_with_128_and_256_row_blocks(device, dtype, crowded):
    """Enough 128 x 256 tiles for the form of which two share a compute unit, in both GEMMs; even routing, and every token to
    the same four experts."""
    T, H, I, E, k = 600, 1024, 512, 64, 4
    g = torch.Generator(device=device).manual_seed(7 + crowded)
    x = torch.randn(T, H, generator=g, device=device).to(dtype)
    w1, w2 = (torch.randn(E, n, kk, generator=g, device=device).to(FP8) for n, kk in ((2 * I, H), (H, I)))
    s1, s2 = (torch.rand(E, n // 128, kk // 128, generator=g, device=device) * 0.02 + 0.001 for n, kk in ((2 * I, H), (H, I)))
    ids = torch.rand(T, E, generator=g, device=device).topk(k, dim=1).indices.to(torch.int32)
    if crowded:
        ids = torch.tensor([3, 9, 41, 63], dtype=torch.int32, device=device).expand(T, k).contiguous()
    weights = torch.rand(T, k, generator=g, device=device)
    outs = []
    for block_m in (128, 256):
        out = torch.empty(T, H, dtype=dtype, device=device)
        _lib.fp8_fused_moe(out, x, w1, w2, s1, s2, weights, ids, block_m)
        outs.append(out)
    assert torch.isfinite(outs[0]).all()
    assert torch.equal(*outs)


@pytest.mark.parametrize("dtype,bits", [(torch.bfloat16, 7), (torch.float16, 10)])
@pytest.mark.parametrize("rule,eps", [(0, 0.0), (1, 1e-10), (1, 0.3)])
def test_quantizer_divides_as_ieee_division_does(device, dtype, bits, rule, eps):
    """Significands of a group's maximum (all of bf16's 128, 128 spread over f16's 1024) against 127 significands of its elements,
    at every distance in binades that leaves a code; eps above some maxima, below others.  The codes of the IEEE quotient."""
    n = 1 << bits
    amax = 1.0 + (torch.arange(128) * (n // 128) + (n // 256 if bits > 7 else 0)).float() / n
    frac = 1.0 + (torch.arange(127) * (n // 128) + 1).float() / n
    x = torch.stack([torch.cat([amax[:, None], torch.minimum(frac[None] * 2.0 ** -d, amax[:, None])], dim=1) for d in range(14)])  # (14, 128, 128)
    x = (x * torch.where(torch.arange(128) % 2 == 1, -1.0, 1.0) * (0.25 if eps > 0.1 else 1.0)).reshape(14, 128 * 128).to(dtype)
    q, scales = _lib.fp8_quant_group(x.to(device), 128, eps, rule)
    f = x.float().reshape(14, 128, 128)
    s = f.abs().amax(dim=-1).clamp(min=eps) / 448.0
    want = (f / s[..., None]).clamp(-448.0, 448.0).to(FP8).reshape(14, -1)
    assert torch.equal(scales.cpu(), s)
    assert torch.equal(q.cpu().view(torch.uint8), want.view(torch.uint8))


def test_ragged_many_experts_and_permutation(device):
    g = _g(31)
    sizes = torch.randint(0, 40, (150,), generator=g).tolist()  # > 64 experts: multi-pass expert search
    a, b, a_s, b_s, ptr = _ragged_inputs(sizes, 128, 128, 5)
    ref = R.ref_ragged_block_scaled_bmm(a, b, a_s, b_s, ptr)
    out = ragged_block_scaled_bmm(a.to(device), b.to(device), a_s.to(device), b_s.to(device), ptr.to(device), max(sizes))
    check(out, ref, what="150 experts")
    again = ragged_block_scaled_bmm(a.to(device), b.to(device), a_s.to(device), b_s.to(device), ptr.to(device), max(sizes))
    assert torch.equal(out, again)


def test_ragged_fallback_for_odd_k(device):
    g = _g(8)
    sizes = [3, 0, 9]
    Q, N, K = 3, 40, 200
    ptr = torch.tensor([0, 3, 3, 12], dtype=torch.int32)
    a, b = fp8_randn((12, K), g), fp8_randn((Q, N, K), g)
    a_s = torch.rand(12, 2, generator=g) + 0.1
    b_s = torch.rand(Q, 1, 2, generator=g) + 0.1
    ref = R.ref_ragged_block_scaled_bmm(a, b, a_s, b_s, ptr)
    L = _lib
    c = torch.empty(12, N, dtype=torch.bfloat16, device=device)
    L.fp8_ragged_gemm(c, a.to(device), b.to(device), a_s.to(device), b_s.to(device), ptr.to(device))
    used("fallback")
    check(c, ref)


@pytest.mark.parametrize("bm,bn,K", [(32, 128, 1024), (64, 128, 1152), (64, 256, 640), (64, 256, 1152), (128, 256, 640), (128, 256, 2176), (64, 192, 640), (128, 192, 1152)])
@pytest.mark.parametrize("many", [False, True])
def test_ragged_ring_tiles(device, bm, bn, K, many):
    """The persistent tiles: the fewest K steps they take (5, 8), chunks of scales that end inside K or hold one step (9, 17), experts
    without rows, with one, with more than a tile; fewer tiles than workgroups and several tiles on each; every output type, columns
    that end inside a tile and odd ones.  Same bits as 128 x 128 tiles."""
    g = _g(K + bm)
    if many:   # 130 experts (the search for a tile's expert crosses 64), about nine hundred tiles of 128 columns
        sizes, N = torch.randint(0, 2 * bm // 3, (130,), generator=g).tolist(), 904
        sizes[64], sizes[129] = 0, bm + 1
    else:
        sizes, N = [0, 1, 128, 129, 77, 300, 0, 16], 392
    a, b, a_s, b_s, ptr = _ragged_inputs(sizes, N, K, K, total_extra=3)
    dev = [t.to(device) for t in (a, b, a_s, b_s, ptr)]
    for dtype in (torch.bfloat16, torch.float32, torch.float16, FP8):
        out, base = (torch.zeros(a.shape[0], N, device=device).to(dtype) for _ in range(2))
        _lib.fp8_ragged_gemm(out, *dev, {"KERNEL": "tiled", "BLOCK_M": bm, "BLOCK_N": bn, "ROW_GROUPS": 1})
        cfg = used("tiled")
        assert (cfg["BLOCK_M"], cfg["BLOCK_N"], cfg["ROW_GROUPS"]) == (bm, bn, 1), cfg
        _lib.fp8_ragged_gemm(base, *dev, {"KERNEL": "tiled", "BLOCK_M": 128, "BLOCK_N": 128})
        assert _lib.last_config()["ROW_GROUPS"] != 1
        assert torch.equal(out.view(torch.uint8), base.view(torch.uint8)), dtype
    if not many:
        res = torch.zeros(a.shape[0], N, dtype=torch.bfloat16, device=device)
        _lib.fp8_ragged_gemm(res, *dev, {"KERNEL": "tiled", "BLOCK_M": bm, "BLOCK_N": bn, "ROW_GROUPS": 1})
        check(res[: sum(sizes)], R.ref_ragged_block_scaled_bmm(a, b, a_s, b_s, ptr)[: sum(sizes)], what=f"ragged ring {bm}x{bn} K={K}")
    odd = torch.zeros(a.shape[0], N - 5, dtype=torch.bfloat16, device=device)
    want = torch.zeros_like(odd)
    bo, so = b[:, : N - 5].contiguous().to(device), dev[3]
    _lib.fp8_ragged_gemm(odd, dev[0], bo, dev[2], so, dev[4], {"KERNEL": "tiled", "BLOCK_M": bm, "BLOCK_N": bn, "ROW_GROUPS": 1})
    _lib.fp8_ragged_gemm(want, dev[0], bo, dev[2], so, dev[4], {"KERNEL": "tiled", "BLOCK_M": 128, "BLOCK_N": 128})
    assert torch.equal(odd, want)


@pytest.mark.parametrize("rows,want", [(40, None), (400, None), (401, (32, 128)), (1500, (64, 128)), (2000, (128, 128))])  # None: streaming
def test_ragged_ring_tiles_are_the_default_for_few_rows_per_expert(device, rows, want):
    g = _g(rows)
    E, N, K = 40, 512, 2048
    sizes = torch.bincount(torch.randint(0, E, (rows,), generator=g), minlength=E).tolist()
    a, b, a_s, b_s, ptr = _ragged_inputs(sizes, N, K, rows)
    out = ragged_block_scaled_bmm(a.to(device), b.to(device), a_s.to(device), b_s.to(device), ptr.to(device), max(sizes))
    cfg = used("tiled" if want else "stream")
    if want:
        assert (cfg["BLOCK_M"], cfg["BLOCK_N"]) == want and (cfg["ROW_GROUPS"] == 1) == (rows <= 40 * E), cfg
    check(out, R.ref_ragged_block_scaled_bmm(a, b, a_s, b_s, ptr), what=f"{rows} rows")


@pytest.mark.parametrize("routing", ["even", "one expert", "a third on two experts", "two thirds of the experts"])
def test_ragged_ring_tiles_take_their_columns_from_the_routing(device, routing):
    """32 row tiles over 1536 columns: 192 columns are one round of 256 workgroups; a row tile more and 256 columns are, a third of the experts
    without rows and 128 are.  Crowded experts walk several row tiles over the same columns.  Same bits as 128 x 128 tiles."""
    E, N, K, rows = 32, 1536, 2048, 640
    gen = torch.Generator(device=device).manual_seed(7)
    ids = torch.arange(rows, device=device) % E
    if routing.startswith("one"):
        ids[:] = 5
    elif routing.startswith("a third"):
        ids[::6], ids[1::6] = 0, E - 1
    elif routing.startswith("two"):
        ids %= 2 * E // 3
    ptr = torch.zeros(E + 1, dtype=torch.int32, device=device)
    ptr[1:] = torch.cumsum(torch.bincount(ids, minlength=E), 0)
    a, b = (torch.randint(0, 0x70, s, generator=gen, dtype=torch.uint8, device=device).view(FP8) for s in ((rows, K), (E, N, K)))
    sa, sb = (torch.rand(*s, generator=gen, device=device) for s in ((rows, K // 128), (E, N // 128, K // 128)))
    out = ragged_block_scaled_bmm(a, b, sa, sb, ptr, rows)
    cfg = used("tiled")
    assert (cfg["BLOCK_M"], cfg["BLOCK_N"], cfg["ROW_GROUPS"]) == (64, 256, 1), cfg
    want = torch.empty_like(out)
    _lib.fp8_ragged_gemm(want, a, b, sa, sb, ptr, {"KERNEL": "tiled", "BLOCK_M": 128, "BLOCK_N": 128})
    assert torch.equal(out, want)


# ----------------------------------------------------------------------------- MoE token gather
@pytest.mark.parametrize("block_m,K", [(64, 640), (64, 1152), (128, 640), (128, 1152)])
def test_moe_gather_on_ring_tiles(device, block_m, K):
    """The persistent tiles of the gather form and of the form with the activation epilogue: several tiles on a workgroup, slots masked out
    in the middle of an expert's rows, ids beyond the output's rows, an expert without tokens, routed weights.  Same bits as the kernels of one workgroup
    per tile and as the two steps."""
    g = _g(block_m + K)
    T, E, N, top_k = 300, 40, 1792, 3
    A, B = fp8_randn((T, K), g).to(device), fp8_randn((E, N, K), g, 0.5).to(device)
    a_s, b_s = (torch.rand(T, K // 128, generator=g) * 0.05 + 0.01).to(device), (torch.rand(E, N // 128, K // 128, generator=g) + 0.1).to(device)
    w, ids = W.moe_routing(T, E, top_k, seed=11)
    ids[ids == 3] = 4
    sorted_ids, expert_ids, post, _, _ = moe_align_block_size(ids.to(device), block_m, E)
    sorted_ids = sorted_ids.clone()
    hole = torch.rand(sorted_ids.numel(), generator=g) < 0.2
    hole[:40] = True
    sorted_ids[hole.to(device)] = T * top_k
    num_valid = T * top_k - 37
    wd = w.to(device)
    for dtype in (torch.bfloat16, torch.float32):
        got, want = (torch.zeros(num_valid, N, dtype=dtype, device=device) for _ in range(2))
        for mul in (True, False):
            _lib.fp8_moe_gemm(got, A, B, a_s, b_s, wd, sorted_ids, expert_ids, post, mul, top_k, block_m)
            cfg = used("tiled")
            assert cfg["ROW_GROUPS"] == 1 and cfg["BLOCK_M"] == block_m, cfg
            _lib.fp8_moe_gemm(want, A, B, a_s, b_s, wd, sorted_ids, expert_ids, post, mul, top_k, block_m, {"BLOCK_M": 64, "BLOCK_N": 128})
            assert _lib.last_config()["ROW_GROUPS"] != 1
            assert torch.equal(got, want)
    if block_m == 128:
        c = want.to(torch.bfloat16)
        _lib.fp8_moe_gemm(c, A, B, a_s, b_s, wd, sorted_ids, expert_ids, post, False, top_k, block_m, {"BLOCK_M": 64, "BLOCK_N": 128})
        q2, s2 = _lib.silu_mul_quant_1x128(c)
        q, s = _lib.fp8_moe_gemm_silu_quant(A, B, a_s, b_s, sorted_ids, expert_ids, post, top_k, block_m, num_valid, torch.bfloat16)
        assert _lib.last_config()["ROW_GROUPS"] == 1
        live = sorted_ids[(sorted_ids >= 0) & (sorted_ids < num_valid)].long()
        assert torch.equal(q.view(torch.uint8)[live], q2.view(torch.uint8)[live]) and torch.equal(s[live], s2[live])


@pytest.mark.parametrize("T,H,I,E,k", [(200, 1024, 1024, 16, 2), (150, 1152, 640, 40, 4), (300, 640, 1024, 24, 3), (90, 1024, 512, 8, 4), (75, 1024, 512, 8, 4)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_moe_layer_on_64_row_blocks(device, T, H, I, E, k, dtype, monkeypatch):
    """Up to 40 rows per expert (47 over 256 MB) the one-call layer pads experts to 64 rows and runs on the ring tiles (GEMM2 on 64 x 128 tiles where its K
    is too short for them); ids outside [0, E) included.  Same bits as the call-by-call layer on 128-row blocks."""
    from tilegym_amd.ops import fused_moe, moe_interface

    g = _g(T + H + I)
    x = torch.randn(T, H, generator=g).to(dtype).to(device)
    w1, w2 = fp8_randn((E, 2 * I, H), g, 0.5).to(device), fp8_randn((E, H, I), g, 0.5).to(device)
    s1, s2 = (torch.rand(E, 2 * I // 128, H // 128, generator=g) * 0.02).to(device), (torch.rand(E, H // 128, I // 128, generator=g) * 0.02).to(device)
    tw, ids = W.moe_routing(T, E, k, seed=5)
    ids[5, 0], ids[7, k - 1] = -1, E
    args = (x, w1, w2, tw.to(device), ids.to(device))
    got = fused_moe(*args, w1_scale=s1, w2_scale=s2)
    cfg = _lib.last_config()  # (of the second GEMM, over the same blocks as the first, which runs on 64-row blocks on ring tiles only)
    assert (cfg["BLOCK_M"] == 64) == (T * k <= 40 * E), cfg  # (more rows only over 256 MB)
    assert cfg["BLOCK_M"] != 64 or (cfg["ROW_GROUPS"] == 1) == (I >= 640), cfg
    assert T * k > E * 7   # (past the decoding form)
    monkeypatch.setattr(_lib, "native", None)
    monkeypatch.setattr(moe_interface, "USE_ONE_CALL_LAYER", False)
    assert torch.equal(got, fused_moe(*args, w1_scale=s1, w2_scale=s2))


@pytest.mark.parametrize("block_m", [64, 128, 16, 256])
@pytest.mark.parametrize("mul_w", [False, True])
def test_moe_gather_gemm(device, block_m, mul_w):
    g = _g(block_m)
    T, E, N, K, top_k = 70, 8, 264, 256, 2
    A = fp8_randn((T, K), g)
    B = fp8_randn((E, N, K), g, 0.5)
    a_s = torch.rand(T, K // 128, generator=g) + 0.1
    b_s = torch.rand(E, -(-N // 128), K // 128, generator=g) + 0.1
    w, ids = W.moe_routing(T, E, top_k, seed=1)
    ids[ids == 3] = 2  # an expert without tokens
    ref = R.ref_fused_moe_gemm(A, B, a_s, b_s, w, ids, mul_w, top_k)
    sorted_ids, expert_ids, post, _, _ = moe_align_block_size(ids.to(device), block_m, E)
    rs, re_, rpost, _, _ = R.moe_align_block_size_ref(ids, block_m, E)
    assert torch.equal(sorted_ids.cpu(), rs) and int(post) == int(rpost)
    assert torch.equal(expert_ids.cpu()[: int(rpost) // block_m], re_[: int(rpost) // block_m])
    C = torch.zeros(T, top_k, N, dtype=torch.bfloat16, device=device)
    ret = invoke_fused_moe_kernel(A.to(device), B.to(device), C, a_s.to(device), b_s.to(device), w.to(device), ids.to(device),
                                  sorted_ids, expert_ids, post, mul_w, top_k, {"BLOCK_SIZE_M": block_m},
                                  use_fp8_w8a8=True, block_shape=[128, 128])
    assert ret is None
    used("tiled" if block_m % 64 == 0 else "fallback")
    check(C, ref, what=f"moe gather block_m={block_m} mul={mul_w}")


@pytest.mark.parametrize("block_m", [256, 128, 64])
def test_moe_gather_with_holes_in_the_slot_sequence(device, block_m):
    """Slots masked out in the middle of an expert's group (sentinel ids) and ids beyond the output's rows: the row
    groups a wave skips are decided from the row map itself, not from a "valid rows are a prefix" assumption.  Rows
    that stay valid match the oracle, every other output row is left untouched."""
    g = _g(block_m + 1)
    T, E, N, K, top_k = 300, 3, 256, 256, 2
    A = fp8_randn((T, K), g)
    B = fp8_randn((E, N, K), g, 0.5)
    a_s = torch.rand(T, K // 128, generator=g) + 0.1
    b_s = torch.rand(E, N // 128, K // 128, generator=g) + 0.1
    w, ids = W.moe_routing(T, E, top_k, seed=7)
    ref = R.ref_fused_moe_gemm(A, B, a_s, b_s, w, ids, False, top_k).reshape(T * top_k, N)
    sorted_ids, expert_ids, post, _, _ = moe_align_block_size(ids.to(device), block_m, E)
    sorted_ids = sorted_ids.clone()
    hole = torch.rand(sorted_ids.numel(), generator=g) < 0.3
    hole[:40] = True                                  # a whole leading stretch of the first tile as well
    sorted_ids[hole.to(device)] = T * top_k           # the sentinel
    num_valid = T * top_k - 37                        # ids >= num_valid have no output row
    C = torch.zeros(num_valid, N, dtype=torch.bfloat16, device=device)
    _lib.fp8_moe_gemm(C, A.to(device), B.to(device), a_s.to(device), b_s.to(device), w.to(device), sorted_ids, expert_ids, post,
                      False, top_k, block_m)
    used("tiled")
    kept = torch.zeros(T * top_k, dtype=torch.bool)
    live = sorted_ids.cpu()
    live = live[(live >= 0) & (live < num_valid)].long()
    kept[live] = True
    kept = kept[:num_valid]
    check(C[kept.to(device)], ref[:num_valid][kept], what=f"gather with holes, block_m={block_m}")
    assert (C[(~kept).to(device)] == 0).all()
    if block_m >= 128:
        B2 = fp8_randn((E, 2 * 128, K), g, 0.5)
        b2_s = torch.rand(E, 2, K // 128, generator=g) + 0.1
        C1 = torch.zeros(T, top_k, 256, dtype=torch.bfloat16, device=device)
        invoke_fused_moe_kernel(A.to(device), B2.to(device), C1, a_s.to(device), b2_s.to(device), w.to(device), ids.to(device),
                                sorted_ids, expert_ids, post, False, top_k, {"BLOCK_SIZE_M": block_m}, use_fp8_w8a8=True)
        q2, s2 = _lib.silu_mul_quant_1x128(C1.view(T * top_k, 256)[:num_valid].contiguous())
        q, s_ = _lib.fp8_moe_gemm_silu_quant(A.to(device), B2.to(device), a_s.to(device), b2_s.to(device), sorted_ids, expert_ids, post,
                                             top_k, block_m, num_valid, torch.bfloat16)
        kd = kept.to(device)
        assert torch.equal(q.view(torch.uint8)[kd], q2.view(torch.uint8)[kd]) and torch.equal(s_[kd], s2[kd])


@pytest.mark.parametrize("bm,bn", [(96, 128), (160, 128), (192, 128), (256, 320)])
def test_grouped_gemms_replace_an_override_by_a_tile_that_only_dense_problems_have(device, bm, bn):
    """Tile overrides that name a dense kernel's tile: the ragged and the gather GEMM run with the tile they pick themselves."""
    impl = tilegym_amd.backend._REGISTRY["flashinfer.gemm.ragged_block_scaled_bmm"]["hip"]
    sizes = [300, 0, 17]
    a, b, a_s, b_s, ptr = _ragged_inputs(sizes, 384, 256, bm)
    args = [t.to(device) for t in (a, b, a_s, b_s, ptr)] + [max(sizes)]
    base = impl(*args)
    want = used("tiled")
    out = impl(*args, kernel_configs={"BLOCK_M": bm, "BLOCK_N": bn})
    assert used("tiled") == want
    assert torch.equal(out, base)
    check(out, R.ref_ragged_block_scaled_bmm(a, b, a_s, b_s, ptr), what=f"ragged, {bm} x {bn} asked for")
    T, E, N, K, top_k = 200, 3, 384, 256, 2
    block_m = 192 if bm == 96 else bm                 # (a multiple of the override's rows)
    g = _g(bm)
    A, B = fp8_randn((T, K), g).to(device), fp8_randn((E, N, K), g, 0.5).to(device)
    as_, bs_ = (torch.rand(T, K // 128, generator=g) + 0.1).to(device), (torch.rand(E, N // 128, K // 128, generator=g) + 0.1).to(device)
    w, ids = W.moe_routing(T, E, top_k, seed=9)
    sorted_ids, expert_ids, post, _, _ = moe_align_block_size(ids.to(device), block_m, E)
    outs, cfgs = [], []
    for kc in (None, {"BLOCK_M": bm, "BLOCK_N": bn}):
        C = torch.zeros(T * top_k, N, dtype=torch.bfloat16, device=device)
        _lib.fp8_moe_gemm(C, A, B, as_, bs_, w.to(device), sorted_ids, expert_ids, post, False, top_k, block_m, kc)
        outs.append(C)
        cfgs.append(_lib.last_config())
    assert cfgs[0] == cfgs[1] and torch.equal(*outs)
    ref = R.ref_fused_moe_gemm(A.cpu(), B.cpu(), as_.cpu(), bs_.cpu(), w, ids, False, top_k)
    check(outs[1].view(T, top_k, N), ref, what=f"gather, {bm} x {bn} asked for")


def test_moe_fc2_shape_top_k_1(device):
    """Second MoE GEMM: activations already expanded per slot (top_k = 1), routed weight applied
    (src/tilegym/ops/moe_interface.py:290-307)."""
    g = _g(77)
    T, E, N, K, top_k = 40, 4, 128, 384, 2
    w, ids = W.moe_routing(T, E, top_k, seed=2)
    A = fp8_randn((T * top_k, K), g)
    B = fp8_randn((E, N, K), g, 0.5)
    a_s = torch.rand(T * top_k, 3, generator=g) + 0.1
    b_s = torch.rand(E, 1, 3, generator=g) + 0.1
    ref = R.ref_fused_moe_gemm(A, B, a_s, b_s, w, ids, True, 1)
    sorted_ids, expert_ids, post, _, _ = moe_align_block_size(ids.to(device), 64, E)
    C = torch.zeros(T, top_k, N, dtype=torch.bfloat16, device=device)
    invoke_fused_moe_kernel(A.to(device), B.to(device), C, a_s.to(device), b_s.to(device), w.to(device), ids.to(device),
                            sorted_ids, expert_ids, post, True, 1, {"BLOCK_SIZE_M": 64})
    check(C, ref, what="moe fc2")


@pytest.mark.parametrize("T,top_k,E,bs,dtype", [(4, 3, 4, 4, torch.int64), (1, 1, 1, 16, torch.int32), (77, 6, 64, 16, torch.int64),
                                                 (4096, 6, 64, 128, torch.int32), (1000, 2, 512, 64, torch.int64),
                                                 (333, 8, 8, 1, torch.int32),
                                                 (7001, 6, 160, 256, torch.int32), (1025, 1, 3, 64, torch.int64)])
def test_moe_align_kernel_matches_oracle(device, T, top_k, E, bs, dtype):
    """All five outputs, bit for bit, against the oracle (stable order inside an expert, sentinel
    fill, padded prefix sums); empty experts, one expert, block size 1, int32 and int64 ids, one to
    the largest number of workgroups (one per 1024 ids, at most 32), slices that end inside the last
    workgroup."""
    g = _g(T + E)
    ids = torch.randint(0, E, (T, top_k), generator=g)
    if E >= 8:
        ids[ids == 3] = 5  # an expert without tokens
    want = R.moe_align_block_size_ref(ids, bs, E)
    got = moe_align_block_size(ids.to(dtype).to(device), bs, E)
    names = ["sorted_ids", "expert_ids", "num_tokens_post_padded", "cumsum", "max_expert_count"]
    nblk_used = int(want[2]) // bs
    for name, w, gt in zip(names, want, got):
        w, gt = w.reshape(-1).long(), gt.reshape(-1).long().cpu()
        if name == "expert_ids":  # entries past the padded total are unspecified in the reference
            w, gt = w[:nblk_used], gt[:nblk_used]
        assert w.numel() == gt.numel(), name
        assert torch.equal(w, gt), f"{name} differs"
    again = moe_align_block_size(ids.to(dtype).to(device), bs, E)
    assert all(torch.equal(a, b) for a, b in zip(got, again))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("ids_dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("T,k,E,bs,H", [(4096, 6, 64, 256, 2048), (33, 2, 8, 16, 128), (1, 8, 512, 64, 1024), (700, 4, 20, 128, 384)])
def test_moe_align_and_quantizer_in_one_launch(device, dtype, ids_dtype, T, k, E, bs, H):
    """tg_moe_align_quant_1x128: all seven outputs bit for bit those of the two stand-alone launches (and so of the oracle)."""
    from tilegym_amd.suites.unsloth.ops import act_quant

    g = _g(T * 3 + E + H)
    ids = torch.randint(0, E, (T, k), generator=g).to(ids_dtype).to(device)
    x = (torch.randn(T, H, generator=g) * torch.exp(torch.randn(T, 1, generator=g))).to(dtype)
    x[0, :128] = 0.0
    xd = x.to(device)
    want = moe_align_block_size(ids, bs, E)
    q_want, s_want = act_quant(xd, 128)
    got = _lib.moe_align_quant_1x128(ids, bs, E, xd)
    for a_, b_ in zip(got[:5], want):
        assert torch.equal(a_, b_)
    assert torch.equal(got[5].view(torch.uint8), q_want.view(torch.uint8)) and torch.equal(got[6], s_want)
    q_ref, s_ref = R.quantize_act_1x128(x, 128, None)
    assert torch.equal(got[5].cpu().view(torch.uint8), q_ref.view(torch.uint8)) and torch.equal(got[6].cpu(), s_ref)


def test_moe_align_limits(device):
    """More experts than the one-launch kernel takes is an explicit error (no torch-op path); an empty routing
    gives the fill values."""
    with pytest.raises(NotImplementedError):
        moe_align_block_size(torch.zeros(50, 4, dtype=torch.int64, device=device), 32, 600)
    s_, e_, post, cum, mx = moe_align_block_size(torch.zeros(0, 2, dtype=torch.int64, device=device), 16, 8)
    want = R.moe_align_block_size_ref(torch.zeros(0, 2, dtype=torch.int64), 16, 8)
    assert s_.numel() == want[0].numel() and int(post) == 0 and int(mx) == 0 and cum.cpu().tolist() == [0] * 9


# ----------------------------------------------------------------------------- activation quantizers
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape", [(1, 128), (7, 384), (3, 5, 256), (4096, 2048)])
def test_act_quant_kernels_bit_exact(device, dtype, shape):
    """Codes and scales, bit for bit, against the oracle: both scale rules, an all-zero group,
    values that hit +-448, tiny groups (subnormal codes), ties."""
    from tilegym_amd.suites.flashinfer.ops import per_token_group_quant_8bit
    from tilegym_amd.suites.unsloth.ops import act_quant

    g = _g(sum(shape))
    x = torch.randn(shape, generator=g) * torch.exp(torch.randn(shape[:-1] + (1,), generator=g) * 3)
    flat = x.reshape(-1, 128)
    flat[0] = 0.0                                   # all-zero group
    if flat.shape[0] > 2:
        flat[1] *= 1e-12                            # amax below the flashinfer eps
        flat[2, :8] = torch.tensor([448.0, -448.0, 224.0, 0.5, 17.0, 19.0, 21.0, 23.0])
    x = x.clamp(-6e4, 6e4).to(dtype)  # finite in f16
    for rule, fn, eps in (("unsloth", lambda t: act_quant(t, 128), None),
                          ("flashinfer", lambda t: per_token_group_quant_8bit(t, 128), 1e-10)):
        q_ref, s_ref = R.quantize_act_1x128(x, 128, eps)
        q, s = fn(x.to(device))
        assert q.dtype == FP8 and s.dtype == torch.float32 and q.shape == x.shape and s.shape == s_ref.shape
        assert torch.equal(s.cpu().view(torch.int32), s_ref.view(torch.int32)), f"{rule}: scales differ"
        bad = q.cpu().view(torch.uint8) != q_ref.view(torch.uint8)
        assert not bad.any(), f"{rule}: {int(bad.sum())} of {bad.numel()} codes differ"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("group", [16, 32, 64, 128])
@pytest.mark.parametrize("tokens,hidden", [(1, 128), (513, 2048), (37, 384)])
def test_group_quantizer_forms_bit_exact(device, dtype, group, tokens, hidden):
    """Group sizes and scale layouts of per_token_group_quant_8bit
    (tests/suites/flashinfer/test_per_token_group_quant_8bit.py:70-110 sweeps the same group sizes and
    513 tokens): row-major, column-major, the aligned column-major form (returned row-major, as the
    reference returns it), power-of-two scales; and act_quant with the same group sizes.  Codes and
    scales bit for bit against the oracle."""
    from tilegym_amd.suites.flashinfer.ops import per_token_group_quant_8bit
    from tilegym_amd.suites.unsloth.ops import act_quant

    g = _g(tokens + hidden + group)
    x = torch.randn(tokens, hidden, generator=g) * torch.exp(torch.randn(tokens, 1, generator=g) * 2)
    flat = x.reshape(-1, group)
    flat[0] = 0.0
    if flat.shape[0] > 3:
        flat[1] *= 1e-12
        flat[2] = 448.0 * 2.0 ** -5 * torch.sign(flat[2] + 1e-30)   # plain scale exactly 2^-5
        flat[3, 0] = 448.0 * 2.0 ** -5 * 1.5                        # plain scale 1.5 * 2^-5 at least
    x = x.clamp(-6e4, 6e4).to(dtype)
    xd = x.to(device)
    G = hidden // group

    def same(q, s, q_ref, s_ref, what):
        assert q.dtype == q_ref.dtype and s.dtype == torch.float32 and q.shape == x.shape and s.shape == s_ref.shape, what
        assert torch.equal(s.cpu().view(torch.int32), s_ref.view(torch.int32)), f"{what}: scales differ"
        bad = q.cpu().view(torch.uint8) != q_ref.view(torch.uint8)
        assert not bad.any(), f"{what}: {int(bad.sum())} of {bad.numel()} codes differ"

    q_ref, s_ref = R.quantize_act_1x128(x, group, 1e-10)
    q, s = per_token_group_quant_8bit(xd, group)
    assert s.is_contiguous()
    same(q, s, q_ref, s_ref, "row-major")
    q, s = per_token_group_quant_8bit(xd, group, column_major_scales=True)
    assert s.shape == (tokens, G) and (G == 1 or tokens == 1 or s.stride() == (1, tokens))
    same(q, s, q_ref, s_ref, "column-major")
    q, s = per_token_group_quant_8bit(xd, group, column_major_scales=True, scale_tma_aligned=True)
    assert s.is_contiguous()
    same(q, s, q_ref, s_ref, "aligned column-major")
    q_ref2, s_ref2 = R.quantize_act_1x128(x, group, 1e-10, ue8m0=True)
    q, s = per_token_group_quant_8bit(xd, group, column_major_scales=True, scale_ue8m0=True)
    same(q, s, q_ref2, s_ref2, "power-of-two scales")
    q, s = per_token_group_quant_8bit(xd, group, column_major_scales=True, scale_tma_aligned=True, scale_ue8m0=True)
    same(q, s, q_ref2, s_ref2, "power-of-two scales, aligned")
    q_ref3, s_ref3 = R.quantize_act_1x128(x, group, None)
    q, s = act_quant(xd, group)
    same(q, s, q_ref3, s_ref3, "act_quant")
    with pytest.raises(AssertionError):
        per_token_group_quant_8bit(xd, group, scale_ue8m0=True)     # needs column_major_scales, as in the reference
    # int8 destination (the reference's test sweeps dst_dtype over e4m3 and int8, test_per_token_group_quant_8bit.py:73)
    qi_ref, si_ref = R.quantize_act_1x128(x, group, 1e-10, dst_dtype=torch.int8)
    q, s = per_token_group_quant_8bit(xd, group, dst_dtype=torch.int8)
    same(q, s, qi_ref, si_ref, "int8 row-major")
    q, s = per_token_group_quant_8bit(xd, group, dst_dtype=torch.int8, column_major_scales=True)
    same(q, s, qi_ref, si_ref, "int8 column-major")
    qi_ref2, si_ref2 = R.quantize_act_1x128(x, group, 1e-10, ue8m0=True, dst_dtype=torch.int8)
    q, s = per_token_group_quant_8bit(xd, group, dst_dtype=torch.int8, column_major_scales=True, scale_tma_aligned=True, scale_ue8m0=True)
    same(q, s, qi_ref2, si_ref2, "int8 power-of-two scales, aligned")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("M,N,bs", [(256, 384, 128), (200, 300, 128), (70, 150, 32), (2816, 2048, 128), (33, 48, 16), (5, 7, 3)])
def test_weight_dequant_bit_exact(device, dtype, M, N, bs):
    """Every e4m3 code (NaN codes included) times a block scale, rounded once to the output type,
    against the oracle; ragged edge blocks, vector and element forms of the kernel."""
    from tilegym_amd.suites.unsloth.ops import weight_dequant

    g = _g(M + N + bs)
    codes = torch.randint(0, 256, (M, N), generator=g, dtype=torch.int32).to(torch.uint8)
    w = codes.view(FP8)
    sc = torch.exp(torch.randn(-(-M // bs), -(-N // bs), generator=g) * 2)
    y_ref = R.weight_dequant(w, sc, bs, dtype)
    y = weight_dequant(w.to(device), sc.to(device), bs, dtype)
    assert y.dtype == dtype and y.shape == (M, N)
    nan = torch.isnan(y_ref.float())
    assert torch.equal(torch.isnan(y.cpu().float()), nan)
    bits = torch.int32 if dtype == torch.float32 else torch.int16
    assert torch.equal(y.cpu().view(bits)[~nan], y_ref.view(bits)[~nan])


def test_quantizers_at_the_reference_tests_shapes(device):
    """The shapes the reference's own tests sweep: weight_dequant (tests/suites/unsloth/test_fp8.py:41-50),
    act_quant (:99-108,129-135), per_token_group_quant_8bit with 512 and 513 tokens of 2048
    (tests/suites/flashinfer/test_per_token_group_quant_8bit.py:71-73), bf16 inputs as there."""
    from tilegym_amd.suites.flashinfer.ops import per_token_group_quant_8bit
    from tilegym_amd.suites.unsloth.ops import act_quant, weight_dequant

    for (M, N) in ((256, 256), (512, 1024), (384, 768), (2048, 4096), (4096, 8192)):
        g = _g(M + N)
        w = torch.randn(M, N, generator=g)
        wq, ws = R.quantize_weight_128x128(w)
        y = weight_dequant(wq.to(device), ws.to(device), 128)
        assert y.dtype == torch.bfloat16
        assert torch.equal(y.cpu().view(torch.int16), R.weight_dequant(wq, ws, 128, torch.bfloat16).view(torch.int16)), (M, N)
    for shape in ((256, 256), (64, 1024), (128, 512), (1024, 4096), (2048, 8192), (256, 128), (128, 384)):
        x = torch.randn(shape, generator=_g(sum(shape))).to(torch.bfloat16)
        q, sc = act_quant(x.to(device), block_size=128)
        q_ref, s_ref = R.quantize_act_1x128(x, 128, None)
        assert torch.equal(sc.cpu(), s_ref) and torch.equal(q.cpu().view(torch.uint8), q_ref.view(torch.uint8)), shape
    for tokens in (512, 513):
        x = torch.randn(tokens, 2048, generator=_g(tokens)).to(torch.bfloat16)
        for group in (16, 32, 64, 128):
            for col, aligned, pow2 in ((False, False, False), (True, False, False), (True, True, False), (True, False, True), (True, True, True)):
                q, sc = per_token_group_quant_8bit(x.to(device), group_size=group, eps=1e-10, dst_dtype=torch.float8_e4m3fn,
                                                   column_major_scales=col, scale_tma_aligned=aligned, scale_ue8m0=pow2)
                q_ref, s_ref = R.quantize_act_1x128(x, group, 1e-10, ue8m0=pow2)
                assert torch.equal(sc.cpu(), s_ref) and torch.equal(q.cpu().view(torch.uint8), q_ref.view(torch.uint8)), (tokens, group, col, aligned, pow2)


def test_quantize_then_gemm_end_to_end(device):
    """bf16 activations -> HIP quantizer -> block-scaled GEMM, against the oracle on the same bf16 input."""
    from tilegym_amd.suites.unsloth.ops import act_quant

    g = _g(5)
    x = torch.randn(96, 512, generator=g).to(torch.bfloat16)
    case = W.block_scaled_case(8, 384, 512, seed=3)
    qa_ref, sa_ref = R.quantize_act_1x128(x, 128, None)
    ref = R.ref_w8a8_block_fp8_matmul(qa_ref, case.b, sa_ref, case.scale_b, None, torch.bfloat16)
    qa, sa = act_quant(x.to(device), 128)
    out = w8a8_block_fp8_matmul(qa, case.b.to(device), sa, case.scale_b.to(device), None, torch.bfloat16)
    check(out, ref, what="quantize + block-scaled GEMM")


# ----------------------------------------------------------------------------- the MoE layer around the GEMMs
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("R_,I", [(5, 128), (64, 1408), (33, 200), (1, 8)])
def test_silu_mul_quant_kernel(device, dtype, R_, I):
    """Dequantized activation within one 16-bit ulp of the oracle's and scales equal to 1e-6 relative (device
    and host exp differ in the last bit now and then, which can move the 16-bit rounding of one value)."""
    g = _g(R_ + I)
    x = (torch.randn(R_, 2 * I, generator=g) * 2).to(dtype)
    x[0, :8] = 0
    q_ref, s_ref, act = R.ref_silu_mul_quant(x)
    q, s = _lib.silu_mul_quant_1x128(x.to(device))
    assert q.shape == q_ref.shape and s.shape == s_ref.shape
    assert torch.allclose(s.cpu(), s_ref, rtol=1e-2, atol=0)
    deq = R.fp8_to_f32(q.cpu()) * s.cpu().repeat_interleave(128, 1)[:, :I]
    deq_ref = R.fp8_to_f32(q_ref) * s_ref.repeat_interleave(128, 1)[:, :I]
    step = s_ref.repeat_interleave(128, 1)[:, :I] * 32          # one e4m3 step at the top binade is 32 * scale
    assert ((deq - deq_ref).abs() <= step + 1e-12).all()
    same = (q.cpu().view(torch.uint8) == q_ref.view(torch.uint8)).float().mean()
    assert same > 0.995, f"only {same:.4f} of the codes equal the oracle's"


@pytest.mark.parametrize("block_m", [256, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,E,top_k,H,I", [(64, 4, 2, 256, 128), (300, 8, 2, 512, 384), (700, 3, 1, 128, 1408)])
def test_moe_gemm_silu_quant_equals_the_two_steps(device, dtype, T, E, top_k, H, I, block_m):
    """GEMM1 with the activation and the 1x128 re-quantization in its epilogue returns the very bits of
    GEMM1 (same row blocks) followed by the stand-alone activation kernel, and stays within that kernel's
    bar against the oracle (src/tilegym/ops/moe_interface.py:252-277, src/tilegym/ops/ops.py:172-193)."""
    g = _g(T + I)
    A = fp8_randn((T, H), g)
    B = fp8_randn((E, 2 * I, H), g, 0.5)
    a_s = torch.rand(T, H // 128, generator=g) * 0.05 + 0.01
    b_s = torch.rand(E, 2 * I // 128, H // 128, generator=g) + 0.1
    w, ids = W.moe_routing(T, E, top_k, seed=3)
    if E > 2:
        ids[ids == 1] = 2  # an expert without tokens
    Ad, Bd, asd, bsd = A.to(device), B.to(device), a_s.to(device), b_s.to(device)
    sorted_ids, expert_ids, post, _, _ = moe_align_block_size(ids.to(device), block_m, E)
    C = torch.zeros(T, top_k, 2 * I, dtype=dtype, device=device)
    invoke_fused_moe_kernel(Ad, Bd, C, asd, bsd, w.to(device), ids.to(device), sorted_ids, expert_ids, post,
                            False, top_k, {"BLOCK_SIZE_M": block_m}, compute_type=dtype, use_fp8_w8a8=True)
    q2, s2 = _lib.silu_mul_quant_1x128(C.view(T * top_k, 2 * I))
    assert _lib.moe_gemm_silu_quant_ok(Bd, block_m)
    q, s = _lib.fp8_moe_gemm_silu_quant(Ad, Bd, asd, bsd, sorted_ids, expert_ids, post, top_k, block_m, T * top_k, dtype)
    used("tiled")
    assert torch.equal(q.view(torch.uint8), q2.view(torch.uint8)) and torch.equal(s, s2)
    # against the oracle: its GEMM1 output rounded to the 16-bit type, then its activation + quantization
    ref_c = R.ref_fused_moe_gemm(A, B, a_s, b_s, w, ids, False, top_k, out_dtype=dtype).reshape(T * top_k, 2 * I)
    q_ref, s_ref, _ = R.ref_silu_mul_quant(ref_c)
    assert torch.allclose(s.cpu(), s_ref, rtol=2e-2, atol=0)
    deq = R.fp8_to_f32(q.cpu()) * s.cpu().repeat_interleave(128, 1)
    deq_ref = R.fp8_to_f32(q_ref) * s_ref.repeat_interleave(128, 1)
    step = s_ref.repeat_interleave(128, 1) * 32
    # an fp32 re-association difference in the GEMM can move a 16-bit rounding of gate or up, hence two steps
    assert ((deq - deq_ref).abs() <= 2 * step + 1e-12).float().mean() > 0.9999


def test_fused_experts_fp8_fused_activation_path(device):
    """Enough rows per expert for 256-row blocks: fused_moe takes the GEMM1 + activation + quantization
    entry point; checked against the oracle of the whole layer."""
    from tilegym_amd.ops import fused_moe

    g = _g(32)
    T, E, k, H, I = 600, 4, 2, 256, 384
    hidden = torch.randn(T, H, generator=g).to(torch.bfloat16)
    w1q, w1s = R.quantize_weight_128x128(torch.randn(E * 2 * I, H, generator=g) * 0.05)
    w2q, w2s = R.quantize_weight_128x128(torch.randn(E * H, I, generator=g) * 0.05)
    w1q, w1s = w1q.reshape(E, 2 * I, H), w1s.reshape(E, 2 * I // 128, H // 128)
    w2q, w2s = w2q.reshape(E, H, I), w2s.reshape(E, H // 128, I // 128)
    tw, ids = W.moe_routing(T, E, k, seed=5)
    assert (T * k) // E >= 192 and _lib.moe_gemm_silu_quant_ok(w1q, 256)
    ref = R.ref_fused_experts_fp8(hidden, w1q, w2q, w1s, w2s, tw, ids)
    out = fused_moe(hidden.to(device), w1q.to(device), w2q.to(device), tw.to(device), ids.to(device),
                    w1_scale=w1s.to(device), w2_scale=w2s.to(device))
    ok, rep = R.compare_to_oracle(out, ref, RTOL, ATOL)
    assert rep["matched"] >= 0.999 and rep["max_rel_to_sigma"] <= 0.1, rep


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_moe_sum_kernel(device, dtype):
    g = _g(8)
    x = torch.randn(37, 6, 264, generator=g).to(dtype)
    out = torch.empty(37, 264, dtype=dtype, device=device)
    _lib.moe_sum(x.to(device), out)
    acc = x[:, 0].float()
    for j in range(1, 6):
        acc = acc + x[:, j].float()
    assert torch.equal(out.cpu(), acc.to(dtype))


@pytest.mark.parametrize("in_dtype", [torch.bfloat16, torch.float16, "fp8"])
def test_fused_experts_fp8_small(device, in_dtype):
    from tilegym_amd.ops import fused_experts_impl, fused_moe

    g = _g(31)
    T, E, k, H, I = 40, 8, 2, 256, 384
    dt = torch.bfloat16 if in_dtype == "fp8" else in_dtype
    hidden = torch.randn(T, H, generator=g).to(dt)
    w1q, w1s = R.quantize_weight_128x128(torch.randn(E * 2 * I, H, generator=g) * 0.05)
    w2q, w2s = R.quantize_weight_128x128(torch.randn(E * H, I, generator=g) * 0.05)
    w1q, w1s = w1q.reshape(E, 2 * I, H), w1s.reshape(E, 2 * I // 128, H // 128)
    w2q, w2s = w2q.reshape(E, H, I), w2s.reshape(E, H // 128, I // 128)
    tw, ids = W.moe_routing(T, E, k, seed=4)
    ids[ids == 5] = 6  # an expert without tokens
    if in_dtype == "fp8":
        xq, xs = R.quantize_act_1x128(hidden, 128, None)
        ref = R.ref_fused_experts_fp8(xq, w1q, w2q, w1s, w2s, tw, ids, a1_scale=xs)
        # fp8 input: the reference types the output f16 unless the input is bf16 (moe_interface.py:196)
        out = fused_experts_impl(xq.to(device), w1q.to(device), w2q.to(device), tw.to(device), ids.to(device), use_fp8_w8a8=True,
                                 w1_scale=w1s.to(device), w2_scale=w2s.to(device), a1_scale=xs.to(device))
        assert out.dtype == torch.float16
    else:
        ref = R.ref_fused_experts_fp8(hidden, w1q, w2q, w1s, w2s, tw, ids)
        out = fused_moe(hidden.to(device), w1q.to(device), w2q.to(device), tw.to(device), ids.to(device),
                        w1_scale=w1s.to(device), w2_scale=w2s.to(device))
        assert out.dtype == in_dtype
    # a flipped activation code (host / device exp) moves one input of the second GEMM by one e4m3 step:
    # within the stated tolerance, not within one output ulp
    ok, rep = R.compare_to_oracle(out, ref, RTOL, ATOL)
    assert ok, rep
    with pytest.raises(NotImplementedError):
        fused_experts_impl(hidden.to(device), w1q.to(device), w2q.to(device), tw.to(device), ids.to(device), use_fp8_w8a8=False)


@pytest.mark.parametrize("T,H,I,E,k", [(16, 512, 256, 8, 2), (32, 1024, 512, 16, 4), (64, 1024, 512, 20, 8)])
def test_fused_moe_fp8_at_the_reference_tests_configurations(device, T, H, I, E, k):
    """Token / width / expert counts and data recipe of Test_MOE.test_op (tests/ops/test_moe.py:73-145: hidden N(0, 0.5),
    weights N(0, 0.1), topk_ids drawn with randint, so a token may name one expert twice, softmax of N(0,1) routing
    weights) through the block-scaled FP8 layer, against the oracle."""
    from tilegym_amd.ops import fused_moe

    g = _g(T + E)
    hidden = (torch.randn(T, H, generator=g) * 0.5).to(torch.float16)
    w1q, w1s = R.quantize_weight_128x128(torch.randn(E * 2 * I, H, generator=g) * 0.1)
    w2q, w2s = R.quantize_weight_128x128(torch.randn(E * H, I, generator=g) * 0.1)
    w1q, w1s = w1q.reshape(E, 2 * I, H), w1s.reshape(E, 2 * I // 128, H // 128)
    w2q, w2s = w2q.reshape(E, H, I), w2s.reshape(E, H // 128, I // 128)
    ids = torch.randint(0, E, (T, k), generator=g)
    tw = torch.softmax(torch.randn(T, k, generator=g), dim=-1).to(torch.float16)
    ref = R.ref_fused_experts_fp8(hidden, w1q, w2q, w1s, w2s, tw.float(), ids.to(torch.int32))
    out = fused_moe(hidden.to(device), w1q.to(device), w2q.to(device), tw.to(device), ids.to(device),
                    w1_scale=w1s.to(device), w2_scale=w2s.to(device))
    assert out.dtype == torch.float16 and out.shape == (T, H)
    ok, rep = R.compare_to_oracle(out, ref, RTOL, ATOL)
    assert rep["matched"] >= 0.999 and rep["max_rel_to_sigma"] <= 0.1, rep


def test_launches_replay_from_a_hip_graph(device):
    """Every entry point only enqueues on the caller's stream (no allocation, synchronisation or memset of its
    own), so a caller may capture it: the MoE layer (align, quantizer, both grouped GEMMs with the fused
    activation epilogue, top-k sum), a split-K decode GEMM with its workspace and the persistent 256x256 kernel are
    captured once and replayed three times with eager work in between; every replay must reproduce the eager result
    bit for bit."""
    from tilegym_amd.ops import fused_moe

    g = _g(33)
    T, E, k, H, I = 600, 4, 2, 256, 384
    hidden = torch.randn(T, H, generator=g).to(torch.bfloat16).to(device)
    w1q, w1s = R.quantize_weight_128x128(torch.randn(E * 2 * I, H, generator=g) * 0.05)
    w2q, w2s = R.quantize_weight_128x128(torch.randn(E * H, I, generator=g) * 0.05)
    w1q, w1s = w1q.reshape(E, 2 * I, H).to(device), w1s.reshape(E, 2 * I // 128, H // 128).to(device)
    w2q, w2s = w2q.reshape(E, H, I).to(device), w2s.reshape(E, H // 128, I // 128).to(device)
    tw, ids = W.moe_routing(T, E, k, seed=6)
    tw, ids = tw.to(device), ids.to(device)
    a = fp8_randn((16, 14336), g).to(device)
    b = fp8_randn((4096, 14336), g, 0.05).to(device)
    one = torch.ones(1, device=device)
    a2 = fp8_randn((700, 640), g).to(device)
    b2 = fp8_randn((520, 640), g, 0.05).to(device)

    def work():
        out = fused_moe(hidden, w1q, w2q, tw, ids, w1_scale=w1s, w2_scale=w2s)
        big = matmul(a2, b2, trans_b=True, scale_a=one, scale_b=one, out_dtype=torch.bfloat16,
                     kernel_configs={"KERNEL": "tiled", "BLOCK_M": 256, "BLOCK_N": 256})
        assert _lib.last_config()["BLOCK_M"] == 256
        return out, matmul(a, b, trans_b=True, scale_a=one, scale_b=one, out_dtype=torch.bfloat16), big

    eager_moe, eager_mm, eager_big = work()
    assert _lib.last_config()["SPLIT_K"] > 1  # the decode GEMM (the last launch of work()) takes the split-K path (workspace + reduction)
    assert torch.equal(eager_big, matmul(a2, b2, trans_b=True, scale_a=one, scale_b=one, out_dtype=torch.bfloat16,
                                         kernel_configs={"KERNEL": "tiled", "BLOCK_M": 128, "BLOCK_N": 128}))
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        work()  # warm-up on a side stream; torch.cuda.graph captures on a stream of its own, so the workspace of the
        # captured split-K GEMM is allocated under capture, from the graph's pool (see _lib.workspace_for)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        g_moe, g_mm, g_big = work()
    for rep in range(3):
        g_moe.zero_()
        g_mm.zero_()
        g_big.zero_()
        hidden.add_(0.0)  # eager work between the replays
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(g_moe, eager_moe), f"MoE layer differs on replay {rep}"
        assert torch.equal(g_mm, eager_mm), f"split-K GEMM differs on replay {rep}"
        assert torch.equal(g_big, eager_big), f"persistent 256x256 GEMM differs on replay {rep}"


def test_graph_workspace_survives_a_larger_eager_gemm(device):
    """A captured split-K GEMM keeps writing its partial sums to the workspace it was captured with.  A later,
    larger GEMM on the same stream makes the binding allocate a bigger workspace: the captured one must stay
    alive (never returned to the allocator), so that tensors allocated afterwards cannot land in it and be
    overwritten by a replay."""
    g = _g(41)
    a = fp8_randn((16, 14336), g).to(device)
    b = fp8_randn((4096, 14336), g, 0.05).to(device)
    one = torch.ones(1, device=device)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        eager = matmul(a, b, trans_b=True, scale_a=one, scale_b=one, out_dtype=torch.bfloat16)
        assert _lib.last_config()["SPLIT_K"] > 1
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            captured = matmul(a, b, trans_b=True, scale_a=one, scale_b=one, out_dtype=torch.bfloat16)
        # a larger split-K problem on the same stream: the binding has to grow that stream's workspace
        a2 = fp8_randn((64, 14336), g).to(device)
        big = matmul(a2, b, trans_b=True, scale_a=one, scale_b=one, out_dtype=torch.bfloat16)
        assert _lib.last_config()["SPLIT_K"] > 1
        torch.cuda.synchronize()
        # fill freshly allocated memory with a pattern, replay, and check that neither side was disturbed
        fresh = [torch.full((1 << 20,), 3, dtype=torch.int32, device=device) for _ in range(16)]
        for rep in range(3):
            captured.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(captured, eager), f"replay {rep} differs"
            assert all(int(t.min()) == 3 and int(t.max()) == 3 for t in fresh), "a replay wrote into memory it no longer owns"
        del big


def test_fused_moe_more_tokens_than_one_chunk(device):
    """33000 tokens: fused_experts_impl works in chunks of 32768 tokens (src/tilegym/ops/moe_interface.py:216-233);
    rows around the chunk boundary and at both ends against the oracle."""
    from tilegym_amd.ops import fused_moe

    g = _g(3)
    T, E, k, H, I = 33000, 4, 2, 256, 128
    hidden = torch.randn(T, H, generator=g).to(torch.bfloat16)
    w1q, w1s = R.quantize_weight_128x128(torch.randn(E * 2 * I, H, generator=g) * 0.05)
    w2q, w2s = R.quantize_weight_128x128(torch.randn(E * H, I, generator=g) * 0.05)
    w1q, w1s = w1q.reshape(E, 2 * I, H), w1s.reshape(E, 2 * I // 128, H // 128)
    w2q, w2s = w2q.reshape(E, H, I), w2s.reshape(E, H // 128, I // 128)
    tw, ids = W.moe_routing(T, E, k, seed=5)
    out = fused_moe(hidden.to(device), w1q.to(device), w2q.to(device), tw.to(device), ids.to(device),
                    w1_scale=w1s.to(device), w2_scale=w2s.to(device))
    rows = torch.cat([torch.arange(0, 40), torch.arange(32748, 32808), torch.arange(T - 40, T)])
    ref = R.ref_fused_experts_fp8(hidden[rows], w1q, w2q, w1s, w2s, tw[rows], ids[rows])
    ok, rep = R.compare_to_oracle(out[rows.to(device)], ref, RTOL, ATOL)
    # one flipped activation code moves the 256 outputs of its token (I = 128: one of 128 inputs of the second GEMM)
    assert rep["matched"] >= 0.99 and rep["max_rel_to_sigma"] <= 0.1, rep


def test_config5_fused_experts_full_size(device):
    """DeepSeek-V2-Lite MoE layer at full size (4096 tokens, 64 experts, top-6, H 2048, I 1408) through
    fused_moe; the oracle is evaluated on 24 sampled tokens (a token's output depends on its own row only)."""
    from tilegym_amd.ops import fused_moe

    up, down = _moe_base("gate_up"), _moe_base("down")
    ids, tw = up.extra["topk_ids"], up.extra["topk_weights"]
    T, H = ids.shape[0], up.b.shape[2]
    hidden = torch.randn(T, H, generator=_g(9)).to(torch.bfloat16)
    out = fused_moe(hidden.to(device), up.b.to(device), down.b.to(device), tw.to(device), ids.to(device),
                    w1_scale=up.b_scale.to(device), w2_scale=down.b_scale.to(device))
    assert out.shape == (T, H) and torch.isfinite(out.float()).all()
    rows = _rows_subset(T, 24)
    ref = R.ref_fused_experts_fp8(hidden[rows], up.b, down.b, up.b_scale, down.b_scale, tw[rows], ids[rows])
    # Two roundings (16-bit, then e4m3) sit between the GEMMs: an fp32 re-association difference in GEMM1
    # now and then flips one activation code, i.e. moves one of the 1408 inputs of GEMM2 by an e4m3 step.
    # Bar for the chained layer: >= 99.9 % of the outputs inside the GEMM tolerance, none beyond 0.1 sigma.
    ok, rep = R.compare_to_oracle(out[rows.to(device)], ref, RTOL, ATOL)
    assert rep["matched"] >= 0.999 and rep["max_rel_to_sigma"] <= 0.1, rep
    again = fused_moe(hidden.to(device), up.b.to(device), down.b.to(device), tw.to(device), ids.to(device),
                      w1_scale=up.b_scale.to(device), w2_scale=down.b_scale.to(device))
    assert torch.equal(out, again)


_MOE_BASE = {}


def _moe_base(which):
    """config 5's full-size grouped case, built once per test process (64 experts' weights are quantized on the CPU)."""
    if which not in _MOE_BASE:
        _MOE_BASE[which] = W.moe_grouped_case(which)
    return _MOE_BASE[which]


@pytest.mark.parametrize("T,E,H,I,k,which", [(3, 8, 512, 256, 2, "gate_up"), (3, 8, 512, 384, 2, "down"), (40, 8, 1024, 128, 2, "gate_up"),
                                             (5, 4, 2048, 1408, 2, "down"), (1, 6, 640, 128, 3, "down"), (2, 5, 128, 200, 1, "gate_up")])
def test_ragged_stream_form(device, T, E, H, I, k, which):
    """The streaming ragged kernel (one grid row per expert) forced at several row counts: empty experts, experts with more
    than 16 rows (several passes over their weights), K of 1 .. 3 steps past a multiple of 512 (the short last piece), N that
    is no multiple of 64, against per-expert oracle GEMMs; untouched rows of the output do not exist.  With four, six
    and eight waves (64 .. 128 weight rows) per workgroup."""
    base = W.moe_grouped_case(which, tokens=max(T, 8), experts=E, hidden=H, inter=I, top_k=k)
    case = W.moe_decode_case(base, T)
    d = case.to(device)
    for waves in (None, 4, 6, 8):
        out = torch.full((case.a.shape[0], case.b.shape[1]), 7.0, dtype=torch.bfloat16, device=device)
        _lib.fp8_ragged_gemm(out, d.a, d.b, d.a_scale, d.b_scale, d.m_indptr, {"KERNEL": "stream"} if waves is None else {"KERNEL": "stream", "WAVES": waves})
        cfg = used("stream")
        assert cfg["ROW_GROUPS"] == 4 and (waves is None or cfg["WAVES"] == waves), cfg
        for e in range(E):
            lo, hi = int(case.m_indptr[e]), int(case.m_indptr[e + 1])
            if hi > lo:
                ref = R.ref_w8a8_block_fp8_matmul(case.a[lo:hi], case.b[e], case.a_scale[lo:hi], case.b_scale[e], None, torch.bfloat16)
                check(out[lo:hi], ref, what=f"ragged stream {which} T={T} expert {e} waves {waves}")


def test_ragged_stream_form_is_the_default_for_one_token(device):
    case = W.moe_decode_case(_moe_base("down"), 1)
    d = case.to(device)
    out = ragged_block_scaled_bmm(d.a, d.b, d.a_scale, d.b_scale, d.m_indptr, 1)
    assert used("stream")["WAVES"] == 4          # six rows x 32 workgroups of 64 weight rows: one per compute unit as it is
    case = W.moe_decode_case(_moe_base("gate_up"), 1)
    d = case.to(device)
    out = ragged_block_scaled_bmm(d.a, d.b, d.a_scale, d.b_scale, d.m_indptr, 1)
    assert used("stream")["WAVES"] == 6          # six rows x 44 workgroups are 264: 96 weight rows per workgroup make it 180
    case = W.moe_decode_case(_moe_base("down"), 16)
    d = case.to(device)
    out = ragged_block_scaled_bmm(d.a, d.b, d.a_scale, d.b_scale, d.m_indptr, 16)
    used("tiled")


@pytest.mark.parametrize("waves", [4, 6, 8])
@pytest.mark.parametrize("sizes", [[0, 16, 17, 1, 32, 33, 0, 5], [0] * 70 + [49, 0, 15, 64] + [0] * 60 + [31], [200], [3] * 5 + [400]])
def test_ragged_stream_form_with_crowded_experts(device, sizes, waves):
    """Experts whose rows end at, before and behind a multiple of 16, on either side of 64 experts, with most of the rows and with all."""
    N, K = 392, 1152
    a, b, a_s, b_s, ptr = _ragged_inputs(sizes, N, K, len(sizes) + sum(sizes), total_extra=7)
    out = torch.zeros(a.shape[0], N, dtype=torch.bfloat16, device=device)
    _lib.fp8_ragged_gemm(out, *[t.to(device) for t in (a, b, a_s, b_s, ptr)], {"KERNEL": "stream", "WAVES": waves})
    assert used("stream")["WAVES"] == waves
    check(out[: sum(sizes)], R.ref_ragged_block_scaled_bmm(a, b, a_s, b_s, ptr)[: sum(sizes)], what=f"{sizes}")
    assert not out[sum(sizes):].any()


@pytest.mark.parametrize("kc", [None, {"KERNEL": "stream"}, {"KERNEL": "tiled"}])
@pytest.mark.parametrize("ptr", [[0, 7, 7, 18, 29], [0, 20, 24, 24, 29], [-5, 7, 7, 18, 20]])
def test_ragged_segments_past_the_rows_are_contained(device, ptr, kc):
    """An m_indptr that gives rows outside the 20 that A and C have: rows inside come out as documented (none of a segment that starts
    below 0), and nothing is written past C.  Operands and result lie inside larger buffers, so that a missing clamp shows as a value."""
    M, N, K, slack = 20, 256, 1024, 32
    a, b, a_s, b_s, _ = _ragged_inputs([M + 2 * slack, 0, 0, 0], N, K, M)
    big = torch.full((M + 2 * slack, N), 3.0, dtype=torch.bfloat16, device=device)
    out = big[slack:slack + M]
    _lib.fp8_ragged_gemm(out, a.to(device)[slack:slack + M], b.to(device), a_s.to(device)[slack:slack + M], b_s.to(device),
                         torch.tensor(ptr, dtype=torch.int32, device=device), kc)
    used("stream" if kc is None else kc["KERNEL"])
    assert bool((big[:slack] == 3).all()) and bool((big[slack + M:] == 3).all())
    a, a_s = a[slack:slack + M], a_s[slack:slack + M]
    for e in range(4):
        lo, hi = ptr[e], min(ptr[e + 1], M)
        if 0 <= lo < hi:
            check(out[lo:hi], R.ref_w8a8_block_fp8_matmul(a[lo:hi], b[e], a_s[lo:hi], b_s[e], None, torch.bfloat16), what=f"{ptr} expert {e}")


@pytest.mark.parametrize("T", [1, 16, 64])
@pytest.mark.parametrize("which", ["gate_up", "down"])
def test_config5_moe_decode_regime(device, which, T):
    """The full-size expert weights (64 x 2816 x 2048 and 64 x 2048 x 1408) with 1 / 16 / 64 tokens routed over them: most
    experts receive no row, the others one to a dozen.  Whole output against per-expert oracle GEMMs; rows of experts
    that received nothing do not exist, and the result does not depend on what the output buffer held."""
    case = W.moe_decode_case(_moe_base(which), T)
    sizes = case.m_indptr[1:] - case.m_indptr[:-1]
    assert int(case.m_indptr[-1]) == T * 6 and int((sizes == 0).sum()) >= 64 - 6 * T
    d = case.to(device)
    out = ragged_block_scaled_bmm(d.a, d.b, d.a_scale, d.b_scale, d.m_indptr, int(sizes.max()))
    for e in range(case.b.shape[0]):
        lo, hi = int(case.m_indptr[e]), int(case.m_indptr[e + 1])
        if hi > lo:
            ref = R.ref_w8a8_block_fp8_matmul(case.a[lo:hi], case.b[e], case.a_scale[lo:hi], case.b_scale[e], None, torch.bfloat16)
            check(out[lo:hi], ref, what=f"config 5 {which} T={T} expert {e}")
    again = ragged_block_scaled_bmm(d.a, d.b, d.a_scale, d.b_scale, d.m_indptr, int(sizes.max()))
    assert torch.equal(out, again)


@pytest.mark.parametrize("T,H,I,E,k,dtype", [(1, 256, 128, 8, 2, torch.bfloat16), (16, 512, 256, 16, 4, torch.float16), (300, 256, 384, 8, 1, torch.bfloat16),
                                            (700, 1024, 128, 64, 6, torch.bfloat16), (5, 128, 128, 3, 3, torch.float16)])
def test_fused_moe_one_call_layer_gives_the_bits_of_the_call_by_call_layer(device, T, H, I, E, k, dtype):
    """tg_fp8_fused_moe (align + quantize, GEMM1 with the activation epilogue, GEMM2, sum from one call, intermediates carved
    from the stream's scratch buffer) against the same four entry points called one by one from Python: identical bits,
    also in place, with top_k = 1, and when the scratch buffer held something else before."""
    from tilegym_amd.ops import fused_moe, moe_interface

    g = _g(T + H + E)
    hidden = (torch.randn(T, H, generator=g) * 0.5).to(dtype).to(device)
    w1q, w1s = R.quantize_weight_128x128(torch.randn(E * 2 * I, H, generator=g) * 0.1)
    w2q, w2s = R.quantize_weight_128x128(torch.randn(E * H, I, generator=g) * 0.1)
    w1q, w1s = w1q.reshape(E, 2 * I, H).to(device), w1s.reshape(E, 2 * I // 128, H // 128).to(device)
    w2q, w2s = w2q.reshape(E, H, I).to(device), w2s.reshape(E, H // 128, -(-I // 128)).to(device)
    ids = torch.randint(0, E, (T, k), generator=g).to(device)
    tw = torch.softmax(torch.randn(T, k, generator=g), dim=-1).to(device)
    assert moe_interface.USE_ONE_CALL_LAYER
    try:
        moe_interface.USE_ONE_CALL_LAYER = False
        want = fused_moe(hidden, w1q, w2q, tw, ids, w1_scale=w1s, w2_scale=w2s)
    finally:
        moe_interface.USE_ONE_CALL_LAYER = True
    # dirty the scratch buffer the one-call form will carve up
    _lib.workspace_for(hidden.device, 1 << 20).fill_(0xAB)
    got = fused_moe(hidden, w1q, w2q, tw, ids, w1_scale=w1s, w2_scale=w2s)
    assert got.dtype == dtype and torch.equal(got, want)
    again = fused_moe(hidden, w1q, w2q, tw.to(torch.float16), ids.to(torch.int32), w1_scale=w1s, w2_scale=w2s)
    assert torch.equal(again, fused_moe(hidden, w1q, w2q, tw.to(torch.float16).float(), ids, w1_scale=w1s, w2_scale=w2s))
    h2 = hidden.clone()
    out = moe_interface.fused_experts_impl(h2, w1q, w2q, tw, ids, inplace=True, use_fp8_w8a8=True, w1_scale=w1s, w2_scale=w2s)
    assert out.data_ptr() == h2.data_ptr() and torch.equal(h2, want)
    ref = R.ref_fused_experts_fp8(hidden.cpu(), w1q.cpu(), w2q.cpu(), w1s.cpu(), w2s.cpu(), tw.cpu(), ids.cpu().to(torch.int32))
    # (a loose bar: with I = 128 the second GEMM has a single quantization group per row, where one flipped e4m3 code of
    # the activation weighs most; the layer's own bar is in the tests of the reference's configurations)
    ok, rep = R.compare_to_oracle(got, ref, RTOL, ATOL)
    assert rep["matched"] >= 0.995 and rep["max_rel_to_sigma"] <= 0.2, rep


@pytest.mark.parametrize("T", [1, 16, 64])
def test_config5_fused_experts_decode_regime(device, T):
    """The whole layer at 1 / 16 / 64 tokens over the full-size weights, every token against the oracle."""
    from tilegym_amd.ops import fused_moe

    up, down = _moe_base("gate_up"), _moe_base("down")
    tw, ids = W.moe_routing(T, up.b.shape[0], up.extra["top_k"], seed=T)
    H = up.b.shape[2]
    hidden = torch.randn(T, H, generator=_g(90 + T)).to(torch.bfloat16)
    out = fused_moe(hidden.to(device), up.b.to(device), down.b.to(device), tw.to(device), ids.to(device),
                    w1_scale=up.b_scale.to(device), w2_scale=down.b_scale.to(device))
    assert out.shape == (T, H) and torch.isfinite(out.float()).all()
    ref = R.ref_fused_experts_fp8(hidden, up.b, down.b, up.b_scale, down.b_scale, tw, ids)
    ok, rep = R.compare_to_oracle(out, ref, RTOL, ATOL)
    assert rep["matched"] >= 0.999 and rep["max_rel_to_sigma"] <= 0.1, rep


def test_native_binding_agrees_with_the_general_path(device):
    """The same call through the native module and, by an option it leaves to Python, through the general path: number
    scales, 3-D activations, f16 scales (converted in Python), empty problems, and the errors both raise."""
    g = _g(77)
    a, b = fp8_randn((6, 256), g).to(device), fp8_randn((24, 256), g, 0.1).to(device)
    s = torch.tensor([0.5], device=device)
    want = matmul(a, b, trans_b=True, scale_a=s, scale_b=0.25, out_dtype=torch.float32, kernel_configs={})
    for sa in (s, 0.5, s.to(torch.float16), s.double()):
        assert torch.equal(matmul(a, b, trans_b=True, scale_a=sa, scale_b=0.25, out_dtype=torch.float32), want)
    kw = dict(trans_a=True, trans_b=True, scale_a=s, scale_b=0.25, out_dtype=torch.float32)
    at = a.t().contiguous()
    assert torch.equal(matmul(at, b, **kw), matmul(at, b, kernel_configs={}, **kw))
    assert matmul(a[:0], b, trans_b=True).shape == (0, 24)
    As, Bs = torch.rand(6, 2, generator=g).to(device), torch.rand(1, 2, generator=g).to(device)
    want = w8a8_block_fp8_matmul(a, b, As, Bs, None, torch.float32, kernel_configs={})
    got = w8a8_block_fp8_matmul(a.view(2, 3, 256), b, As.view(2, 3, 2), Bs, [128, 128], torch.float32)
    assert got.shape == (2, 3, 24) and torch.equal(got.view(6, 24), want)
    assert torch.equal(w8a8_block_fp8_matmul(a, b, As.half(), Bs, None, torch.float32),
                       w8a8_block_fp8_matmul(a, b, As.half().float(), Bs, None, torch.float32))
    with pytest.raises(AssertionError):
        matmul(a, b[:, :128].contiguous(), trans_b=True)
    with pytest.raises(AssertionError):
        matmul(a, b.t(), out_dtype=torch.float32)
    with pytest.raises(NotImplementedError):
        matmul(a, b, trans_b=True, out_dtype=torch.float64)
    with pytest.raises(_lib.TileGymHipError):
        _lib.fp8_gemm(torch.empty(6, 23, device=device), a, b)


def test_calls_without_the_native_binding(device, monkeypatch):
    """The same calls where the native module could not be imported: the ctypes path reaches the same kernels."""
    from tilegym_amd.ops import fused_moe
    from tilegym_amd.quant import act_quant

    g = _g(78)
    a, b = fp8_randn((6, 256), g).to(device), fp8_randn((128, 256), g, 0.1).to(device)
    layer = _device_moe_layer(device, 3, 256, 128, 8, 2, seed=5)
    indptr = torch.tensor([0, 2, 6], dtype=torch.int32, device=device)

    def calls():
        q, s = act_quant(layer[0], 128)
        x, w1, w2, s1, s2, tw, ids = layer
        return [matmul(a, b, trans_b=True, scale_a=0.5, out_dtype=torch.float32), matmul(a, b[:6].t().contiguous(), out_dtype=torch.bfloat16),
                w8a8_block_fp8_matmul(q, b, s, s1[0, :1], [128, 128], torch.bfloat16), q.view(torch.uint8), s,
                ragged_block_scaled_bmm(a, w1[:2], torch.ones(6, 2, device=device), s1[:2], indptr, 4),
                fused_moe(x, w1, w2, tw, ids, w1_scale=s1, w2_scale=s2)]

    want = calls()
    monkeypatch.setattr(_lib, "native", None)
    for got, w in zip(calls(), want):
        assert torch.equal(got, w)


@pytest.mark.parametrize("M,N,K", [(70, 16, 128), (96, 144, 256), (130, 272, 1040), (65, 4112, 4096), (300, 128, 200), (20, 4080, 1008)])
def test_kn_weights_give_the_bits_of_nk_weights(device, M, N, K):
    """(K, N) weights through the 16-byte transpose: edges of its 128 x 128 tiles in both directions, a padded K (rows of the copy
    longer than K: 1040, 200, 1008 are no multiples of 128), against the same weight handed over as (N, K).  A kernel asked for by
    name takes the copy; without one, the narrow tiles may read the weight as it lies."""
    g = _g(M + N + K)
    a, b = fp8_randn((M, K), g).to(device), fp8_randn((N, K), g, 0.3).to(device)
    kn = b.view(torch.uint8).t().contiguous().view(FP8)
    for kernel_configs in ({"KERNEL": "tiled"}, None):
        want = matmul(a, b, trans_b=True, out_dtype=torch.float32, kernel_configs=kernel_configs)
        assert torch.equal(matmul(a, kn, out_dtype=torch.float32, kernel_configs=kernel_configs), want)


@pytest.mark.parametrize("M,N,K", [(1, 16, 128), (16, 48, 256), (17, 4112, 384), (33, 80, 640), (64, 144, 1152), (65, 208, 128), (100, 2064, 1024),
                                   (256, 1040, 512), (512, 64, 512), (64, 16400, 1152)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32, FP8])
def test_kn_weights_read_as_they_lie(device, M, N, K, out_dtype):
    """(K, N) weights that the narrow tiles turn inside LDS: columns and rows that end inside a tile, fewer K steps than waves.
    The same tile asked for by name works on the (N, K) copy: the same products added in the same order, so the bits agree."""
    g = _g(M * 3 + N + K)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.3)
    kn = b.view(torch.uint8).t().contiguous().view(FP8).to(device)
    kw = dict(scale_a=0.25, scale_b=0.5, out_dtype=out_dtype)
    got = matmul(a.to(device), kn, **kw)
    cfg = _lib.last_config()
    assert cfg["KERNEL_NAME"] == "tiled" and cfg["BLOCK_N"] <= 64
    kc = {"KERNEL": "tiled", "BLOCK_M": cfg["BLOCK_M"], "BLOCK_N": cfg["BLOCK_N"]}
    want = matmul(a.to(device), kn, kernel_configs=kc, **kw)
    assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))
    if out_dtype is torch.bfloat16:
        check(got, R.ref_gemm_per_tensor(a, b, 0.25, 0.5, trans_b=True))


@pytest.mark.parametrize("M,N,K", [(1, 8208, 1280), (17, 9232, 1408), (50, 1040, 5120), (33, 12304, 1280), (60, 20496, 1280), (70, 6160, 1664), (129, 6160, 1280),
                                   (200, 8208, 2176), (300, 4112, 1280), (256, 28688, 1280), (500, 4112, 4096), (1025, 1040, 1280)])
def test_kn_weights_on_ring_tiles(device, M, N, K):
    """(K, N) weights that the ring tiles turn inside LDS, over every tile they choose from: rows and columns that end inside a tile,
    split K, alpha and beta.  The same tile and split asked for by name works on the (N, K) copy: the bits agree."""
    g = _g(M * 5 + N + K)
    a, b = fp8_randn((M, K), g), fp8_randn((N, K), g, 0.3)
    ad, kn = a.to(device), b.view(torch.uint8).t().contiguous().view(FP8).to(device)
    for out_dtype in (torch.bfloat16, torch.float32, FP8):
        kw = dict(scale_a=0.25, scale_b=0.125, out_dtype=out_dtype)
        got = matmul(ad, kn, **kw)
        cfg = used("tiled")
        assert cfg["WAVES"] == 8 or M > 1024, cfg
        kc = {"KERNEL": "tiled", "BLOCK_M": cfg["BLOCK_M"], "BLOCK_N": cfg["BLOCK_N"], "SPLIT_K": cfg["SPLIT_K"], "WAVES": 8}
        want = matmul(ad, kn, kernel_configs=kc, **kw)
        assert torch.equal(got.view(torch.uint8), want.view(torch.uint8)), cfg
    check(matmul(ad, kn, scale_a=0.25, scale_b=0.125, out_dtype=torch.bfloat16), R.ref_gemm_per_tensor(a, b, 0.25, 0.125, trans_b=True), what=str(cfg))
    c0 = torch.randn(M, N, generator=g)
    c, c2 = c0.to(device), c0.to(device)
    one = torch.ones(1, device=device)
    _lib.fp8_gemm(c, ad, kn, one, None, False, False, 1.5, 0.5)
    _lib.fp8_gemm(c2, ad, kn, one, None, False, False, 1.5, 0.5, kc)
    assert torch.equal(c, c2)


@pytest.mark.parametrize("rows", [8191, 8192, 8195])
def test_quantizer_with_one_and_four_groups_per_lane(device, rows):
    """67 M elements are the line between the quantizer's two forms; a tensor on either side of it, and one whose last workgroup
    is not full, against the same rows in pieces small enough for the other form."""
    from tilegym_amd.quant import act_quant

    x = torch.randn(rows, 8192, generator=torch.Generator(device=device).manual_seed(rows), device=device).to(torch.bfloat16)
    x[3, 128:256] = 0
    q, s = act_quant(x, 128)
    for lo in range(0, rows, 4096):
        qp, sp = act_quant(x[lo:lo + 4096], 128)
        assert torch.equal(q[lo:lo + 4096].view(torch.uint8), qp.view(torch.uint8)) and torch.equal(s[lo:lo + 4096], sp)


@pytest.mark.parametrize("T,H,I,E,k,dtype,skew", [
    (1, 640, 384, 40, 8, torch.bfloat16, 0),      # sum form; K tails of one and of three steps (5 and 3 K steps)
    (2, 512, 1408, 64, 6, torch.float16, 0),      # sum form, two tokens
    (3, 128, 128, 3, 2, torch.bfloat16, 0),       # one K step; more slots than experts
    (16, 1152, 256, 64, 4, torch.float16, 0),     # 16 rows held, row-per-slot form
    (40, 256, 640, 33, 5, torch.bfloat16, 0),     # an expert count over one mask word
    (44, 256, 256, 40, 6, torch.bfloat16, 44),    # every token also to one expert: more rows than are held, several passes
    (75, 384, 384, 64, 6, torch.bfloat16, 0),     # seven rows per expert on average
    (5, 7168, 256, 16, 8, torch.bfloat16, 0),     # a long K: more than one batch of activations, fewer rows held
])
def test_decoding_moe_layer_gives_the_bits_of_the_row_tiled_layer(device, T, H, I, E, k, dtype, skew):
    """The layer on the weight-streaming kernels (few rows per expert) against the row-tiled kernels called one by one: K blocks
    are added in the same order with the same fused multiply-adds and both quantizations round alike, so the bits agree;
    first call, repeated call, ids as int32 and int64."""
    from tilegym_amd.ops import fused_moe, moe_interface

    g = _g(1000 * T + H + E)
    hidden = torch.randn(T, H, generator=g).to(dtype).to(device)
    hidden[0, :128] = 0                             # (an all-zero group: scale 1)
    w1q, w1s = R.quantize_weight_128x128(torch.randn(E * 2 * I, H, generator=g) * 0.1)
    w2q, w2s = R.quantize_weight_128x128(torch.randn(E * H, I, generator=g) * 0.1)
    w1q, w1s = w1q.reshape(E, 2 * I, H).to(device), w1s.reshape(E, 2 * I // 128, H // 128).to(device)
    w2q, w2s = w2q.reshape(E, H, I).to(device), w2s.reshape(E, H // 128, I // 128).to(device)
    ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)])
    if skew:
        ids = torch.where(ids == E - 1, ids[:, :1], ids)
        ids[:skew, 0] = E - 1
    ids = ids.to(device)
    tw = torch.softmax(torch.randn(T, k, generator=g), dim=-1).to(device)
    try:
        moe_interface.USE_ONE_CALL_LAYER = False
        want = fused_moe(hidden, w1q, w2q, tw, ids, w1_scale=w1s, w2_scale=w2s)
    finally:
        moe_interface.USE_ONE_CALL_LAYER = True
    for again in (ids, ids.to(torch.int32), ids):
        _lib.workspace_for(hidden.device, 1 << 20).fill_(0xAB)
        got = fused_moe(hidden, w1q, w2q, tw, again, w1_scale=w1s, w2_scale=w2s)
        assert _lib.last_config()["KERNEL_NAME"] == "stream"
        assert torch.isfinite(got.float()).all() and torch.equal(got, want)


def _device_moe_layer(device, T, H, I, E, k, seed):
    """An FP8 MoE layer made on the device: activations, weights with their scales, routing (even)."""
    g = torch.Generator(device=device).manual_seed(seed)
    w1 = (torch.randn(E, 2 * I, H, generator=g, device=device, dtype=torch.float16) * 16).to(FP8)
    w2 = (torch.randn(E, H, I, generator=g, device=device, dtype=torch.float16) * 16).to(FP8)
    s1 = torch.rand(E, 2 * I // 128, H // 128, generator=g, device=device) * 4e-3 + 1e-3
    s2 = torch.rand(E, H // 128, I // 128, generator=g, device=device) * 4e-3 + 1e-3
    x = torch.randn(T, H, generator=g, device=device).to(torch.bfloat16)
    tw, ids = torch.topk(torch.softmax(torch.randn(T, E, generator=g, device=device), dim=-1), k, dim=-1)
    return x, w1, w2, s1, s2, tw, ids


def _both_forms(x, w1, w2, s1, s2, tw, ids):
    """(the layer as one call, the same on the row-tiled kernels called one by one, the kernel that the one call chose)"""
    from tilegym_amd.ops import fused_moe, moe_interface

    _lib.workspace_for(x.device, 1 << 20).fill_(0xFF)
    got = fused_moe(x, w1, w2, tw, ids, w1_scale=s1, w2_scale=s2)
    kernel = _lib.last_config()["KERNEL_NAME"]
    try:
        moe_interface.USE_ONE_CALL_LAYER = False
        want = fused_moe(x, w1, w2, tw, ids, w1_scale=s1, w2_scale=s2)
    finally:
        moe_interface.USE_ONE_CALL_LAYER = True
    return got, want, kernel


@pytest.mark.parametrize("T,H,I,E,k", [(12, 4864, 384, 16, 2), (33, 4736, 384, 64, 8), (75, 4608, 768, 64, 6), (11, 4096, 6400, 16, 2),
                                       (75, 2048, 1408, 64, 6), (76, 2048, 1408, 64, 6)])
def test_decoding_moe_layer_where_its_lds_is_full(device, T, H, I, E, k):
    """Layers whose decoding form asks for (almost) all of a compute unit's LDS, and both sides of the line between the forms."""
    layer = _device_moe_layer(device, T, H, I, E, k, seed=T)
    got, want, kernel = _both_forms(*layer)
    lds = _lib.load().tg_diag_moe_lds_bytes(T, k, E, H, I)
    assert lds <= 160 * 1024 and kernel == ("stream" if lds else "tiled")
    assert torch.isfinite(got.float()).all() and torch.equal(got, want)


@pytest.mark.parametrize("T,H,I,k", [(1, 640, 128, 1), (1, 384, 640, 2), (16, 640, 128, 1), (16, 384, 640, 2)])
def test_decoding_moe_layer_with_infinities_in_the_last_group(device, T, H, I, k):
    """Rows whose last quantization group holds an infinity or a NaN, and a K that is no multiple of the 512 bytes of a piece: K steps
    past the end add nothing, whatever the scale in front of them is, so the layer gives what the row-tiled kernels give."""
    x, w1, w2, s1, s2, tw, ids = _device_moe_layer(device, T, H, I, 64, k, seed=H + T)
    x[0, -1], x[T // 2, -3] = float("inf"), float("-inf")
    x[T - 1, -128] = float("nan")
    got, want, kernel = _both_forms(x, w1, w2, s1, s2, tw, ids)
    assert kernel == "stream" and torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.nan_to_num(nan=0.0), want.nan_to_num(nan=0.0))
    if I == 128:
        assert got[0].isinf().any()


@pytest.mark.parametrize("T,E,k,routing", [(1, 64, 6, "duplicates"), (5, 200, 8, "duplicates"), (40, 64, 6, "same"), (70, 64, 6, "same"),
                                           (100, 130, 6, "one"), (100, 130, 6, "far"), (60, 200, 4, "half"), (256, 512, 4, "far"),
                                           (90, 33, 2, "half")])
def test_decoding_moe_layer_with_more_rows_than_are_held(device, T, E, k, routing):
    """Experts with more rows than a workgroup holds at a time, streamed once per pass: every token to the same experts, one or
    several experts in every token (in the first and in the last of the mask's words), half of the batch alike, an id twice in a
    token."""
    x, w1, w2, s1, s2, tw, _ = _device_moe_layer(device, T, 384, 256, E, k, seed=T + E)
    p = torch.rand(T, E, generator=torch.Generator(device=device).manual_seed(E), device=device)
    if routing == "same":
        p[:] = p[0].clone()
    elif routing == "half":
        p[T // 2:] = p[0].clone()
    elif routing == "one":
        p[:, 0] = 2.0
    elif routing == "far":
        p[:, E - 1], p[:, 65], p[T // 2:, 66] = 4.0, 3.0, 2.0
    ids = p.topk(k, dim=1).indices
    if routing == "duplicates":
        ids[:] = ids[:, :1].clone()
    got, want, kernel = _both_forms(x, w1, w2, s1, s2, tw, ids)
    assert kernel == "stream" and torch.equal(got, want)


@pytest.mark.parametrize("T", [1, 16])
def test_decoding_moe_layer_with_a_misaligned_weight(device, T):
    """A w2 off a 16-byte boundary is taken (on the row-tiled form), any other such operand refused as it is there."""
    from tilegym_amd.ops import fused_moe

    def shifted(t):
        raw = torch.empty(t.numel() * t.element_size() + 16, dtype=torch.uint8, device=device)[8:-8]
        return raw.copy_(t.view(torch.uint8).reshape(-1)).view(t.dtype).view(t.shape)

    x, w1, w2, s1, s2, tw, ids = _device_moe_layer(device, T, 256, 384, 16, 2, seed=T)
    want = fused_moe(x, w1, w2, tw, ids, w1_scale=s1, w2_scale=s2)
    assert _lib.last_config()["KERNEL_NAME"] == "stream"
    got = fused_moe(x, w1, shifted(w2), tw, ids, w1_scale=s1, w2_scale=s2)
    assert (got.float() - want.float()).norm() <= 2.0 ** -7 * want.float().norm()   # (bf16 results of sums in another order)
    for bad in ((shifted(x), w1), (x, shifted(w1))):
        with pytest.raises(_lib.TileGymHipError, match="16-byte"):
            fused_moe(*bad, w2, tw, ids, w1_scale=s1, w2_scale=s2)


@pytest.mark.parametrize("T,H,I,E,k", [(1, 256, 384, 64, 6), (16, 384, 256, 64, 6), (400, 256, 256, 16, 3), (9, 256, 256, 64, 1), (200, 256, 256, 4, 1)])
def test_moe_slots_without_an_expert_add_nothing(device, T, H, I, E, k):
    """Ids outside [0, E) in every form of the layer (one launch with the sum, decoding, row-tiled, call by call), whatever the
    scratch memory and the slot's weight hold: what the same slots give with an expert of theirs and a weight of zero."""
    x, w1, w2, s1, s2, tw, ids = _device_moe_layer(device, T, H, I, E, k, seed=T + k)
    out_of = torch.rand(T, k, generator=torch.Generator(device=device).manual_seed(T), device=device) < 0.3
    out_of[0, 0] = True
    want = _both_forms(x, w1, w2, s1, s2, tw.masked_fill(out_of, 0.0), ids)[0]
    assert torch.isfinite(want.float()).all()
    for outside in (-1, E, E + 7):
        torch.full((T, k, H), float("nan"), dtype=x.dtype, device=device)  # (freed: what the next allocation may find)
        for dtype in (torch.int32, torch.int64):
            for got in _both_forms(x, w1, w2, s1, s2, tw.masked_fill(out_of, float("inf")), ids.masked_fill(out_of, outside).to(dtype))[:2]:
                assert torch.equal(got, want)


def test_recorded_schedule_is_used_when_no_kernel_configs_are_given(device, tmp_path):
    """A table written by tilegym_amd.tune (here: by hand, and by tune_shape on a small shape) decides the schedule of calls
    that bring no kernel_configs; explicit kernel_configs still win; unloading the table restores the automatic choice."""
    from tilegym_amd import tune

    g = _g(321)
    M, N, K = 8, 4096, 4096
    a, b = fp8_randn((M, K), g).to(device), fp8_randn((N, K), g, 0.02).to(device)
    sa, sb = torch.tensor([0.5], device=device), torch.tensor([0.25], device=device)
    c = torch.empty(M, N, dtype=torch.bfloat16, device=device)
    ref = ((a.float() * 0.5) @ (b.float() * 0.25).t()).to(torch.bfloat16).cpu()
    _lib.fp8_gemm(c, a, b, sa, sb)
    auto = _lib.last_config()
    assert (auto["ROW_GROUPS"], auto["SPLIT_K"]) == (1, 1), auto       # the narrow form
    path = str(tmp_path / "tune.json")
    tune.write_table([{"M": M, "N": N, "K": K, "block_scaled": False, "kernel_configs": {"KERNEL": "stream", "ROW_GROUPS": 4, "SPLIT_K": 2},
                       "us": 0.0, "auto_us": 0.0, "auto_schedule": {}}], path)
    try:
        _lib.load_tune_table(path)
        for _ in range(2):                                             # the table applies to every call
            _lib.fp8_gemm(c, a, b, sa, sb)
            got = _lib.last_config()
            assert (got["KERNEL_NAME"], got["ROW_GROUPS"], got["SPLIT_K"]) == ("stream", 4, 2), got
            check(c, ref, what="recorded schedule")
        _lib.fp8_gemm(c, a, b, sa, sb, kernel_configs={"KERNEL": "stream", "WAVES": 8})
        assert _lib.last_config()["WAVES"] == 8
    finally:
        _lib.load_tune_table("")
    _lib.fp8_gemm(c, a, b, sa, sb)
    assert _lib.last_config() == auto
    entry = tune.tune_shape(8, 1024, 2048, False)
    assert entry["us"] <= entry["auto_us"] and entry["auto_schedule"]["KERNEL_NAME"] == "stream"
    assert entry["kernel_configs"] == {} or entry["us"] <= 0.97 * entry["auto_us"]


def test_prepared_call_cache_follows_the_tensors(device):
    """The binding describes a call's tensors on every call.  The same objects again: same result; an operand given new storage, a
    resized output, fresh outputs whose Python ids repeat, a dead weight whose id is taken over by another tensor: never a stale
    pointer."""
    from tilegym_amd import _lib

    g = _g(123)
    M, N, K = 8, 512, 1024
    a1, a2 = fp8_randn((M, K), g).to(device), fp8_randn((M, K), g).to(device)
    b1, b2 = fp8_randn((N, K), g, 0.02).to(device), fp8_randn((N, K), g, 0.02).to(device)
    sa, sb = torch.tensor([0.5], device=device), torch.tensor([0.25], device=device)

    def ref(a, b):
        return ((a.float() * 0.5) @ (b.float() * 0.25).t()).to(torch.bfloat16)

    c = torch.empty(M, N, dtype=torch.bfloat16, device=device)
    for _ in range(3):
        _lib.fp8_gemm(c, a1, b1, sa, sb)
        check(c, ref(a1, b1).cpu(), what="same objects")
    a = a1.clone()
    _lib.fp8_gemm(c, a, b1, sa, sb)
    _lib.fp8_gemm(c, a, b1, sa, sb)
    a.data = a2.clone()                      # same object, new storage
    _lib.fp8_gemm(c, a, b1, sa, sb)
    check(c, ref(a2, b1).cpu(), what="operand with new storage")
    for i in range(6):                       # fresh outputs: ids repeat, every one must be written
        out = torch.zeros(M, N, dtype=torch.bfloat16, device=device)
        _lib.fp8_gemm(out, a1, b2 if i % 2 else b1, sa, sb)
        check(out, ref(a1, b2 if i % 2 else b1).cpu(), what=f"fresh output {i}")
        del out
    w = b1.clone()
    _lib.fp8_gemm(c, a1, w, sa, sb)
    del w
    w = b2.clone()                           # likely the dead weight's id and address
    _lib.fp8_gemm(c, a1, w, sa, sb)
    check(c, ref(a1, b2).cpu(), what="weight object replaced")
    c2 = torch.empty(2 * M, N, dtype=torch.bfloat16, device=device)
    a_big = torch.cat([a1, a2])
    _lib.fp8_gemm(c2, a_big, b1, sa, sb)
    check(c2, ref(a_big, b1).cpu(), what="other M")
    _lib.release_call_caches()
    _lib.fp8_gemm(c, a1, b1, sa, sb)
    check(c, ref(a1, b1).cpu(), what="after release_call_caches")


# ----------------------------------------------------------------------------- group_gemm (list form)
def test_group_gemm_list_form(device):
    g = _g(12)
    shapes = [(64, 128, 256), (130, 72, 128), (8, 264, 512)]
    As = [fp8_randn((m, k), g) for m, n, k in shapes]
    Bs = [fp8_randn((k, n), g) for m, n, k in shapes]
    outs = group_gemm([x.to(device) for x in As], [x.to(device) for x in Bs], out_dtype=torch.bfloat16)
    refs = R.ref_group_gemm(As, Bs, out_dtype=torch.bfloat16)
    for o, r in zip(outs, refs):
        check(o, r)
    Bt = [b.view(torch.uint8).t().contiguous().view(FP8) for b in Bs]
    outs_t = group_gemm([x.to(device) for x in As], [x.to(device) for x in Bt], transpose_b=True, out_dtype=torch.bfloat16,
                        scales_a=[0.5] * 3, scales_b=[torch.tensor([2.0], device=device)] * 3)
    for o, r in zip(outs_t, refs):
        check(o, r)
    default = group_gemm([As[0].to(device)], [Bs[0].to(device)])
    assert default[0].dtype == FP8


@pytest.mark.parametrize("tile", [None, (64, 128), (128, 128), (256, 256)])
def test_group_gemm_single_launch(device, tile):
    """(N,K) weights with K % 128 == 0: the whole list is one launch of the tiled kernel; ragged M and N,
    an empty problem, more problems than one launch carries (40), per-problem scales."""
    g = _g(13)
    shapes = [(64, 128, 256), (130, 72, 128), (8, 264, 512), (0, 128, 128), (300, 520, 384)] + [(17 + i, 136, 128) for i in range(44)]
    As = [fp8_randn((m, k), g) for m, n, k in shapes]
    Bs = [fp8_randn((n, k), g, 0.1) for m, n, k in shapes]
    sa = [0.25 + 0.01 * i for i in range(len(shapes))]
    sb = [torch.tensor([1.0 + 0.5 * (i % 3)]) for i in range(len(shapes))]
    kc = None if tile is None else {"BLOCK_M": tile[0], "BLOCK_N": tile[1]}
    outs = group_gemm([x.to(device) for x in As], [x.to(device) for x in Bs], transpose_b=True, out_dtype=torch.bfloat16,
                      scales_a=sa, scales_b=[t.to(device) for t in sb], kernel_configs=kc)
    cfg = used("tiled")
    if tile is not None:
        assert (cfg["BLOCK_M"], cfg["BLOCK_N"]) == tile
    for i, (A, B, o) in enumerate(zip(As, Bs, outs)):
        assert o.shape == (A.shape[0], B.shape[0])
        if A.shape[0]:
            check(o, R.ref_gemm_per_tensor(A, B, torch.tensor([sa[i]]), sb[i], trans_b=True), what=f"problem {i}")


# ----------------------------------------------------------------------------- BASELINE configs at full size
def _rows_subset(M, count, seed=0):
    if M <= count:
        return torch.arange(M)
    idx = torch.randperm(M, generator=_g(seed))[:count].sort().values
    idx[0], idx[-1] = 0, M - 1
    return idx


def _rows_stratified(M, per_tile, seed=0, tile=256):
    """`per_tile` rows from every `tile`-row tile of an M-row problem; over the tiles the rows walk through all sixteen
    16-row group slots of a tile (the unit a wave owns), at a random offset inside the slot; first and last row included."""
    g = _g(seed)
    rows = []
    for t in range(-(-M // tile)):
        for j in range(per_tile):
            slot = (t * per_tile + j) % (tile // 16)
            r = t * tile + slot * 16 + int(torch.randint(0, 16, (1,), generator=g))
            rows.append(min(r, M - 1))
    rows += [0, M - 1]
    return torch.tensor(sorted(set(rows)))


def test_ops_through_torchs_dispatcher(device):
    """torch.ops.tilegym_hip.*: same bits as the direct calls; traceable by torch.compile (aot_eager: the graph is captured
    through the fake implementations and run through the dispatcher)."""
    g = _g(8)
    M, N, K = 40, 520, 1024
    a, b = fp8_randn((M, K), g).to(device), fp8_randn((N, K), g, 0.02).to(device)
    sa, sb = torch.tensor([0.02], device=device), torch.tensor([0.01], device=device)
    direct = matmul(a, b, trans_b=True, scale_a=sa, scale_b=sb, out_dtype=torch.bfloat16)
    via = torch.ops.tilegym_hip.fp8_gemm(a, b, sa, sb, False, True, 1.0, torch.bfloat16)
    assert torch.equal(direct, via)
    c = torch.ones(M, N, dtype=torch.bfloat16, device=device)
    torch.ops.tilegym_hip.fp8_gemm_out(c, a, b, sa, sb, False, True, 1.0, 1.0)
    expect = gemm_alpha_beta(a, b, torch.ones(M, N, dtype=torch.bfloat16, device=device), alpha=0.02 * 0.01, beta=1.0)
    check(c, expect.cpu(), what="fp8_gemm_out, beta = 1")

    @torch.compile(backend="aot_eager", fullgraph=True)
    def f(a, b, sa, sb):
        return torch.ops.tilegym_hip.fp8_gemm(a, b, sa, sb, False, True, 1.0, torch.bfloat16).float() * 2

    assert torch.equal(f(a, b, sa, sb), direct.float() * 2)
    ra, rb, ras, rbs, ptr = _ragged_inputs([100, 0, 300], 256, 512, 3)
    dev = [t.to(device) for t in (ra, rb, ras, rbs, ptr)]
    assert torch.equal(torch.ops.tilegym_hip.fp8_ragged_gemm(*dev, torch.bfloat16), ragged_block_scaled_bmm(*dev, 300))
    x = torch.randn(33, 384, generator=g).to(torch.bfloat16).to(device)
    q, s = torch.ops.tilegym_hip.fp8_quant_1x128(x)
    q2, s2 = _lib.fp8_quant_1x128(x, 0.0, False)
    assert torch.equal(q.view(torch.uint8), q2.view(torch.uint8)) and torch.equal(s, s2)
    from tilegym_amd.ops import fused_moe
    T, H, I, E, k = 9, 256, 128, 4, 2
    hidden = (torch.randn(T, H, generator=g) * 0.5).to(torch.bfloat16).to(device)
    w1q, w1s = R.quantize_weight_128x128(torch.randn(E * 2 * I, H, generator=g) * 0.1)
    w2q, w2s = R.quantize_weight_128x128(torch.randn(E * H, I, generator=g) * 0.1)
    w1q, w1s = w1q.reshape(E, 2 * I, H).to(device), w1s.reshape(E, 2 * I // 128, H // 128).to(device)
    w2q, w2s = w2q.reshape(E, H, I).to(device), w2s.reshape(E, H // 128, 1).to(device)
    ids, tw = torch.randint(0, E, (T, k), generator=g).to(device), torch.softmax(torch.randn(T, k, generator=g), dim=-1).to(device)
    assert torch.equal(torch.ops.tilegym_hip.fp8_fused_moe(hidden, w1q, w2q, w1s, w2s, tw, ids),
                       fused_moe(hidden, w1q, w2q, tw, ids, w1_scale=w1s, w2_scale=w2s))


def test_config1_full(device):
    for trans_b in (True, False):
        case = W.config1(trans_b=trans_b)
        ref = R.ref_gemm_per_tensor(case.a, case.b, case.scale_a, case.scale_b, trans_b=trans_b)
        d = case.to(device)
        out = matmul(d.a, d.b, trans_b=trans_b, scale_a=d.scale_a, scale_b=d.scale_b, out_dtype=torch.bfloat16)
        assert _lib.last_config()["KERNEL_NAME"] == "tiled"
        check(out, ref, what=f"config 1 trans_b={trans_b}")


@pytest.mark.parametrize("proj", list(W.LLAMA_SHAPES))
def test_config2_llama_decode_full(device, proj):
    N, K = W.LLAMA_SHAPES[proj]
    big = W.llama_decode_case(64, proj)
    bd = big.b.to(device)
    bref = R.fp8_to_f32(big.b) * big.scale_b
    for M in W.DECODE_M:
        a = big.a[:M].contiguous()
        ref = ((R.fp8_to_f32(a) * big.scale_a) @ bref.t()).to(torch.bfloat16)
        out = matmul(a.to(device), bd, trans_b=True, scale_a=big.scale_a.to(device), scale_b=big.scale_b.to(device), out_dtype=torch.bfloat16)
        used("stream" if M <= 16 else "tiled")
        check(out, ref, what=f"config 2 {proj} M={M}")


def check_all_rows(out, ref_rows, M, what, rows_per_pass=2048):
    """Every row of `out` (on the device) against the oracle, `rows_per_pass` rows at a time: ref_rows(lo, hi) returns the
    oracle's rows lo .. hi-1.  Bounds the host memory of a full-size comparison."""
    for lo in range(0, M, rows_per_pass):
        hi = min(M, lo + rows_per_pass)
        check(out[lo:hi], ref_rows(lo, hi), what=f"{what} rows {lo}..{hi - 1}")


@pytest.mark.parametrize("proj", list(W.LLAMA_SHAPES))
def test_config3_llama_prefill_sampled_rows(device, proj):
    """Full-size launch, and the whole output against the oracle: every tile, wave and row-group slot of the persistent
    kernel's walk (the name is from when rows were sampled).  Plus linearity across the whole output."""
    case = W.llama_prefill_case(proj)
    d = case.to(device)
    out = matmul(d.a, d.b, trans_b=True, scale_a=d.scale_a, scale_b=d.scale_b, out_dtype=torch.bfloat16)
    cfg = used("tiled")
    assert (cfg["BLOCK_M"], cfg["BLOCK_N"]) == (256, 256)
    b_deq_t = (R.fp8_to_f32(case.b) * case.scale_b).t().contiguous()
    check_all_rows(out, lambda lo, hi: ((R.fp8_to_f32(case.a[lo:hi]) * case.scale_a) @ b_deq_t).to(torch.bfloat16), case.M,
                   f"config 3 {proj}")
    del b_deq_t
    assert torch.isfinite(out.float()).all()
    # doubling a scale doubles every element exactly (bf16, power of two)
    out2 = matmul(d.a, d.b, trans_b=True, scale_a=d.scale_a * 2, scale_b=d.scale_b, out_dtype=torch.bfloat16)
    assert torch.equal(out2.float(), out.float() * 2)


@pytest.mark.parametrize("N,K", W.BLOCK_SCALED_SHAPES)
def test_config4_block_scaled_full(device, N, K):
    big = W.block_scaled_case(4096, N, K)
    d = big.to(device)
    out = w8a8_block_fp8_matmul(d.a, d.b, d.scale_a, d.scale_b, None, torch.bfloat16)
    used("tiled")
    # the whole output (the weights are dequantized once)
    b_deq_t = (R.fp8_to_f32(big.b).view(N // 128, 128, K // 128, 128) * big.scale_b[:, None, :, None]).view(N, K).t().contiguous()
    check_all_rows(out, lambda lo, hi: ((R.fp8_to_f32(big.a[lo:hi]).view(hi - lo, K // 128, 128) * big.scale_a[lo:hi, :, None])
                                        .view(hi - lo, K) @ b_deq_t).to(torch.bfloat16), 4096, f"config 4 M=4096 {N}x{K}", 1024)
    del b_deq_t
    rows = _rows_stratified(4096, 1)  # and the oracle function itself on a few rows (it dequantizes the same way)
    ref = R.ref_w8a8_block_fp8_matmul(big.a[rows], big.b, big.scale_a[rows], big.scale_b, None, torch.bfloat16)
    check(out[rows.to(device)], ref, what=f"config 4 M=4096 {N}x{K} (oracle function)")
    out16 = w8a8_block_fp8_matmul(d.a[:16].contiguous(), d.b, d.scale_a[:16].contiguous(), d.scale_b, None, torch.bfloat16)
    used("stream")
    ref16 = R.ref_w8a8_block_fp8_matmul(big.a[:16], big.b, big.scale_a[:16], big.scale_b, None, torch.bfloat16)
    check(out16, ref16, what=f"config 4 M=16 {N}x{K}")


@pytest.mark.parametrize("which", ["gate_up", "down"])
def test_config5_moe_grouped_full(device, which):
    case = _moe_base(which)
    d = case.to(device)
    sizes = (case.m_indptr[1:] - case.m_indptr[:-1])
    assert int(case.m_indptr[-1]) == 4096 * 6 and sizes.min() != sizes.max()  # uneven experts
    out = ragged_block_scaled_bmm(d.a, d.b, d.a_scale, d.b_scale, d.m_indptr, int(sizes.max()))
    used("tiled")
    # per-expert reference GEMMs, all 64 experts
    for e in range(case.b.shape[0]):
        lo, hi = int(case.m_indptr[e]), int(case.m_indptr[e + 1])
        ref = R.ref_w8a8_block_fp8_matmul(case.a[lo:hi], case.b[e], case.a_scale[lo:hi], case.b_scale[e], None, torch.bfloat16)
        check(out[lo:hi], ref, what=f"config 5 {which} expert {e}")
    assert torch.isfinite(out.float()).all()
    # the token-gather form of the same GEMM gives the same numbers slot by slot
    if which == "gate_up":
        ids, order, k = case.extra["topk_ids"], case.extra["order"], case.extra["top_k"]
        T = ids.shape[0]
        x_rows = torch.empty(T, case.a.shape[1], dtype=torch.uint8)
        x_rows[order // k] = case.a.view(torch.uint8)
        xs = torch.empty(T, case.a_scale.shape[1])
        xs[order // k] = case.a_scale
        sorted_ids, expert_ids, post, _, _ = moe_align_block_size(ids.to(device), 128, 64)
        C = torch.zeros(T, k, case.b.shape[1], dtype=torch.bfloat16, device=device)
        invoke_fused_moe_kernel(x_rows.view(FP8).to(device), d.b, C, xs.to(device), d.b_scale, None, ids.to(device),
                                sorted_ids, expert_ids, post, False, k, {"BLOCK_SIZE_M": 128})
        used("tiled")
        gathered = C.view(T * k, -1)[order.to(device)]
        assert torch.equal(gathered, out)
