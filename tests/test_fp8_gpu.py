"""fp8 paths on the GPU: per-row e4m3 activation quantization (bit-exact vs the
oracle) and the W8A8 GEMM (tolerance vs the oracle's exact-product reference),
plus W8A16 at the benchmark config-4 shapes. The W8A8 mode has no reference
counterpart: its parity is pinned only by the oracle restatement."""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from pulsarlm_amd import ops
from tests._util import TDT, assert_close, fp8_case, mfma_plan, to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("m,k", [(1, 128), (16, 5120), (37, 1040), (3, 1044), (2, 40000), (600, 17408), (520, 96)])
def test_quantize_rows_bit_exact(m, k, dtype):
    """Rows of 8-value chunks take the vectorised kernel (1024 threads a row below 512 rows,
    256 above; K = 40000 and 17408 also exercise the chunks read twice); K = 1044 (not a
    multiple of 8) takes the scalar kernel."""
    rng = np.random.default_rng(m + k)
    x = O.round_to(rng.standard_normal((m, k)).astype(np.float32) * np.exp2(rng.integers(-6, 6, (m, 1))), dtype)
    x[0, :3] = 0.0
    codes, scale = ops.quantize_rows_e4m3_cuda(to_dev(x, TDT[dtype]))
    ref_codes, ref_scale = O.quantize_per_token_e4m3(x)
    assert np.array_equal(scale.cpu().numpy(), ref_scale)
    assert np.array_equal(codes.cpu().numpy(), ref_codes)


def _fp8_weights(n, k, seed):
    rng = np.random.default_rng(seed)
    w = O.bf16_round(rng.standard_normal((n, k)).astype(np.float32) * 0.02)
    codes, scale = O.fp8_block_quantize(w, 128, 128)
    wt, st = ops.repack_fp8_marlin_cuda(to_dev(codes).view(torch.float8_e4m3fn), to_dev(scale), 128, 128)
    return codes, scale, wt, st


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("m", [1, 5, 16, 17, 300])
def test_w8a8_matches_oracle(m, dtype):
    n, k = 520, 1024
    codes, scale, wt, st = _fp8_weights(n, k, seed=m)
    x = O.round_to(np.random.default_rng(m).standard_normal((m, k)).astype(np.float32), dtype)
    y = ops.gemm_fp8_w8a8_cuda(to_dev(x, TDT[dtype]), wt, st, n, 128, 128)
    xc, xs = O.quantize_per_token_e4m3(x)
    ref = O.gemm_w8a8_ref(xc, xs, codes, scale, 128, 128, dtype=None)
    assert_close(y, ref, f"w8a8 m={m}")


@pytest.mark.parametrize("shape", [(5120, 7168), (5120, 5120), (5120, 34816), (17408, 5120)])
@pytest.mark.parametrize("m", [1, 16, 2048])
def test_config4_qwen3_27b_shapes(shape, m):
    """benchmark config 4: fp8 128x128 block weights, W8A16 (bf16 x) and W8A8."""
    k, n = shape
    codes, scale, wt, st = _fp8_weights(n, k, seed=k + n)
    x = O.bf16_round(np.random.default_rng(m).standard_normal((m, k)).astype(np.float32))
    xd = to_dev(x, torch.bfloat16)
    w_deq = O.dequant_fp8(codes, scale, 128, 128)
    rows = slice(0, min(m, 64))  # the CPU reference on a row sample at M=2048
    y = ops.gemm_fp8_marlin_cuda(xd, wt, st, n, 128, 128)
    assert_close(y[rows], O.gemm_ref(x[rows], w_deq, None), f"w8a16 {shape} m={m}")
    y8 = ops.gemm_fp8_w8a8_cuda(xd, wt, st, n, 128, 128)
    xc, xs = O.quantize_per_token_e4m3(x[rows])
    assert_close(y8[rows], O.gemm_w8a8_ref(xc, xs, codes, scale, 128, 128, dtype=None), f"w8a8 {shape} m={m}")


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("m", [1, 4, 16, 17, 25, 32, 100, 300])
def test_w8a16_32x32_blocks(m, dtype):
    """The reference's model-level fp8 configuration (test_qwen3_5.cpp:691-696): 32 x 32
    quantization blocks, so block_n = 32 (one scale per two 16-column strips) and 32-wide
    scale groups (four per 128-wide K tile), through the decode and MFMA kernels."""
    n, k = 200, 416
    rng = np.random.default_rng(m)
    w = O.bf16_round(rng.standard_normal((n, k)).astype(np.float32) * 0.02)
    codes, scale = O.fp8_block_quantize(w, 32, 32)
    wt, st = ops.repack_fp8_marlin_cuda(to_dev(codes).view(torch.float8_e4m3fn), to_dev(scale), 32, 32)
    x = O.round_to(rng.standard_normal((m, k)).astype(np.float32), dtype)
    y = ops.gemm_fp8_marlin_cuda(to_dev(x, TDT[dtype]), wt, st, n, 32, 32)
    assert_close(y, O.gemm_ref(x, O.dequant_fp8(codes, scale, 32, 32, dtype), None), f"fp8 32x32 m={m}")


def test_w8a8_rejects_small_groups():
    codes = np.zeros((64, 256), np.uint8)
    wt, st = ops.repack_fp8_marlin_cuda(to_dev(codes).view(torch.float8_e4m3fn),
                                        torch.ones((1, 4), device="cuda"), 128, 64)
    with pytest.raises(RuntimeError, match="gemm_fp8_w8a8: group_size must be a multiple of 128"):
        ops.gemm_fp8_w8a8_cuda(torch.zeros((4, 256), dtype=torch.bfloat16, device="cuda"), wt, st, 64, 128, 64)


def test_w8a8_full_size_tall_tail():
    """W8A8 at the config-4 gate_up shape (M=2048, K=5120, N=34816): 1088 tall 256x256 tiles,
    whose last 64 (whole tile columns) run as 128-row halves in a second launch. Checked
    against a GPU fp32 reference of the same arithmetic: per-token e4m3 x times its row
    scale, e4m3 weights times their 128x128 block scale. The products are exact, so the
    only differences are fp32 summation order and the bf16 output rounding."""
    m, k, n = 2048, 5120, 34816
    plan = mfma_plan("w8a8", m, n, k)
    assert plan["tile"] == (256, 256) and plan["tail"] == 64 and plan["halves"], plan
    g = torch.Generator(device="cpu").manual_seed(91)
    codes = torch.randint(0, 256, (n, k), generator=g, dtype=torch.int32).to(torch.uint8)
    codes[(codes == 0x7F) | (codes == 0xFF)] = 0  # no NaN codes
    scale = (torch.rand((n // 128, k // 128), generator=g) * 0.1 + 0.01).float()
    x = torch.randn((m, k), generator=g).bfloat16().cuda()
    wt, st = ops.repack_fp8_marlin_cuda(codes.cuda().view(torch.float8_e4m3fn), scale.cuda(), 128, 128)
    y = ops.gemm_fp8_w8a8_cuda(x, wt, st, n, 128, 128)
    xq, sx = ops.quantize_rows_e4m3_cuda(x)
    xf = xq.view(torch.float8_e4m3fn).float() * sx[:, None]
    wf = codes.cuda().view(torch.float8_e4m3fn).float()
    wf *= scale.cuda().repeat_interleave(128, 0).repeat_interleave(128, 1)
    torch.backends.cuda.matmul.allow_tf32 = False
    ref = xf @ wf.T
    del wf
    err = (y.float() - ref).abs()
    assert bool((err <= 2.0**-8 * ref.abs() + 1e-3 * ref.abs().max()).all()), f"max err {err.max().item():.4g}"
    rel = (torch.linalg.vector_norm(y.float() - ref) / torch.linalg.vector_norm(ref)).item()
    assert rel <= 5e-3, rel


@pytest.mark.parametrize("shape", [(5120, 7168), (5120, 5120), (5120, 34816), (17408, 5120)])
def test_config4_w8a16_m2048_every_row(shape):
    """Config 4, W8A16 at M=2048, every row of every shape: the weights come from
    plm_dequant (bit-exact, pinned against the oracle) and the reference product is
    torch's fp32 matmul of the rounded operands on the GPU. gate_up runs the tall
    register-weight tiles with the K-split tail launch."""
    from tests.test_gemm_gpu import _check_full
    k, n = shape
    if n == 34816:
        plan = mfma_plan("fp8", 2048, n, k)
        assert plan["tile"] == (256, 256) and plan["tail"] == 64 and plan["tail_splits"] > 1, plan
    g = torch.Generator(device="cpu").manual_seed(k + n)
    codes = torch.randint(0, 256, (n, k), generator=g, dtype=torch.int32).to(torch.uint8)
    codes[(codes == 0x7F) | (codes == 0xFF)] = 0
    scale = (torch.rand((n // 128, k // 128), generator=g) * 0.02 + 1e-3).float()
    x = torch.randn((2048, k), generator=g).bfloat16().cuda()
    wt, st = ops.repack_fp8_marlin_cuda(codes.cuda().view(torch.float8_e4m3fn), scale.cuda(), 128, 128)
    wd = ops.dequant_marlin_cuda("fp8", wt, st, n, k, 128, 128)
    y = ops.gemm_fp8_marlin_cuda(x, wt, st, n, 128, 128)
    print(shape, "rel-L2", _check_full(y, x, wd))


_FUSED_SCALES = [(128, np.float32, "bf16"), (16, np.float32, "fp16"), (16, "bf16", "bf16")]
_FUSED_CASES = ([(m, 5120, 5120, *c) for m in (1, 2, 3, 4) for c in _FUSED_SCALES]
                + [(m, 4992, 1040, *c) for m in (1, 3) for c in _FUSED_SCALES]
                + [(m, 2048, 16384, 128, np.float32, "bf16") for m in (1, 4)]
                + [(3, 5120, 34816, 128, np.float32, "bf16"), (2, 1280, 520, 16, np.float32, "fp16"),
                   (2, 8192, 1040, 128, np.float32, "bf16")]
                + [(1, 17408, 5120, *c) for c in _FUSED_SCALES]
                + [(2, 17408, 4096, 128, np.float32, "fp16"), (3, 17408, 5120, 128, np.float32, "bf16")])


@pytest.mark.parametrize("m,k,n,block_n,sdt,dtype", _FUSED_CASES)
def test_w8a8_fused_quantizer_bit_exact(m, k, n, block_n, sdt, dtype, tuning_env):
    """W8A8 at M <= 4 quantizes x inside the GEMM kernel when each wavefront of the
    workgroup holds one to three K tiles: 16 wavefronts at K = 5120 and 4992 (40 and 39
    tiles; N = 34816 too, where the unfused kernel takes 8), 8 at N = 16384 (16 tiles).
    K = 1280 (10 tiles for 16 wavefronts) and K = 8192 (64) keep the separate quantizer
    launch. K = 17408 runs the split-K decode kernel: fused at M <= 2 (one workgroup over
    all of K, x staged in LDS), separate at M = 3 (x too large to stage). The fused path
    must give the two-launch result bit for bit (same codes, same row scales, same sums),
    which PLM_W8A8_UNFUSED selects, wherever both run the same wavefront count; both are
    also checked against the oracle. Row 1 is all
    zeros (scale 1e-12 / 448) and row 2 spans 2^-12 .. 2^4."""
    print(f"fused w8a8 m={m} k={k} n={n} block_n={block_n} scale={sdt} x={dtype}", flush=True)
    rng = np.random.default_rng(m * 7 + k + n)
    # Every e4m3 code but the NaNs; block scales in [0.01, 0.11), bf16-rounded for bf16.
    codes, scale = fp8_case(n, k, 128, block_n, seed=m + n)
    if sdt == "bf16":
        scale = O.bf16_round(scale)
        st_in = to_dev(scale, torch.bfloat16)
    else:
        st_in = to_dev(scale)
    wt, st = ops.repack_fp8_marlin_cuda(to_dev(codes).view(torch.float8_e4m3fn), st_in, block_n, 128)
    x = rng.standard_normal((m, k)).astype(np.float32)
    if m > 1:
        x[1] = 0.0
    if m > 2:
        x[2] *= np.exp2(rng.integers(-12, 5, k))  # 2^16 in scale; small enough for fp16 outputs
    x = O.round_to(x, dtype)
    xd = to_dev(x, TDT[dtype])
    fused = ops.gemm_fp8_w8a8_cuda(xd, wt, st, n, block_n, 128)
    tuning_env("PLM_W8A8_UNFUSED", "1")
    split = ops.gemm_fp8_w8a8_cuda(xd, wt, st, n, block_n, 128)
    tuning_env("PLM_W8A8_UNFUSED", None)
    torch.cuda.synchronize()
    # N = 34816: the fused kernel runs 16 wavefronts and the unfused one 8, so the
    # wavefronts' partial sums are added in another order; both are held to the bound below.
    same_order = n != 34816
    if same_order:
        assert torch.equal(fused, split)
    # The oracle on the first 1024 output columns (the CPU reference is slow at N = 34816).
    nc = min(n, 1024)
    codes, scale, fused = codes[:nc], scale[:-(-nc // block_n)], fused[:, :nc]
    xc, xs = O.quantize_per_token_e4m3(x)
    ref = O.gemm_w8a8_ref(xc, xs, codes, scale, block_n, 128, dtype=None)
    # The fp8 MFMA does not sum its 128 products exactly: it keeps about 2^-15 of the sum
    # of their magnitudes (measured), which shows where the codes span all of e4m3 and on
    # row 2. Bound: bf16 output rounding plus 2^-13 of sum |x| |w| over each row.
    xa = np.abs(O.e4m3_decode(xc).astype(np.float64) * xs[:, None])
    wa = np.abs(O.dequant_fp8(codes, scale, block_n, 128).astype(np.float64))
    bound = 2.0**-8 * np.abs(ref) + 2.0**-13 * (xa @ wa.T)
    for out in (fused, split[:, :nc]):
        err = np.abs(out.double().cpu().numpy() - ref)
        assert bool((err <= bound).all()), f"max err / bound {(err / np.maximum(bound, 1e-30)).max():.3g}"
