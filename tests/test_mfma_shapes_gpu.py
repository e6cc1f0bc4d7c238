"""Every tile shape and K split of the MFMA kernel, at row counts around its tile edges, against the
dequantized weights (pinned to the oracle elsewhere) in float64."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle as O
from pulsarlm_amd import _lib, ops
from tests._util import TDT, assert_close, force_mfma, fp8_case, int4_case, mfma_plan, scale_tensor, to_dev, to_np, x_case

pytestmark = pytest.mark.gpu

# N = 1016: the last strip is half empty and no shape's strips divide its 64; K = 3072: 24 K tiles, so that
# splits of 5 (the last one a tile shorter) and 8 exist.
N, K = 1016, 3072
ROWS = {"R": 64, "W": 256, "X": 256, "Q": 64, "H": 128, "B": 128, "C": 96, "D": 112, "F": 96, "A": 128, "G": 256, "S": 128}


def _splits(shape, m):
    """8 where the plan allows it: its limits are the partial sums' bytes and the tiles per CU."""
    return (1, 5, 8 if m <= ROWS[shape] + 1 else 4)


@pytest.fixture(autouse=True)
def no_rows_kernel(tuning_env):
    tuning_env("PLM_ROWS", "0")


@pytest.mark.parametrize("g,dtype,sdt", [(128, "bf16", "fp16"), (32, "fp16", "fp16"), (48, "bf16", "fp32"), (384, "bf16", "fp32")])
@pytest.mark.parametrize("shape", list("RWXQHBCDF"))
def test_int4_shapes(shape, g, dtype, sdt, tuning_env):
    packed, s = int4_case(N, K, g, 1, seed=g)
    s = s.astype(np.float16 if sdt == "fp16" else np.float32)
    w, sc = ops.repack_int4_marlin_cuda(to_dev(packed), scale_tensor(s), 1, g)
    dense = ops.dequant_marlin_cuda("int4", w, sc, N, K, 1, g, TDT[dtype]).double()
    for m in (33, ROWS[shape] - 1, ROWS[shape] + 1, 3 * ROWS[shape] + 17):
        x = to_dev(x_case(m, K, dtype, seed=m), TDT[dtype])
        ref = to_np(x.double() @ dense.t())
        for splits in _splits(shape, m):
            force_mfma(tuning_env, "int4", m, N, K, shape, splits)
            y = ops.gemm_int4_marlin_cuda(x, w, sc, N, 1, g)
            assert_close(y, ref, f"{shape} m={m} splits={splits}")
            assert torch.equal(y, ops.gemm_int4_marlin_cuda(x, w, sc, N, 1, g)), "not deterministic"


@pytest.mark.parametrize("block_n,dtype", [(128, "bf16"), (1, "fp16")])
@pytest.mark.parametrize("shape", list("RXGABCDF"))
def test_fp8_shapes(shape, block_n, dtype, tuning_env):
    codes, s = fp8_case(N, K, 128, block_n, seed=5)
    w, sc = ops.repack_fp8_marlin_cuda(to_dev(codes).view(torch.float8_e4m3fn), scale_tensor(s), block_n, 128)
    dense = ops.dequant_marlin_cuda("fp8", w, sc, N, K, block_n, 128, TDT[dtype]).double()
    for m in (33, ROWS[shape] - 1, ROWS[shape] + 1, 2 * ROWS[shape] + 17):
        x = to_dev(O.round_to(x_case(m, K, dtype, seed=m) * np.float32(0.05), dtype), TDT[dtype])
        ref = to_np(x.double() @ dense.t())
        for splits in _splits(shape, m):
            force_mfma(tuning_env, "fp8", m, N, K, shape, splits)
            assert_close(ops.gemm_fp8_marlin_cuda(x, w, sc, N, block_n, 128), ref, f"{shape} m={m} splits={splits}")


@pytest.mark.parametrize("shape", list("SRWXHABCD"))
def test_w8a8_shapes(shape, tuning_env):
    rng = np.random.default_rng(7)
    codes, scale = O.fp8_block_quantize(O.bf16_round(rng.standard_normal((N, K)).astype(np.float32) * 0.02), 128, 128)
    w, sc = ops.repack_fp8_marlin_cuda(to_dev(codes).view(torch.float8_e4m3fn), to_dev(scale), 128, 128)
    for m in (33, ROWS[shape] - 1, ROWS[shape] + 1, 2 * ROWS[shape] + 17):
        x = x_case(m, K, "bf16", seed=m)
        xc, xs = O.quantize_per_token_e4m3(x)
        ref = O.gemm_w8a8_ref(xc, xs, codes, scale, 128, 128, dtype=None)
        for splits in _splits(shape, m):
            force_mfma(tuning_env, "w8a8", m, N, K, shape, splits)
            y = ops.gemm_fp8_w8a8_cuda(to_dev(x, torch.bfloat16), w, sc, N, 128, 128)
            assert_close(y, ref, f"{shape} m={m} splits={splits}")


def test_random_sizes_by_the_rule(tuning_env):
    """The plan's own pick at random sizes, ragged in every dimension."""
    tuning_env("PLM_ROWS", None)
    rng = np.random.default_rng(3)
    for _ in range(30):
        m, n = int(2 ** rng.uniform(4, 11)), int(2 ** rng.uniform(5, 12.5))
        g = int(rng.choice([16, 32, 64, 128]))
        k = g * max(1, int(2 ** rng.uniform(6, 12)) // g)
        packed, s = int4_case(n, k, g, 1, seed=m)
        w, sc = ops.repack_int4_marlin_cuda(to_dev(packed), to_dev(s), 1, g)
        x = to_dev(x_case(m, k, "bf16", seed=n), torch.bfloat16)
        dense = ops.dequant_marlin_cuda("int4", w, sc, n, k, 1, g).double()
        print(m, n, k, g, flush=True)
        assert_close(ops.gemm_int4_marlin_cuda(x, w, sc, n, 1, g), to_np(x.double() @ dense.t()), f"{m}x{n}x{k} g{g}")


@pytest.mark.parametrize("m,n,shape,splits", [(5 * 64 - 3, 1016, "R", 1), (9 * 64, 136, "R", 2), (16 * 64, 1016, "R", 1),
                                              (17 * 64 + 1, 264, "R", 1), (2040, 8440, "X", 0)])
def test_xcd_patches(m, n, shape, splits, tuning_env):
    """Every work tile once, for row blocks below, at and past the patch height and at 16 (id order),
    tile counts that 8 does not divide, and the launch before a tail of half tiles."""
    k = 1152
    packed, s = int4_case(n, k, 128, 1, seed=n)
    w, sc = ops.repack_int4_marlin_cuda(to_dev(packed), to_dev(s), 1, 128)
    dense = ops.dequant_marlin_cuda("int4", w, sc, n, k, 1, 128).double()
    x = to_dev(x_case(m, k, "bf16", seed=m), torch.bfloat16)
    if splits:
        force_mfma(tuning_env, "int4", m, n, k, shape, splits)
    else:
        tuning_env("PLM_MFMA", shape)
        p = mfma_plan("int4", m, n, k)
        assert p["tile"] == (256, 256) and p["halves"], p
    y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    assert_close(ops.gemm_int4_marlin_cuda(x, w, sc, n, 1, 128, out=y), to_np(x.double() @ dense.t()), f"{shape} {m}x{n}")


@pytest.mark.parametrize("fmt,m,n,k", [("int4", 333, 4096, 4096), ("fp8", 300, 1024, 4096)])
def test_plan_follows_the_workspace(fmt, m, n, k):
    """Calls of one size with several workspaces in turn, from what the plan asks for down to what is
    refused: each is within tolerance, a smaller one splits K otherwise, and each size of workspace gives
    its own bits every time (plans are kept by the bytes they may use)."""
    lib = _lib.load()
    rng = np.random.default_rng(4)
    x = to_dev(x_case(m, k, "bf16", seed=4), torch.bfloat16)
    if fmt == "int4":
        packed, s = int4_case(n, k, 128, 1, seed=4)
        w, sc = ops.repack_int4_marlin_cuda(to_dev(packed), to_dev(s), 1, 128)
        f, bn, sdt = _lib.PLM_INT4, 1, _lib.PLM_FP16
    else:
        codes, scale = O.fp8_block_quantize(O.bf16_round(rng.standard_normal((n, k)).astype(np.float32) * 0.02), 128, 128)
        w, sc = ops.repack_fp8_marlin_cuda(to_dev(codes).view(torch.float8_e4m3fn), to_dev(scale), 128, 128)
        f, bn, sdt = _lib.PLM_FP8, 128, _lib.PLM_FP32
    ref = to_np(x.double() @ ops.dequant_marlin_cuda(fmt, w, sc, n, k, bn, 128).double().t())
    full = lib.plm_gemm_workspace_bytes(f, m, n, k)
    sizes, seen = [full, full - 1, 3 * full // 4, full // 2 + 65536], {}
    ws = torch.zeros(full, dtype=torch.uint8, device="cuda")
    for i in range(3):
        for nbytes in sizes:
            y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
            rc = lib.plm_gemm(f, x.data_ptr(), _lib.PLM_BF16, w.data_ptr(), sc.data_ptr(), sdt, m, n, k, bn, 128, y.data_ptr(),
                              ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream)
            if rc == _lib.PLM_ERR_WORKSPACE:
                assert nbytes < full - 1
                continue
            assert rc == _lib.PLM_OK
            assert_close(y, ref, f"{nbytes} of {full} bytes, call {i}")
            assert torch.equal(seen.setdefault(nbytes, y), y), f"{nbytes} of {full} bytes, call {i}"
    assert any(not torch.equal(y, seen[full]) for y in seen.values())


@pytest.mark.parametrize("fmt,shape,m,n,k,splits", [
    ("fp8", "G", 999, 8296, 1408, 2), ("fp8", "G", 1511, 5480, 2944, 5), ("int4", "H", 487, 16616, 2944, 5),
    ("int4", "H", 743, 10984, 2176, 4), ("w8a8", "W", 999, 12456, 2944, 5)])
def test_k_split_tails(fmt, shape, m, n, k, splits, tuning_env):
    """Whole rounds of a shape and the tiles past them with K split, in a second launch: the last row block and
    the last strip are ragged and lie in the tail."""
    tuning_env("PLM_MFMA", shape)
    plan = mfma_plan(fmt, m, n, k)
    assert plan["tile"][0] == ROWS[shape] and plan["tail"] > 0 and plan["tail_splits"] == splits and not plan["halves"], plan
    x = to_dev(x_case(m, k, "bf16", seed=m), torch.bfloat16)
    if fmt == "w8a8":
        rng = np.random.default_rng(3)
        codes, scale = O.fp8_block_quantize(O.bf16_round(rng.standard_normal((n, k)).astype(np.float32) * 0.02), 128, 128)
        w, sc = ops.repack_fp8_marlin_cuda(to_dev(codes).view(torch.float8_e4m3fn), to_dev(scale), 128, 128)
        ref = O.gemm_w8a8_ref(*O.quantize_per_token_e4m3(to_np(x)), codes, scale, 128, 128, dtype=None)
        run = lambda: ops.gemm_fp8_w8a8_cuda(x, w, sc, n, 128, 128)
    else:
        block_n = 1 if fmt == "int4" else 128
        if fmt == "int4":
            packed, s = int4_case(n, k, 128, 1, seed=n)
            w, sc = ops.repack_int4_marlin_cuda(to_dev(packed), scale_tensor(s.astype(np.float16)), 1, 128)
            run = lambda: ops.gemm_int4_marlin_cuda(x, w, sc, n, 1, 128)
        else:
            codes, s = fp8_case(n, k, 128, 128, seed=n)
            x = (x * 0.05).contiguous()
            w, sc = ops.repack_fp8_marlin_cuda(to_dev(codes).view(torch.float8_e4m3fn), scale_tensor(s), 128, 128)
            run = lambda: ops.gemm_fp8_marlin_cuda(x, w, sc, n, 128, 128)
        ref = to_np(x.double() @ ops.dequant_marlin_cuda(fmt, w, sc, n, k, block_n, 128, torch.bfloat16).double().t())
    y = run()
    assert_close(y, ref, f"{fmt} {shape} m={m}")
    assert torch.equal(y, run()), "not deterministic"
