"""The partial-sum stores of the MFMA and rows kernels' K splits."""

from __future__ import annotations

import numpy as np
import pytest

import torch

from pulsarlm_amd import ops
from tests._util import MFMA_TILES, assert_close, force_mfma, force_rows, fp8_case, scale_tensor, to_dev, to_np

pytestmark = pytest.mark.gpu

CUS = 256


def _case(fmt, m, n, k):
    """A call and its float64 result (W8A8: of the quantized x)."""
    rng = np.random.default_rng(9)
    x = to_dev(rng.standard_normal((m, k)).astype(np.float32) * 0.1, torch.bfloat16)
    if fmt == "int4":
        packed = to_dev(rng.integers(-(2**31), 2**31, size=(n, k // 8), dtype=np.int64).astype(np.int32))
        s = to_dev((np.abs(rng.standard_normal((n, k // 128))) * 0.02 + 1e-3).astype(np.float16))
        w, sc = ops.repack_int4_marlin_cuda(packed, s, 1, 128)
        dense = ops.dequant_marlin_cuda("int4", w, sc, n, k, 1, 128)
        return lambda: ops.gemm_int4_marlin_cuda(x, w, sc, n, 1, 128), to_np(x.double() @ dense.double().t())
    codes, s = fp8_case(n, k, 128, 128, seed=6)
    cd = to_dev(codes).view(torch.float8_e4m3fn)
    w, sc = ops.repack_fp8_marlin_cuda(cd, scale_tensor(s), 128, 128)
    if fmt == "fp8":
        dense = ops.dequant_marlin_cuda("fp8", w, sc, n, k, 128, 128)
        return lambda: ops.gemm_fp8_marlin_cuda(x, w, sc, n, 128, 128), to_np(x.double() @ dense.double().t())
    xq, sx = ops.quantize_rows_e4m3_cuda(x)
    xd = xq.view(torch.float8_e4m3fn).double() * sx.double()[:, None]
    wide = scale_tensor(s).double().repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)
    return lambda: ops.gemm_fp8_w8a8_cuda(x, w, sc, n, 128, 128), to_np(xd @ (cd.double() * wide).t())


# The shapes of which two workgroups fit on a CU.
@pytest.mark.parametrize("fmt,shape", [("int4", s) for s in "RQBCD"] + [("fp8", s) for s in "RABCD"] + [("w8a8", s) for s in "SRABCD"])
def test_split_k_partials_with_workgroups_sharing_cus(fmt, shape, tuning_env):
    """K splits of the MFMA kernel with more workgroups than CUs: the accumulators must stay
    untouched until their partial-sum stores have read them (the stores run late while another
    workgroup keeps the CU's memory pipeline busy)."""
    bm, bn = MFMA_TILES[shape]
    m, n, k = 2 * bm - 5, min((24 << 20) // (4 * bm * bn * 4), 120) * bn, 1024
    tuning_env("PLM_ROWS", "0")
    p = force_mfma(tuning_env, fmt, m, n, k, shape, 2)
    assert p["tiles"] * p["splits"] > CUS, p
    run, ref = _case(fmt, m, n, k)
    for i in range(5):
        assert_close(run(), ref, f"{fmt} {shape} m={m} call {i}")


@pytest.mark.parametrize("fmt", ["int4", "fp8"])
@pytest.mark.parametrize("m,n,sg,splits", [(16, 4096, 1, 2), (32, 4096, 2, 4), (32, 6144, 3, 3)])
def test_rows_partials_with_workgroups_sharing_cus(fmt, m, n, sg, splits, tuning_env):
    """The same for the rows kernel, two workgroups of which fit on a CU up to 32 rows."""
    k = 2048
    p = force_rows(tuning_env, fmt, m, n, k, 1 if fmt == "int4" else 128, 128, "fp16" if fmt == "int4" else "fp32", sg, splits)
    assert p["m_blocks"] * p["n_blocks"] * p["splits"] > CUS, p
    run, ref = _case(fmt, m, n, k)
    for i in range(5):
        assert_close(run(), ref, f"{fmt} m={m} rows {sg},{splits} call {i}")
