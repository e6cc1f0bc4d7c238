"""The partial-sum stores of the MFMA kernel's K splits."""

from __future__ import annotations

import numpy as np
import pytest

import torch

from pulsarlm_amd import ops
from tests._util import assert_close, fp8_case, scale_tensor, to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,m,n,k", [("fp8", 160, 12800, 1024), ("int4", 200, 12800, 1024), ("fp8", 250, 6400, 2048)])
def test_split_k_partials_with_workgroups_sharing_cus(fmt, m, n, k):
    """K splits of the MFMA kernel with more workgroups than CUs: the accumulators must stay
    untouched until their partial-sum stores have read them (the stores run late while another
    workgroup keeps the CU's memory pipeline busy)."""
    rng = np.random.default_rng(9)
    x = to_dev(rng.standard_normal((m, k)).astype(np.float32) * 0.1, torch.bfloat16)
    if fmt == "int4":
        packed = to_dev(rng.integers(-(2**31), 2**31, size=(n, k // 8), dtype=np.int64).astype(np.int32))
        s = to_dev((np.abs(rng.standard_normal((n, k // 128))) * 0.02 + 1e-3).astype(np.float16))
        w, sc = ops.repack_int4_marlin_cuda(packed, s, 1, 128)
        run = lambda: ops.gemm_int4_marlin_cuda(x, w, sc, n, 1, 128)  # noqa: E731
        dense = ops.dequant_marlin_cuda("int4", w, sc, n, k, 1, 128)
    else:
        codes, s = fp8_case(n, k, 128, 128, seed=6)
        w, sc = ops.repack_fp8_marlin_cuda(to_dev(codes).view(torch.float8_e4m3fn), scale_tensor(s), 128, 128)
        run = lambda: ops.gemm_fp8_marlin_cuda(x, w, sc, n, 128, 128)  # noqa: E731
        dense = ops.dequant_marlin_cuda("fp8", w, sc, n, k, 128, 128)
    ref = to_np(x.double() @ dense.double().t())
    for i in range(5):
        assert_close(run(), ref, f"{fmt} m={m} call {i}")
