"""The MFMA kernel's tile shape and K split, on the CPU (where the library counts 256 CUs), at sizes where the shapes were
timed against each other."""

from __future__ import annotations

import pytest

from pulsarlm_amd import _lib
from tests._util import mfma_plan


@pytest.mark.parametrize("fmt,m,n,k,tile", [
    # Two to three workgroups a CU. The 112-row fp8 tile fits two on a CU, not three: us with it first.
    ("fp8", 402, 33888, 2688, (96, 128)),  # 118.7, 99.9
    ("fp8", 215, 36880, 1408, (64, 128)),  # 42.3, 36.1
    ("fp8", 2862, 3712, 9856, (256, 256)),  # 254.2, 240.7
    ("fp8", 598, 16000, 5632, (128, 128)),  # 159.3, 146.1
    # Three of the 96-row tile do: 128-row tiles first.
    ("fp8", 1572, 10096, 1152, (96, 128)),  # 54.1, 46.9
    ("fp8", 801, 19376, 3328, (96, 128)),  # 139.8, 122.3
])
def test_tile(fmt, m, n, k, tile):
    plan = mfma_plan(fmt, m, n, k)
    assert plan["tile"] == tile and plan["splits"] == 1 and plan["tail"] == 0, plan


@pytest.mark.parametrize("m,n,k,tile,splits", [
    # Short W8A8 calls: us on 96- to 128-row tiles with K in 3 to 6, us here.
    (236, 1568, 2944, (64, 128), 4),  # 21.7, 15.0
    (325, 1216, 1664, (64, 128), 4),  # 21.2, 14.1 (K in 3)
    (705, 1152, 1536, (64, 128), 1),  # 19.6, 14.4
    (570, 5744, 1664, (64, 128), 1),  # 19.3, 16.7
])
def test_w8a8(m, n, k, tile, splits):
    plan = mfma_plan("w8a8", m, n, k)
    assert plan["tile"] == tile and plan["splits"] == splits and plan["tail"] == 0, plan


@pytest.mark.parametrize("m,n,k,tile,splits", [
    # Sums of more than 24 MiB, which the call must bring anyway: us whole, us here.
    (1130, 3344, 17536, (128, 128), 2),  # 136, 99
    (363, 10368, 16384, (128, 128), 2),  # 106, 83
    (1185, 2704, 15744, (112, 128), 2),  # 103, 82
])
def test_w8a8_sums_fill_what_the_call_must_bring(m, n, k, tile, splits, tuning_env):
    plan = mfma_plan("w8a8", m, n, k)
    assert plan["tile"] == tile and plan["splits"] == splits and plan["tail"] == 0, plan
    size = _lib.load().plm_gemm_w8a8_workspace_bytes
    wanted = size(m, n, k)
    tuning_env("PLM_MFMA_UNSPLIT", "1")  # no partial sums: the bytes that any plan's call must bring
    assert size(m, n, k) == wanted
