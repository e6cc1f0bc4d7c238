"""Which kernel a call up to 128 rows takes, on the CPU (where the library counts 256 CUs): measured
sizes on both sides of the rule's lines."""

from __future__ import annotations

import pytest

from pulsarlm_amd import _lib
from tests._util import rows_plan


@pytest.mark.parametrize("fmt,m,n,k,g,rows", [
    # Exactly one strip per CU: the split-K decode kernel as long as it holds x in LDS.
    ("int4", 1, 4096, 13312, 128, False), ("int4", 2, 4096, 20480, 128, False), ("int4", 3, 4096, 16384, 128, False),
    ("int4", 3, 4096, 17408, 128, True), ("int4", 4, 4096, 12288, 128, False), ("int4", 4, 4096, 13312, 128, True),
    ("int4", 1, 4080, 13312, 128, True), ("int4", 1, 4112, 13312, 128, True),
    # More than four strips per CU, few rows.
    ("int4", 1, 18944, 4480, 128, False), ("int4", 2, 17408, 4608, 128, False), ("int4", 3, 18944, 4480, 128, True),
    ("int4", 6, 17856, 4608, 384, False), ("int4", 4, 25024, 2368, 32, False), ("fp8", 1, 10368, 19584, 128, False),
    # Few K tiles.
    ("int4", 1, 640, 384, 384, False), ("int4", 4, 26048, 384, 384, False), ("int4", 17, 25536, 1152, 64, False),
    ("fp8", 17, 32000, 1024, 128, False), ("fp8", 56, 32000, 1024, 128, False), ("fp8", 3, 29685, 768, 384, False),
    # 33 to 64 rows past four strips per CU.
    ("fp8", 56, 18368, 8320, 128, False), ("int4", 40, 22592, 9472, 256, False), ("int4", 48, 24576, 4096, 128, True),
    # Above 64 rows.
    ("int4", 112, 5056, 8448, 256, False), ("fp8", 128, 1216, 18176, 256, True), ("int4", 96, 4096, 12288, 128, True),
    ("fp8", 112, 2752, 8448, 128, True),
])
def test_rows_rule(fmt, m, n, k, g, rows):
    plan = rows_plan(fmt, m, n, k, 1 if fmt == "int4" else 128, g, "fp16" if fmt == "int4" else "fp32")
    assert (plan is not None) == rows


@pytest.mark.parametrize("fmt,m,n,k", [("fp8", 2, 5290, 8576), ("int4", 2, 17026, 4864), ("fp8", 4, 4850, 5088)])
def test_no_workspace_for_a_kernel_that_no_call_of_the_size_takes(fmt, m, n, k, tuning_env):
    """The size query counts the rows kernel's K split only where some group size takes the call there."""
    f = _lib.PLM_INT4 if fmt == "int4" else _lib.PLM_FP8
    assert all(rows_plan(fmt, m, n, k, 1, g, "fp32") is None for g in (16, 128, 256))
    assert _lib.load().plm_gemm_workspace_bytes(f, m, n, k) == 0
    tuning_env("PLM_ROWS", "1")
    assert _lib.load().plm_gemm_workspace_bytes(f, m, n, k) > 0
