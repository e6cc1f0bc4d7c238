"""When whole rounds of the tall tile are followed by a second launch for the rest, on the CPU (where the
library counts 256 CUs): measured sizes on both sides."""

from __future__ import annotations

import pytest

from tests._util import mfma_plan


@pytest.mark.parametrize("fmt,m,n,k,tail", [
    # us whole tiles, us with the tail (K split, then halves of whole columns of tiles).
    ("fp8", 2048, 34816, 5120, True),  # 762, 676
    ("fp8", 4096, 5120, 17408, True),  # 738, 650
    ("fp8", 8479, 1984, 11776, True),  # 526, 413
    ("fp8", 1495, 14416, 5632, False),  # 254, 268
    ("int4", 1206, 27632, 16896, True),  # 1218, 956
    ("int4", 2403, 19968, 1408, False),  # 141, 153
    ("w8a8", 2365, 20672, 7296, True),  # 481, 413
    ("w8a8", 7687, 4176, 7040, False),  # 281, 305
    ("int4", 2048, 34816, 5120, True),  # 664, 616
    ("int4", 886, 38144, 6784, True),  # 479, 422
    ("int4", 422, 35344, 11776, False),  # 415, 436
    ("w8a8", 2048, 34816, 5120, True),  # 406, 391
    ("w8a8", 1024, 24576, 4096, False),  # 113, 126
    ("w8a8", 1835, 10128, 4096, False),  # 98, 106
])
def test_tail(fmt, m, n, k, tail):
    plan = mfma_plan(fmt, m, n, k)
    assert (plan["tail"] > 0) == tail, plan
    if tail:  # the tiles past whole rounds, at most half a round
        assert plan["tile"] == (256, 256) and plan["tail"] == plan["tiles"] % 256 <= 128
        assert plan["halves"] if fmt != "fp8" and plan["tail"] % -(-m // 256) == 0 else plan["tail_splits"] > 1
