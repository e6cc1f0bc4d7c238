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
    ("w8a8", 7687, 4176, 7040, False),  # 281, 305
    ("int4", 2048, 34816, 5120, True),  # 664, 616
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


@pytest.mark.parametrize("fmt,m,n,k,tile,splits", [
    # The other shapes of one workgroup to a CU, us without the tail, us with it; 0: no tail.
    ("fp8", 2048, 5120, 17408, (256, 128), 4),  # 475, 370
    ("fp8", 2048, 5120, 5120, (256, 128), 4),  # 138, 125
    ("fp8", 207, 39536, 6656, (256, 128), 4),  # 198, 154
    ("int4", 2228, 3744, 13696, (128, 256), 8),  # 259, 230
    ("int4", 4330, 1936, 14080, (128, 256), 8),  # 268, 237
    ("int4", 422, 35344, 11776, (128, 256), 5),  # 401 (and 436 with an X tail), 368
    ("w8a8", 1007, 17440, 16896, (256, 192), 2),  # 409, 333
    ("w8a8", 450, 33408, 14464, (256, 192), 2),  # 353, 280
    ("w8a8", 2365, 20672, 7296, (256, 192), 4),  # 481 (and 417 with an X tail), 406
    ("w8a8", 1212, 6544, 15488, (256, 192), 0),  # 168, 197 (128 x 256 tiles)
    ("w8a8", 412, 17312, 17792, (256, 192), 0),  # 186, 228 (128 x 256 tiles)
])
def test_k_split_tail_of_other_shapes(fmt, m, n, k, tile, splits):
    plan = mfma_plan(fmt, m, n, k)
    assert plan["tile"] == tile and plan["tail_splits"] == splits and (plan["tail"] > 0) == (splits > 0), plan
