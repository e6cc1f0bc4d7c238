"""The MoE block's sort in its one-launch and its chunked form, and the register router at the
edges of its expert counts."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle as O
from pulsarlm_amd import ops
from tests._util import to_dev

pytestmark = pytest.mark.gpu

TDTYPE = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}


@pytest.mark.parametrize("t,e,top_k", [(1, 1, 1), (3, 5, 2), (65, 64, 8), (32, 65, 8), (257, 3, 3), (33, 1000, 10), (64, 128, 8)])
def test_both_sorts_agree(t, e, top_k, tuning_env):
    """One bit for bit result, with expert ids in any order, repeated, and out of range (dropped)."""
    rng = np.random.default_rng(t + e)
    hidden = inter = 128
    gu = ops.repack_int4_experts(to_dev(rng.integers(0, 2**31, (e, 2 * inter, hidden // 8), dtype=np.int64).astype(np.int32)),
                                 to_dev((rng.random((e, 2 * inter, 1)) * 0.1).astype(np.float16)), 128)
    dn = ops.repack_int4_experts(to_dev(rng.integers(0, 2**31, (e, hidden, inter // 8), dtype=np.int64).astype(np.int32)),
                                 to_dev((rng.random((e, hidden, 1)) * 0.1).astype(np.float16)), 128)
    h = to_dev(rng.standard_normal((t, hidden)).astype(np.float32), torch.bfloat16)
    ids = rng.integers(-1, e + 2, (t, top_k)).astype(np.int32)
    weights = to_dev(rng.random((t, top_k)).astype(np.float32))
    got = []
    for small in (None, "0"):
        tuning_env("PLM_MOE_SMALL_SORT", small)
        out, offsets = ops.routed_experts_int4_cuda(h, to_dev(ids), weights, gu, dn, inter, 128)
        valid = ids[(ids >= 0) & (ids < e)]
        assert np.array_equal(offsets.cpu().numpy(), np.cumsum(np.bincount(valid, minlength=e)))
        got.append(out)
    assert torch.equal(got[0], got[1])


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("experts", [1, 2, 63, 64, 65, 127, 128, 129, 256, 257, 512, 513, 1024])
def test_register_router_equals_lds_router(experts, dtype):
    """Padded with -inf to 1025 columns the same logits take the kernel that keeps its probabilities
    in LDS; both have to give the same bits, with ties and masked experts."""
    gen = torch.Generator().manual_seed(experts)
    logits = torch.randn(77, experts, generator=gen)
    logits[1] = 0.5
    logits[2, ::2] = logits[2, 0]
    logits[3, 1:] = -float("inf")
    logits[4] = torch.finfo(torch.float16).min
    logits[5, -1] = 60.0
    logits = logits.to(TDTYPE[dtype]).cuda()
    padded = torch.full((77, 1025), -float("inf"), dtype=logits.dtype, device="cuda")
    padded[:, :experts] = logits
    k = min(experts, 64)
    w, c = ops.route_top_k_cuda(logits, k)
    w2, c2 = ops.route_top_k_cuda(padded, k)
    assert torch.equal(c, c2) and torch.equal(w, w2)
    w_ref, c_ref, _ = O.route_top_k_ref(logits.float().cpu().numpy(), k)
    assert torch.allclose(w.cpu(), torch.from_numpy(w_ref), rtol=1e-6, atol=1e-6)
    assert np.array_equal(c[1:5].cpu().numpy(), c_ref[1:5])


def test_register_router_nan_row():
    """Nothing ranks in a row with a NaN: no expert of the range, as before."""
    logits = torch.randn(3, 100, device="cuda")
    logits[1, 40] = float("nan")
    w, c = ops.route_top_k_cuda(logits, 4)
    assert (c[1] == 100).all() and torch.isnan(w[1]).all()
    assert torch.isfinite(w[0]).all() and torch.isfinite(w[2]).all() and (c[0] < 100).all()
