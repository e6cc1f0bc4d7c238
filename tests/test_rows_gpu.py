"""The rows kernel (decode batches and short prefills, up to 128 rows): its tile shapes, K splits, scale
layouts and edges against the oracle, and against the decode / MFMA kernels that take the call
without it."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle as O
from pulsarlm_amd import _lib, ops
from tests._util import TDT, assert_close, force_rows, fp8_case, int4_case, rows_plan, scale_tensor, to_dev, to_np, x_case

pytestmark = pytest.mark.gpu


def _int4(n, k, g, sdt, seed):
    packed, s = int4_case(n, k, g, 1, seed=seed)
    if sdt == "bf16":
        s = O.round_to(s.astype(np.float32), "bf16")
        dev = to_dev(s).to(torch.bfloat16)
    else:
        s = s.astype(np.float16 if sdt == "fp16" else np.float32)
        dev = scale_tensor(s)
    return packed, s, ops.repack_int4_marlin_cuda(to_dev(packed), dev, 1, g)


# Row blocks of one to four (and two row blocks of them), one to four strips and K splits, on a
# strip count that no group divides (N = 1016: 63.5 strips, the last one half empty).
@pytest.mark.parametrize("m", [5, 16, 17, 33, 48, 49, 64, 65, 97, 128])
@pytest.mark.parametrize("shape", [(1, 1), (2, 3), (3, 2), (4, 8), (4, 1), (1, 4)])
def test_int4_shapes_and_splits(m, shape, tuning_env):
    n, k = 1016, 2944  # 23 K tiles: the wavefronts hold two or three, in splits down to none
    packed, s, (w, sc) = _int4(n, k, 128, "fp16", seed=m)
    x = x_case(m, k, "bf16", seed=m)
    ref = O.gemm_ref(x, O.dequant_int4(packed, s, 1, 128), None)
    force_rows(tuning_env, "int4", m, n, k, 1, 128, "fp16", *shape)
    xd = to_dev(x, torch.bfloat16)
    a = ops.gemm_int4_marlin_cuda(xd, w, sc, n, 1, 128)
    assert_close(a, ref, f"m={m} rows {shape}")
    assert torch.equal(a, ops.gemm_int4_marlin_cuda(xd, w, sc, n, 1, 128)), "not deterministic"
    tuning_env("PLM_ROWS", "0")
    assert_close(ops.gemm_int4_marlin_cuda(xd, w, sc, n, 1, 128), ref, f"m={m} without the rows kernel")


# Every scale storage type, groups that divide a K tile, straddle its slices (48, 80, 112) or span
# several tiles (384), K that ends inside a tile, and K of a single tile.
@pytest.mark.parametrize("m", [1, 24, 100])
@pytest.mark.parametrize("g,k", [(16, 144), (32, 4128), (48, 1008), (64, 2112), (80, 1040), (112, 896), (128, 128),
                                 (256, 2560), (384, 2688)])
@pytest.mark.parametrize("sdt,dtype", [("fp16", "fp16"), ("fp32", "bf16"), ("bf16", "bf16")])
def test_int4_groups_and_k_tails(m, g, k, sdt, dtype, tuning_env):
    n = 520
    tuning_env("PLM_ROWS", "1")
    assert rows_plan("int4", m, n, k, 1, g, sdt) is not None
    packed, s, (w, sc) = _int4(n, k, g, sdt, seed=g + m)
    x = x_case(m, k, dtype, seed=k)
    y = ops.gemm_int4_marlin_cuda(to_dev(x, TDT[dtype]), w, sc, n, 1, g)
    assert_close(y, O.gemm_ref(x, O.dequant_int4(packed, s, 1, g, dtype), None), f"m={m} g={g} k={k}")


@pytest.mark.parametrize("m", [4, 16, 31, 48, 64, 80])
@pytest.mark.parametrize("block_n,dtype", [(128, "bf16"), (1, "fp16")])
@pytest.mark.parametrize("n,k,shape", [(7176, 2304, (1, 1)), (7176, 2304, (2, 2)), (7176, 2304, (3, 1)), (7176, 2304, (4, 3)),
                                       (1016, 2944, (4, 8))])
def test_fp8_shapes(m, block_n, dtype, n, k, shape, tuning_env):
    codes, s = fp8_case(n, k, 128, block_n, seed=m)
    w, sc = ops.repack_fp8_marlin_cuda(to_dev(codes).view(torch.float8_e4m3fn), scale_tensor(s), block_n, 128)
    x = x_case(m, k, dtype, seed=m) * np.float32(0.05)
    x = O.round_to(x, dtype)
    force_rows(tuning_env, "fp8", m, n, k, block_n, 128, "fp32", *shape)
    xd = to_dev(x, TDT[dtype])
    y = ops.gemm_fp8_marlin_cuda(xd, w, sc, n, block_n, 128)
    dense = ops.dequant_marlin_cuda("fp8", w, sc, n, k, block_n, 128, TDT[dtype])  # pinned to the oracle elsewhere
    ref = to_np(xd.double() @ dense.double().t())
    assert_close(y, ref, f"m={m} bn={block_n} {shape}")
    tuning_env("PLM_ROWS", "0")
    assert_close(ops.gemm_fp8_marlin_cuda(xd, w, sc, n, block_n, 128), ref, f"m={m} bn={block_n} without the rows kernel")


def test_rows_beside_nan_and_inf():
    """A non-finite value in one row stays in that row, and x past the last row is never read."""
    m, n, k = 20, 512, 4096
    assert rows_plan("int4", m, n, k, 1, 128, "fp16") is not None
    packed, s, (w, sc) = _int4(n, k, 128, "fp16", seed=3)
    x = x_case(64, k, "bf16", seed=4)
    big = to_dev(x, torch.bfloat16)
    big[m:] = float("nan")
    clean = ops.gemm_int4_marlin_cuda(big[:m].contiguous(), w, sc, n, 1, 128)
    xd = big[:m]  # contiguous rows with NaNs right behind them
    assert torch.equal(ops.gemm_int4_marlin_cuda(xd, w, sc, n, 1, 128), clean)
    bad = big[:m].clone()
    bad[7, 100] = float("inf")
    y = ops.gemm_int4_marlin_cuda(bad, w, sc, n, 1, 128)
    assert not torch.isfinite(y[7].float()).all()
    keep = [r for r in range(m) if r != 7]
    assert torch.equal(y[keep], clean[keep])


@pytest.mark.parametrize("fmt,m,n,k", [("int4", 48, 1024, 4096), ("int4", 100, 2048, 8192), ("fp8", 16, 5120, 17408)])
def test_split_rows_graph_replays_match_eager(fmt, m, n, k):
    """Calls whose plan splits K, captured: the arrival counters are left zero by every call."""
    p = rows_plan(fmt, m, n, k, 1 if fmt == "int4" else 128, 128, "fp16" if fmt == "int4" else "fp32")
    assert p is not None and p["splits"] > 1, p
    rng = np.random.default_rng(5)
    x = to_dev(rng.standard_normal((m, k)).astype(np.float32), torch.bfloat16)
    if fmt == "int4":
        packed = to_dev(rng.integers(-(2**31), 2**31, size=(n, k // 8), dtype=np.int64).astype(np.int32))
        s = to_dev((np.abs(rng.standard_normal((n, k // 128))) * 0.02 + 1e-3).astype(np.float16))
        w, sc = ops.repack_int4_marlin_cuda(packed, s, 1, 128)
        run = lambda: ops.gemm_int4_marlin_cuda(x, w, sc, n, 1, 128)  # noqa: E731
    else:
        codes, s = fp8_case(n, k, 128, 128, seed=6)
        w, sc = ops.repack_fp8_marlin_cuda(to_dev(codes).view(torch.float8_e4m3fn), scale_tensor(s), 128, 128)
        run = lambda: ops.gemm_fp8_marlin_cuda(x, w, sc, n, 128, 128)  # noqa: E731
    eager = run()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        run()  # the stream's workspace is allocated (zeroed) outside the capture
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out = run()
    for i in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), f"replay {i}"
        assert torch.equal(run(), eager), f"eager after replay {i}"


@pytest.mark.parametrize("m,n,k", [(24, 4096, 12288), (5, 4096, 12288)])
def test_small_workspace_keeps_the_general_path(m, n, k, tuning_env):
    """A workspace that only the decode kernels' need fits is accepted, with their result to the bit; one
    below that is refused."""
    lib = _lib.load()
    packed, s, (w, sc) = _int4(n, k, 128, "fp16", seed=8)
    x = to_dev(x_case(m, k, "bf16", seed=8), torch.bfloat16)
    full = lib.plm_gemm_workspace_bytes(_lib.PLM_INT4, m, n, k)
    by_rows = ops.gemm_int4_marlin_cuda(x, w, sc, n, 1, 128)
    p = rows_plan("int4", m, n, k, 1, 128, "fp16")
    assert full == 65536 + p["m_blocks"] * p["n_blocks"] * p["splits"] * p["rb"] * p["sg"] * 1024
    tuning_env("PLM_ROWS", "0")
    general = lib.plm_gemm_workspace_bytes(_lib.PLM_INT4, m, n, k)
    by_decode = ops.gemm_int4_marlin_cuda(x, w, sc, n, 1, 128)
    tuning_env("PLM_ROWS", None)
    assert 0 < general < full and not torch.equal(by_rows, by_decode)
    for nbytes, want in ((full, by_rows), (full - 1, by_decode), (general, by_decode), (general - 1, None), (0, None)):
        ws = torch.zeros(max(nbytes, 1), dtype=torch.uint8, device="cuda")
        y = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
        rc = lib.plm_gemm(_lib.PLM_INT4, x.data_ptr(), _lib.PLM_BF16, w.data_ptr(), sc.data_ptr(), _lib.PLM_FP16, m, n, k, 1,
                          128, y.data_ptr(), ws.data_ptr() if nbytes else None, nbytes,
                          torch.cuda.current_stream().cuda_stream)
        if want is None:
            assert rc == _lib.PLM_ERR_WORKSPACE, nbytes
        else:
            assert rc == _lib.PLM_OK and torch.equal(y, want), nbytes
