"""Shared helpers for the parity tests: seeded inputs (numpy, from the oracle's
generators) moved to the GPU, and the oracle comparisons."""

from __future__ import annotations

import ctypes

import numpy as np
import torch

from oracle import oracle as O
from pulsarlm_amd import _lib

TDT = {"bf16": torch.bfloat16, "fp16": torch.float16}


def to_dev(a: np.ndarray, dtype=None, device="cuda") -> torch.Tensor:
    t = torch.from_numpy(np.ascontiguousarray(a))
    if dtype is not None:
        t = t.to(dtype)
    return t.to(device)


def to_np(t: torch.Tensor) -> np.ndarray:
    return t.detach().float().cpu().numpy()


def int4_case(n, k, g, block_n=1, seed=0, scale_dtype=np.float16, scale_kind="baseline"):
    """q uniform [-8, 7] packed LSB-first, scales per the benchmark spec (|N(0,.02)|+1e-3) or the
    reference test's rand*0.1+0.01 (test_marlin.cpp:23-25)."""
    rng = np.random.default_rng(seed)
    q = rng.integers(-8, 8, size=(n, k))
    rows = -(-n // block_n)
    if scale_kind == "baseline":
        s = np.abs(rng.standard_normal((rows, k // g)) * 0.02) + 1e-3
    else:
        s = rng.random((rows, k // g)) * 0.1 + 0.01
    return O.pack_int4(q), s.astype(scale_dtype)


def fp8_case(n, k, g, block_n=1, seed=0, scale_dtype=np.float32):
    """Every e4m3 code except the NaNs (test_marlin.cpp:32-36), scales rand*0.1+0.01."""
    rng = np.random.default_rng(seed)
    codes = rng.integers(0, 256, (n, k), dtype=np.uint8)
    codes[(codes == 0x7F) | (codes == 0xFF)] = 0
    rows = -(-n // block_n)
    s = (rng.random((rows, k // g)) * 0.1 + 0.01).astype(scale_dtype)
    return codes, s


def scale_tensor(s: np.ndarray) -> torch.Tensor:
    if s.dtype == np.float16:
        return to_dev(s)
    if s.dtype == np.float32:
        return to_dev(s)
    raise ValueError(s.dtype)


def x_case(m, k, dtype="bf16", seed=0):
    rng = np.random.default_rng(1000 + seed)
    x = rng.standard_normal((m, k)).astype(np.float32)
    return O.round_to(x, dtype)


def assert_close(y: torch.Tensor, ref: np.ndarray, what=""):
    ok, st = O.check_close(to_np(y), ref)
    assert ok, f"{what}: {st}"
    return st


# Tile rows and columns of the MFMA kernel's shapes, by their PLM_MFMA letter.
MFMA_TILES = {"S": (128, 128), "R": (64, 128), "W": (256, 192), "X": (256, 256), "Q": (64, 128), "G": (256, 128), "H": (128, 256),
              "A": (128, 128), "B": (128, 128), "C": (96, 128), "D": (112, 128), "F": (96, 256)}


def _plan(fn, *args):
    out = (ctypes.c_int32 * 8)()
    f = getattr(_lib.load(), fn)
    f.restype, f.argtypes = None, [ctypes.c_int64] * len(args) + [ctypes.c_void_p]
    f(*args, out)
    return list(out)


def mfma_plan(fmt, m, n, k):
    """The MFMA kernel's plan for a plain call ("int4", "fp8" or "w8a8") under the present knobs."""
    rows, cols, tiles, splits, tail, tail_splits, halves, _ = _plan("plm_internal_mfma_plan", int(fmt != "int4"), m, n, k, int(fmt == "w8a8"))
    return {"tile": (rows, cols), "tiles": tiles, "splits": splits, "tail": tail, "tail_splits": tail_splits, "halves": bool(halves)}


def rows_plan(fmt, m, n, k, block_n, group, scale_dtype):
    """How a plain call runs on the rows kernel under the present knobs; None where another kernel takes it."""
    taken, rb, sg, m_blocks, n_blocks, splits = _plan("plm_internal_rows_plan", int(fmt != "int4"), m, n, k, block_n, group,
                                                      {"fp32": _lib.PLM_FP32, "fp16": _lib.PLM_FP16, "bf16": _lib.PLM_BF16}[scale_dtype])[:6]
    return {"rb": rb, "sg": sg, "m_blocks": m_blocks, "n_blocks": n_blocks, "splits": splits} if taken else None


def force_mfma(tuning_env, fmt, m, n, k, shape, splits):
    """Forces an MFMA shape and K split; a test that asks for one that cannot be had fails."""
    tuning_env("PLM_MFMA", f"{shape},{splits}")
    p = mfma_plan(fmt, m, n, k)
    assert p["tile"] == MFMA_TILES[shape] and p["splits"] == splits and p["tail"] == 0, f"{shape},{splits}: planned {p}"
    return p


def force_rows(tuning_env, fmt, m, n, k, block_n, group, scale_dtype, sg, splits):
    """The same for the rows kernel's strips per workgroup and K split."""
    tuning_env("PLM_ROWS", f"{sg},{splits}")
    p = rows_plan(fmt, m, n, k, block_n, group, scale_dtype)
    assert p is not None and (p["sg"], p["splits"]) == (sg, splits), f"{sg},{splits}: planned {p}"
    return p
