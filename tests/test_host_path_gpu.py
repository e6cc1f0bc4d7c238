"""The host path of a call: the stream it enqueues on and the sizes it keeps."""

import pytest
import torch

from pulsarlm_amd import _lib, ops

pytestmark = pytest.mark.gpu


def test_stream_is_torchs_current_stream():
    device = torch.empty(1, device="cuda").device
    side = torch.cuda.Stream()
    for stream in (torch.cuda.current_stream(), side):
        with torch.cuda.stream(stream):
            assert ops._stream(device) == stream.cuda_stream == ops._stream(torch.device("cuda"))
            ws = ops.workspace(device, 1)
            assert ops._ws[(device.index, stream.cuda_stream)] is ws
            with ops._on(device), ops._on(torch.device("cuda")):
                assert torch.cuda.current_device() == device.index


def test_kept_sizes_follow_the_knobs(tuning_env):
    args = (_lib.PLM_INT4, 300, 4096, 8192)
    for knob in (None, "R,1", "R,4", None):
        tuning_env("PLM_MFMA", knob)
        for _ in range(2):
            assert _lib.gemm_workspace_bytes(*args) == _lib.load().plm_gemm_workspace_bytes(*args)
            assert _lib.gemm_w8a8_workspace_bytes(*args[1:]) == _lib.load().plm_gemm_w8a8_workspace_bytes(*args[1:])
            assert _lib.weight_bytes(args[0], *args[2:]) == _lib.load().plm_weight_bytes(args[0], *args[2:])
