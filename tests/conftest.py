import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU")


def pytest_collection_modifyitems(config, items):
    try:
        import torch
        has_gpu = torch.cuda.is_available()
    except Exception:  # pragma: no cover
        has_gpu = False
    if has_gpu:
        return
    skip = pytest.mark.skip(reason="no GPU in this environment")
    for item in items:
        if "gpu" in item.keywords:
            item.add_marker(skip)


@pytest.fixture
def tuning_env(monkeypatch):
    """Set or clear one of the library's measurement knobs (PLM_* environment variables),
    which it parses once per process, and make it re-read them; on teardown the
    environment is restored and re-read again."""
    from pulsarlm_amd import _lib

    def set_knob(name, value):
        if value is None:
            monkeypatch.delenv(name, raising=False)
        else:
            monkeypatch.setenv(name, value)
        _lib.reload_tuning()

    yield set_knob
    monkeypatch.undo()
    _lib.reload_tuning()


@pytest.fixture(params=[None, "0"], ids=["rule", "no_rows"])
def with_and_without_rows(request, tuning_env):
    """Calls up to 128 rows by the dispatch rule, and without the rows kernel, on the decode and MFMA kernels."""
    tuning_env("PLM_ROWS", request.param)
