"""Shared fixtures. GPU tests are marked ``gpu``; everything else runs on CPU."""
from __future__ import annotations

import os
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
if str(ROOT) not in sys.path:
    sys.path.insert(0, str(ROOT))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU")
    config.addinivalue_line("markers", "slow: CPU test that takes more than a few seconds")


def gpu_available() -> bool:
    try:
        import ctypes
        hip = ctypes.CDLL("libamdhip64.so")
        n = ctypes.c_int(0)
        return hip.hipGetDeviceCount(ctypes.byref(n)) == 0 and n.value > 0
    except OSError:
        return False


@pytest.fixture(scope="session")
def ctx():
    """One tgx context for the whole GPU session (fails loudly without a GPU)."""
    import tg_amd
    c = tg_amd.Context(int(os.environ.get("TGX_DEVICE", "0")))
    yield c
    c.close()


@pytest.fixture(scope="session")
def shipped_tuning(ctx):
    """The tuning a context is created with."""
    return ctx.tuning().copy()


@pytest.fixture(autouse=True)
def start_from_the_shipped_tuning(request):
    """A test on the session's context starts from the tuning that users get,
    whatever the tests before it have set."""
    if "ctx" in request.fixturenames:
        t = request.getfixturevalue("shipped_tuning")
        request.getfixturevalue("ctx").set_tuning(**{k: int(t[k][0]) for k in t.dtype.names})
    yield
