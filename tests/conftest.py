import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU and the built HIP library")


@pytest.fixture
def rng():
    return np.random.default_rng(0)


def rel_err(a, b):
    """max |a - b| / max(|b|) -- the norm-wise relative error used for fp32
    outputs against the torch fake-quant reference (tolerance 1e-3)."""
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-30))


def gemm_form(M, K, N, G, GA=None, mode=0, workspace=False):
    """Which kernel wq_gemm launches for a shape, with no workspace or one of
    the size it asks for: (kernel, weight rows per tile, waves per workgroup,
    K split between workgroup pairs); kernel "tiles" (128 tokens) or "waves"
    (K split between the waves of a workgroup)."""
    import ctypes

    from webyiq_amd import _lib
    lib = _lib.load()
    GA = K if GA is None else GA
    nbytes = lib.wq_gemm_workspace_bytes(N, K, G, M, GA, mode) if workspace else 0
    form = (ctypes.c_int32 * 4)()
    hook = lib.wq_gemm_debug_form
    hook.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int32, ctypes.c_int64, ctypes.c_int32, ctypes.c_int32,
                     ctypes.c_size_t, ctypes.c_void_p]
    assert hook(N, K, G, M, GA, mode, nbytes, form) == 0, lib.wq_last_error()
    return ("tiles", "waves")[form[0]], form[1], form[2], bool(form[3])
