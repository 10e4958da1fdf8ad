"""The C requests of a batch (euc_amd/renderer.py, _requests_c) whose uniforms were
replaced after construction, on the CPU: each request's own first 64 floats, or a
ValueError where a request has fewer (also where another has as many more)."""
from types import SimpleNamespace

import numpy as np
import pytest

from euc_amd.renderer import N_UNIFORMS, Request, _requests_c


def requests(*uniforms):
    rs = [Request(SimpleNamespace(handle=k + 1), None, None, np.full(N_UNIFORMS, k, np.float32)) for k in range(len(uniforms))]
    for r, u in zip(rs, uniforms):
        if u is not None:
            r.uniforms = u
    return rs


def floats(arr, k):
    import ctypes as C
    return np.ctypeslib.as_array(C.cast(arr[k].uniforms, C.POINTER(C.c_float)), (N_UNIFORMS,))


def ramp(n, dtype=np.float32):
    return np.arange(100, 100 + n).astype(dtype)


@pytest.mark.parametrize("u", [ramp(N_UNIFORMS), ramp(N_UNIFORMS).reshape(4, 16), ramp(N_UNIFORMS + 7), ramp(2 * N_UNIFORMS)[:N_UNIFORMS],
                               ramp(N_UNIFORMS, np.float64), ramp(N_UNIFORMS + 2).reshape(3, 22)])
@pytest.mark.parametrize("at", [0, 1, 2])
def test_replaced_uniforms(u, at):
    rs = requests(*[u if k == at else None for k in range(3)])
    arr = _requests_c(rs)
    for k in range(3):
        assert arr[k].mesh == k + 1
        assert np.array_equal(floats(arr, k), ramp(N_UNIFORMS) if k == at else np.full(N_UNIFORMS, k, np.float32))


@pytest.mark.parametrize("sizes", [(N_UNIFORMS - 1,), (N_UNIFORMS - 1, N_UNIFORMS + 1), (N_UNIFORMS + 1, N_UNIFORMS - 1), (0, 2 * N_UNIFORMS)])
def test_too_few_uniforms(sizes):
    with pytest.raises(ValueError, match="uniforms"):
        _requests_c(requests(*map(ramp, sizes)))
