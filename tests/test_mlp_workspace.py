"""The training workspace holds what a batch needs: no more than a quarter over the FP32 rows
(pre-activations, their gradients, activations), the outputs and the partial sums of a plain layout."""
import ctypes
import os

import pytest

from tests.conftest import ROOT

LIB = os.path.join(ROOT, 'pyvibdmc_amd', 'libpyvibdmc_amd.so')


@pytest.mark.skipif(not os.path.exists(LIB), reason='library not built')
@pytest.mark.parametrize('hidden', [128, 256])
@pytest.mark.parametrize('d', [3, 15, 32])
def test_workspace_grows_with_the_batch(hidden, d):
    f = ctypes.CDLL(LIB).pvd_mlp_workspace_bytes
    f.restype, f.argtypes = ctypes.c_int64, [ctypes.c_int32, ctypes.c_int32, ctypes.c_int64]
    last = 0
    for n in [1, 31, 160, 161, 200, 224, 255, 256, 257, 400, 700, 1000, 1500, 2000, 2048, 2049, 2208, 2209, 4100, 8192, 10001, 20000]:
        rows = (n + 255) // 256
        plain = 4 * (6 * hidden * n + 2 * n + rows * hidden * hidden + 2 * rows) + 64
        got = f(d, hidden, n)
        assert got >= last, n  # a buffer for a batch serves every smaller one
        if n >= 200:
            assert got <= 1.25 * plain, (n, got / plain)
        last = got
