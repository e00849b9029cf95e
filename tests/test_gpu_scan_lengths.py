"""Calls whose counts scan in one kernel or in three: visibility counts at the
ends of a thread's elements, of a round and of the one-kernel form.  Bars
against the serial FP64 oracle as in test_gpu_bands.py: grid 1e-5 norm-wise,
num_skipped exact, norm 1e-12.
"""
import numpy as np
import pytest

from conftest import errors
from oracle import oracle
from test_gpu_bands import _case, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 17, 16383, 16385, 32767, 32768, 32769])
def test_visibility_counts(gpu, n):
    torch, ops = gpu
    c = _case(130, 4, [1, 2], n, seed=n)
    grid0 = np.zeros((130, 130, 2))
    t, tn, ts = oracle.grid_fsel_d(c, grid=grid0.copy(), norm=0.0)
    g, nn, s = _run(torch, ops, c, torch.float32, grid0)
    assert s == ts and abs(nn - tn) <= 1e-12 * abs(tn)
    assert np.abs(t).max() == 0 or errors(g, t)[0] <= 1e-5
