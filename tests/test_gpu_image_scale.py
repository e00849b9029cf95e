"""Where the image's scale is applied and where the image is written: norms
that shift the cells' exponents a little (the scale goes in before the
transform) and far (after it), and images less aligned than the transform's
stores (through the work buffer), against the oracle's direct FP64 sum.

Bars as in the image tests: norm-wise max|I - I64| / max|I64| <= 1e-5 in FP32,
1e-12 in FP64.  A scale that took cells below the normal range would leave
them a few bits: an error of 8e-4 in the third case.
"""
import numpy as np
import pytest

from oracle import oracle

pytestmark = pytest.mark.gpu

G = 128


def _image(torch, ops, grid, norm, offset):
    real = torch.float32 if grid.dtype == np.complex64 else torch.float64
    buf = torch.full((G * G + 4,), -7.0, dtype=real, device="cuda")
    img = buf[offset:offset + G * G].view(G, G)
    ops.grid_to_image(torch.from_numpy(grid).cuda(), G, img, norm=norm)
    torch.cuda.synchronize()
    out = buf.cpu().numpy()
    assert (out[:offset] == -7).all() and (out[offset + G * G:] == -7).all()
    return out[offset:offset + G * G].reshape(G, G).astype(np.float64)


def _grid(prec, size):
    rng = np.random.default_rng(3)
    g = 1 + 0.5 * (rng.normal(size=(G, G)) + 1j * rng.normal(size=(G, G)))
    return (g * size).astype(np.complex64 if prec == "f" else np.complex128)


# (precision, size of the cells, norm): the brightest pixel keeps 19 bits or
# more, though the scaled cells of the third would keep 4
@pytest.mark.parametrize("prec,size,norm", [
    ("f", 1.0, 3.25), ("f", 1.0, -1.1e12), ("f", 3e-29, 9e14), ("f", 1e-10, 2e29),
    ("f", 1e27, 1e-6), ("f", 1e32, 1e9), ("f", 1e-30, 1e-14),
    ("d", 1.0, 3.25), ("d", 1e-250, 1e59), ("d", 1e-270, 1e20)])
@pytest.mark.parametrize("offset", [0, 1, 2, 3])
def test_scale_and_alignment(gpu, prec, size, norm, offset):
    torch, ops = gpu
    grid = _grid(prec, size)
    want = oracle.grid_to_image(grid, norm=norm)
    got = _image(torch, ops, grid, norm, offset)
    err = np.abs(got - want).max() / np.abs(want).max()
    assert err <= (1e-5 if prec == "f" else 1e-12), err
