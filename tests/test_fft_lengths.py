"""The FFT's compiled lengths (8 .. 128, primes up to 13): each radix, tiles with
missing columns, square planes with primes above 5, and the lengths next to the
range, which the run-time kernels take."""
import math

import numpy as np
import pytest

from mini_mdft_amd import luc
from mini_mdft_amd import mdft as M

from conftest import rel_err

torch = pytest.importorskip("torch")

# x, y and z lengths: the smallest and largest compiled ones, 7 and 130 beside
# them, strides that are no multiple of 16 or 32 or fall short of a tile, and
# square planes of 14, 26, 33, 49, 77, 99 and 128 (in LDS once or twice)
SHAPES = [(1, 8, 9, 11), (2, 13, 14, 14), (1, 7, 26, 26), (1, 22, 33, 33), (2, 12, 49, 49), (1, 16, 77, 77),
          (1, 9, 99, 99), (1, 128, 5, 3), (1, 125, 1, 9), (1, 126, 1, 7), (1, 130, 2, 8), (3, 21, 45, 50),
          (1, 96, 10, 10), (1, 11, 121, 13), (3, 2, 128, 128),
          (2, 3, 64, 64), (1, 2, 80, 80), (2, 2, 42, 42)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dt", ["c64", "c128"])
def test_lengths(shape, dt):
    """The default transform against numpy, in both directions, and bitwise
    against per-axis tiles of the run-time kernels (width 4) and both compiled
    strided widths."""
    r = np.random.default_rng(1)
    x = r.standard_normal(shape) + 1j * r.standard_normal(shape)
    t = torch.from_numpy(x).to(torch.complex64 if dt == "c64" else torch.complex128).cuda()
    # rounding of log2(N) butterfly levels
    tol = (2e-6 if dt == "c64" else 1e-13) * math.log2(np.prod(shape[1:]))
    for sign in (-1, 1):
        y = t.clone()
        M.fft3d(y, sign)
        exp = np.fft.fftn(x, axes=(-3, -2, -1)) if sign < 0 else np.fft.ifftn(x, axes=(-3, -2, -1), norm="forward")
        assert rel_err(y.cpu().numpy(), exp) < tol
        for w in (4, 16, 32):
            z = t.clone()
            M.fft3d_config(z, sign, False, wz=4, wy=w, wx=w)
            assert torch.equal(z, y), w


@pytest.mark.gpu
@pytest.mark.parametrize("n", [49, 81, 100, 128])
@pytest.mark.parametrize("dt,tol", [("c64", 2e-5), ("c128", 1e-11)])
def test_tuned_planes(oracle, n, dt, tol):
    """Square planes up to the largest, in the configuration that a convolution
    tunes, with the bounds of the other convolutions."""
    prec = M.FP32 if dt == "c64" else M.FP64
    shape, L = (2, n, n), (2.0, 0.3 * n, 0.3 * n)
    g, ag = M.SpatialGrid(shape, L), M.AngularGrid(1, 1)
    tab = luc.synthetic_c(1, 1, luc.nq_for(luc.qmax_of_grid(shape, L), luc.DQ_TIP3P), seed=3)
    conv = M.Convolution.from_table(tab, g, ag, M.OrientationProjectionMap(ag), prec)
    ocv = oracle.Conv(shape, L, 1, 1, tab.tuples, tab.c, tab.dq)
    r = np.random.default_rng(2)
    p = r.standard_normal((ag.m_np,) + shape) + 1j * r.standard_normal((ag.m_np,) + shape)
    t = torch.from_numpy(p).to(torch.complex64 if dt == "c64" else torch.complex128).cuda()
    conv.execute(t)
    assert rel_err(t.cpu().numpy(), ocv.execute(p)) < tol
