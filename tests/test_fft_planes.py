"""The fused z/y plane pass: the configuration a convolution reports."""
import pytest

from mini_mdft_amd import FP32, FP64, luc
from mini_mdft_amd import mdft as M

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _conv(n, prec):
    shape, L = (2, n, n), (2.0, 0.3 * n, 0.3 * n)
    g, ag = M.SpatialGrid(shape, L), M.AngularGrid(1, 1)
    tab = luc.synthetic_c(1, 1, luc.nq_for(luc.qmax_of_grid(shape, L), luc.DQ_TIP3P), seed=3)
    return shape, ag, M.Convolution.from_table(tab, g, ag, M.OrientationProjectionMap(ag), prec)


@pytest.mark.parametrize("prec", [FP32, FP64])
@pytest.mark.parametrize("n", [12, 20, 28, 36, 72])
def test_reported_threads(n, prec):
    """Planes compiled with one thread count (256 up to 32, else 512) report it,
    before and after tuning."""
    shape, ag, conv = _conv(n, prec)
    p = torch.zeros((ag.m_np,) + shape, dtype=torch.complex64 if prec == FP32 else torch.complex128, device="cuda")
    for _ in range(2):
        c = conv.fft_config()
        if c["plane"]:
            assert c["plane_threads"] == (256 if n <= 32 else 512)
        conv.execute(p)
