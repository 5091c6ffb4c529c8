"""angl2proj with a point per lane from the smallest fields it takes at mmax 2 to
4 on, with a last block of 1, 32 and 63 rows."""
import numpy as np
import pytest

from conftest import rel_err
from mini_mdft_amd import FP32, FP64
from mini_mdft_amd import mdft as M

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# 10241, 10272, 10303, 10240 and (FP32 at mmax 2) 16385 points
CASES = [((1, 1, 10241), 2, 1, FP64), ((3, 32, 107), 2, 2, FP64), ((10303, 1, 1), 3, 1, FP64), ((40, 16, 16), 3, 2, FP64),
         ((11, 7, 133), 4, 2, FP64), ((1, 10303, 1), 3, 1, FP32), ((107, 3, 32), 3, 2, FP32), ((1, 1, 10241), 4, 2, FP32),
         ((5, 29, 113), 2, 1, FP32), ((113, 145, 1), 2, 2, FP32)]


@pytest.mark.parametrize("n,mmax,mrso,prec", CASES)
def test_angl2proj(oracle, n, mmax, mrso, prec):
    """Against the oracle, with the bounds of the small grids."""
    ag = M.AngularGrid(mmax, mrso)
    g = M.SpatialGrid(n, (1.0, 1.0, 1.0))
    opt = M.OrientationProjectionTransform(g, ag, M.OrientationProjectionMap(ag), prec)
    o = np.random.default_rng(2).random((g.N, ag.m_ntheta, ag.m_nphi, ag.m_npsi))
    p = torch.zeros((ag.m_np,) + n, dtype=opt.complex_dtype, device="cuda")
    opt.angl2proj(torch.from_numpy(o).to(opt.real_dtype).cuda(), p)
    assert rel_err(p.cpu().numpy(), oracle.angl2proj(o, n, mmax, mrso)) < (1e-13 if prec == FP64 else 2e-6)
