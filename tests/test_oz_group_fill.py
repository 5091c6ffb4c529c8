"""The OZ pass over groups of stars at the smallest grids that it takes at mmax 5:
one round of groups and two, the last one ragged or full."""
import numpy as np
import pytest

from conftest import rel_err
from mini_mdft_amd import FP32, luc
from mini_mdft_amd import mdft as M

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


# 1728, 1900, 3640 and 4096 stars
@pytest.mark.parametrize("n", [(22, 22, 22), (18, 18, 36), (27, 25, 39), (30, 30, 30)])
def test_execute_matches_oracle(oracle, n):
    L = tuple(0.5 * v for v in n)
    g, ag = M.SpatialGrid(n, L), M.AngularGrid(5, 2)
    tab = luc.synthetic_c(5, 2, luc.nq_for(luc.qmax_of_grid(n, L), luc.DQ_TIP3P), seed=3)
    tab.c = tab.c + 1j * np.roll(tab.c.real, 1, axis=0)  # both parts of every product
    conv = M.Convolution.from_table(tab, g, ag, M.OrientationProjectionMap(ag), FP32)
    ocv = oracle.Conv(n, L, 5, 2, tab.tuples, tab.c, tab.dq)
    r = np.random.default_rng(4)
    p = r.standard_normal((ag.m_np,) + n) + 1j * r.standard_normal((ag.m_np,) + n)
    t = torch.from_numpy(p.astype(np.complex64)).cuda()
    conv.execute(t)
    # FP32 FFTs, rotations and products of at most 18 x 11 terms: the bound of the other FP32 grids
    assert rel_err(t.cpu().numpy(), ocv.execute(p)) < 2e-5
