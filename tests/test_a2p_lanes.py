"""angl2proj of many points (one per lane) on each of its angular grids, with a
last block of 1, 32 and 63 rows, and its fields alone and in a batch."""
import numpy as np
import pytest

from conftest import rel_err
from mini_mdft_amd import FP32, FP64, luc
from mini_mdft_amd import mdft as M

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# 7681, 7776, 7743 and 8000 points
CASES = [((1, 1, 7681), 2, 1), ((24, 18, 18), 2, 2), ((29, 3, 89), 3, 1), ((1, 7681, 1), 3, 2), ((20, 20, 20), 4, 2),
         ((29, 89, 3), 5, 2), ((7681, 1, 1), 6, 2)]


@pytest.mark.parametrize("n,mmax,mrso", CASES)
@pytest.mark.parametrize("prec,tol", [(FP64, 1e-13), (FP32, 2e-6)])
def test_angl2proj(oracle, n, mmax, mrso, prec, tol):
    """Against the oracle, with the bounds of the small grids."""
    ag = M.AngularGrid(mmax, mrso)
    g = M.SpatialGrid(n, (1.0, 1.0, 1.0))
    opt = M.OrientationProjectionTransform(g, ag, M.OrientationProjectionMap(ag), prec)
    o = np.random.default_rng(2).random((g.N, ag.m_ntheta, ag.m_nphi, ag.m_npsi))
    p = torch.zeros((ag.m_np,) + n, dtype=opt.complex_dtype, device="cuda")
    opt.angl2proj(torch.from_numpy(o).to(opt.real_dtype).cuda(), p)
    assert rel_err(p.cpu().numpy(), oracle.angl2proj(o, n, mmax, mrso)) < tol


# below the line alone and above it together, and above it alone
@pytest.mark.parametrize("n,mmax", [((16, 16, 16), 3), ((20, 20, 20), 5)])
@pytest.mark.parametrize("prec", [FP64, FP32])
def test_fields_of_a_batch_and_channel_orders(n, mmax, prec):
    """A field is bitwise the same alone and in a batch, and in both channel
    orders to rounding."""
    L = tuple(0.5 * v for v in n)
    g, ag = M.SpatialGrid(n, L), M.AngularGrid(mmax, 2)
    tab = luc.synthetic_c(mmax, 2, luc.nq_for(luc.qmax_of_grid(n, L), luc.DQ_TIP3P), seed=3)
    conv = M.Convolution.from_table(tab, g, ag, M.OrientationProjectionMap(ag), prec)
    n0 = M.SOLVENTS["spce"]["n0"]
    solver = M.Solver(conv, M.rho0_of(n0, 2), M.prefactor_of(298.15, 2, n0), prec, capacity=3)
    xi = torch.empty((3, g.N, ag.m_no), dtype=torch.float64 if prec == FP64 else torch.float32, device="cuda")
    M.fill_uniform(xi, 11, 0.9, 1.1)
    df, one = torch.empty_like(xi), torch.empty_like(xi[0])
    ff = solver.energy_cproj_batch(xi, df)
    for j in range(3):
        assert solver.energy_cproj(xi[j], one) == ff[j]
        assert torch.equal(one, df[j])
    solver.set_compact(False)
    solver.energy_cproj(xi[2], one)
    assert rel_err(df[2].double().cpu().numpy(), one.double().cpu().numpy()) < (1e-13 if prec == FP64 else 2e-6)
