"""proj2angl with a wave per mu2 (FP64 and FP32): each of its angular grids, last
row blocks of 1, 2, 3 and 63 rows, alone and fused with get_delta_f."""
import numpy as np
import pytest

from conftest import rel_err
from mini_mdft_amd import FP32, FP64, luc
from mini_mdft_amd import mdft as M

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

GRIDS = [(1, 1), (1, 2), (2, 1), (2, 2), (3, 1), (3, 2), (4, 2), (5, 2), (6, 2)]


@pytest.mark.parametrize("mmax,mrso", GRIDS)
@pytest.mark.parametrize("n", [(1, 1, 1), (1, 2, 33), (63, 1, 1), (67, 3, 5)])
@pytest.mark.parametrize("prec,tol", [(FP64, 1e-13), (FP32, 2e-6)])
def test_proj2angl(oracle, n, mmax, mrso, prec, tol):
    """Against the oracle, with the bounds of the other grids."""
    g, ag = M.SpatialGrid(n, (1.0, 1.0, 1.0)), M.AngularGrid(mmax, mrso)
    opt = M.OrientationProjectionTransform(g, ag, M.OrientationProjectionMap(ag), prec)
    r = np.random.default_rng(3)
    p = r.standard_normal((ag.m_np,) + n) + 1j * r.standard_normal((ag.m_np,) + n)
    o = torch.zeros((g.N, ag.m_ntheta, ag.m_nphi, ag.m_npsi), dtype=opt.real_dtype, device="cuda")
    opt.proj2angl(torch.from_numpy(p).to(opt.complex_dtype).cuda(), o)
    assert rel_err(o.cpu().numpy(), oracle.proj2angl(p, mmax, mrso)) < tol


@pytest.mark.parametrize("mmax,mrso", GRIDS[1:])
@pytest.mark.parametrize("n", [(5, 13, 1), (8, 8, 9), (3, 5, 7)])
@pytest.mark.parametrize("prec", [FP64, FP32])
def test_fused_equals_stages(n, mmax, mrso, prec):
    """df and ff of the fused evaluation, in both channel orders, and with the
    column sums of the other kernel, against the stages one by one."""
    L = tuple(0.5 * v for v in n)
    g, ag = M.SpatialGrid(n, L), M.AngularGrid(mmax, mrso)
    mp = M.OrientationProjectionMap(ag)
    tab = luc.synthetic_c(mmax, mrso, luc.nq_for(luc.qmax_of_grid(n, L), luc.DQ_TIP3P), seed=3)
    conv = M.Convolution.from_table(tab, g, ag, mp, prec)
    opt = M.OrientationProjectionTransform(g, ag, mp, prec)
    rho0, pref = 0.00084, -5.0
    xi = torch.empty((g.N, ag.m_no), dtype=opt.real_dtype, device="cuda")
    M.fill_uniform(xi, 5, 0.7, 1.3)
    drho, vexc, df = (torch.empty_like(xi) for _ in range(3))
    M.get_delta_rho(xi, drho, rho0)
    p = torch.empty((ag.m_np,) + n, dtype=opt.complex_dtype, device="cuda")
    opt.angl2proj(drho, p)
    conv.execute(p)
    opt.proj2angl(p, vexc)
    ff = M.get_delta_f(xi, vexc, torch.from_numpy(ag.m_w).cuda(), df, rho0, pref)
    ref = df.double().cpu().numpy()
    tol = 1e-12 if prec == FP64 else 2e-5  # a whole evaluation's rounding
    solver = M.Solver(conv, rho0, pref, prec)
    has = solver.compact  # FP64 at mmax 6 has one order only
    for compact, mean in ((has, False), (False, False), (has, True)):
        solver.set_compact(compact)
        solver.set_mean_fp64(mean)
        df.zero_()
        assert abs(solver.energy_cproj(xi, df) - ff) <= tol * abs(ff)
        assert rel_err(df.double().cpu().numpy(), ref) < tol
