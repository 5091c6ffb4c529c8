"""Fused proj2angl of FP32 at mmax 5 on both sides of the 2^17 points from which a
field goes to the single-wave kernel."""
import pytest

from conftest import rel_err
from mini_mdft_amd import FP32, luc
from mini_mdft_amd import mdft as M

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n", [(64, 64, 32), (63, 64, 32), (65, 55, 42)])  # the last one ends in a short row block
def test_sides(n):
    """df and ff against the stages one by one; two fields are bitwise each alone."""
    L = tuple(0.5 * v for v in n)
    g, ag = M.SpatialGrid(n, L), M.AngularGrid(5, 2)
    mp = M.OrientationProjectionMap(ag)
    tab = luc.synthetic_c(5, 2, luc.nq_for(luc.qmax_of_grid(n, L), luc.DQ_TIP3P), seed=3)
    conv = M.Convolution.from_table(tab, g, ag, mp, FP32)
    opt = M.OrientationProjectionTransform(g, ag, mp, FP32)
    rho0, pref = 0.00084, -5.0
    nb = 2 if g.N % 64 == 0 else 1
    xi = torch.empty((nb, g.N, ag.m_no), dtype=torch.float32, device="cuda")
    M.fill_uniform(xi, 5, 0.7, 1.3)
    drho, vexc, ref = (torch.empty_like(xi[0]) for _ in range(3))
    M.get_delta_rho(xi[0], drho, rho0)
    p = torch.empty((ag.m_np,) + n, dtype=opt.complex_dtype, device="cuda")
    opt.angl2proj(drho, p)
    conv.execute(p)
    opt.proj2angl(p, vexc)
    ff = M.get_delta_f(xi[0], vexc, torch.from_numpy(ag.m_w).cuda(), ref, rho0, pref)
    solver = M.Solver(conv, rho0, pref, FP32, capacity=nb)
    df, one = torch.empty_like(xi), torch.empty_like(xi[0])
    for mean in (False, True):
        solver.set_mean_fp64(mean)
        got = solver.energy_cproj_batch(xi, df)
        # a whole evaluation's rounding
        assert abs(got[0] - ff) <= 2e-5 * abs(ff)
        assert rel_err(df[0].double().cpu().numpy(), ref.double().cpu().numpy()) < 2e-5
        for j in range(nb):
            assert solver.energy_cproj(xi[j], one) == got[j]
            assert torch.equal(one, df[j])
