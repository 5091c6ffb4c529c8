"""The FP64 mean mode at mmax 6, whose rows of one theta are longer than a wave:
it writes every orientation of df, as the evaluation without it does."""
import pytest

from conftest import rel_err
from mini_mdft_amd import FP32, MIXED_X6, MIXED_X6F, luc
from mini_mdft_amd import mdft as M

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("prec", [FP32, MIXED_X6, MIXED_X6F])
@pytest.mark.parametrize("n", [(5, 13, 1), (8, 8, 9)])
def test_on_and_off(n, prec):
    L = tuple(0.5 * v for v in n)
    g, ag = M.SpatialGrid(n, L), M.AngularGrid(6, 2)
    tab = luc.synthetic_c(6, 2, luc.nq_for(luc.qmax_of_grid(n, L), luc.DQ_TIP3P), seed=3)
    conv = M.Convolution.from_table(tab, g, ag, M.OrientationProjectionMap(ag), prec)
    solver = M.Solver(conv, 0.00084, -5.0, prec)
    xi = torch.empty((g.N, ag.m_no), dtype=solver.real_dtype, device="cuda")
    M.fill_uniform(xi, 5, 0.7, 1.3)
    out = []
    for on in (False, True):
        solver.set_mean_fp64(on)
        df = torch.zeros_like(xi)
        out.append((solver.energy_cproj(xi, df), df.double().cpu().numpy()))
    # the mode changes ff by the rounding of an FP32 evaluation, df not at all
    # (FP32: another kernel's rounding)
    assert abs(out[1][0] - out[0][0]) <= 2e-5 * abs(out[0][0])
    assert rel_err(out[1][1], out[0][1]) < 2e-6
