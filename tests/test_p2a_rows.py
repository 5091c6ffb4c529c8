"""Last row blocks of proj2angl that are shorter than one step of a block: which
rows its threads read (on the CPU), and the fused evaluation there."""
import os
import subprocess

import pytest

from conftest import rel_err
from mini_mdft_amd import FP32, FP64, luc
from mini_mdft_amd import mdft as M

torch = pytest.importorskip("torch")

HERE = os.path.dirname(os.path.abspath(__file__))


def test_rows_exist(tmp_path):
    exe = str(tmp_path / "rows")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", os.path.join(HERE, "..", "mini_mdft_amd", "csrc"), "-o",
                    exe, os.path.join(HERE, "cpp", "test_rows.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


# one step of a block holds 14 rows at (1, 1), 16 at (1, 2), 6 at (3, 2), 3 at (5, 2), 2 at (6, 2)
@pytest.mark.gpu
@pytest.mark.parametrize("mmax,mrso", [(1, 1), (1, 2), (3, 2), (5, 2), (6, 2)])
@pytest.mark.parametrize("n", [(1, 1, 3), (1, 1, 13), (5, 13, 1), (2, 3, 11)])  # last blocks of 3, 13, 1 and 2 rows
@pytest.mark.parametrize("prec,tol", [(FP64, 1e-12), (FP32, 2e-5)])  # a whole evaluation's rounding
def test_fused(n, mmax, mrso, prec, tol):
    """df and ff against the stages one by one, whose proj2angl reads no xi (the
    oracle would differ from FP32 by the latter's chop of gamma at 2^-23)."""
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
    solver = M.Solver(conv, rho0, pref, prec)
    for mean in (False, True):
        solver.set_mean_fp64(mean)
        df.zero_()
        assert abs(solver.energy_cproj(xi, df) - ff) <= tol * abs(ff)
        assert rel_err(df.double().cpu().numpy(), ref) < tol
