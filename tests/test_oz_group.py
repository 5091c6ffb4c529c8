"""The OZ pass over groups of stars (FP32, mmax 4 and 5 from a few thousand
stars on) against the FP64 oracle, at grids where its groups are ragged: odd
sides, sides without a Nyquist plane, a last group of fewer than eight stars."""
import numpy as np
import pytest

from conftest import rel_err
from mini_mdft_amd import FP32, MIXED_X6F, luc
from mini_mdft_amd import mdft as M

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

MRSO = 2
# (grid, mmax): 5491, 5600, 4913 and 21168 stars
CASES = [((33, 36, 32), 5), ((26, 39, 39), 5), ((32, 32, 32), 5), ((54, 55, 52), 4)]


def _conv(n, mmax, seed, precision):
    L = tuple(0.5 * v for v in n)
    g, ag = M.SpatialGrid(n, L), M.AngularGrid(mmax, MRSO)
    tab = luc.synthetic_c(mmax, MRSO, luc.nq_for(luc.qmax_of_grid(n, L), luc.DQ_TIP3P), seed=seed)
    # a complex c(q): both parts of every product
    tab.c = tab.c + 1j * np.roll(tab.c.real, 1, axis=0)
    return L, g, ag, tab, M.Convolution.from_table(tab, g, ag, M.OrientationProjectionMap(ag), precision)


@pytest.mark.parametrize("n,mmax", CASES)
def test_execute_matches_oracle(oracle, n, mmax):
    L, g, ag, tab, conv = _conv(n, mmax, 3, FP32)
    ocv = oracle.Conv(n, L, mmax, MRSO, tab.tuples, tab.c, tab.dq)
    r = np.random.default_rng(4)
    p = r.standard_normal((ag.m_np,) + n) + 1j * r.standard_normal((ag.m_np,) + n)
    t = torch.from_numpy(p.astype(np.complex64)).cuda()
    conv.execute(t)
    # FP32 FFTs, rotations and products of at most 18 x 11 terms: the bound of the other FP32 grids
    assert rel_err(t.cpu().numpy(), ocv.execute(p)) < 2e-5


@pytest.mark.parametrize("n", [(32, 32, 32), (36, 32, 35)])
def test_fields_of_a_batch_and_channel_orders(n):
    """Three fields together are bitwise each alone, and the compact channel
    order changes df by rounding only (FP32 values of both orders)."""
    L, g, ag, tab, conv = _conv(n, 5, 5, MIXED_X6F)
    n0 = M.SOLVENTS["spce"]["n0"]
    solver = M.Solver(conv, M.rho0_of(n0, MRSO), M.prefactor_of(298.15, MRSO, n0), MIXED_X6F, capacity=3)
    xi = torch.empty((3, g.N, ag.m_no), dtype=torch.float32, device="cuda")
    M.fill_uniform(xi, 11, 0.9, 1.1)
    df, one = torch.empty_like(xi), torch.empty_like(xi[0])
    ff = solver.energy_cproj_batch(xi, df)
    for j in range(3):
        assert solver.energy_cproj(xi[j], one) == ff[j]
        assert torch.equal(one, df[j])
    assert solver.compact
    solver.set_compact(False)
    solver.energy_cproj(xi[2], one)
    assert rel_err(df[2].double().cpu().numpy(), one.double().cpu().numpy()) < 2e-6
