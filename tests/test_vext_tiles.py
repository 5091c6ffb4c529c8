"""The external potential's node tiles: ragged ones of 2 x 2 and 4 x 4 nodes,
solvents with and without a site at the origin, off-centre Lennard-Jones sites,
a solute site on a node, and coordinates beyond the range of the bare root."""
import numpy as np
import pytest

import mini_mdft_amd as M

torch = pytest.importorskip("torch")

# charge, sigma, epsilon, x, y, z
ORIGIN = [[-0.8, 3.1, 0.6, 0.0, 0.0, 0.0], [0.4, 1.2, 0.2, 0.8, 0.1, 0.6], [0.4, 0.0, 0.0, -0.8, 0.0, 0.6]]


def _solute(n, L, sites):
    r = np.random.default_rng(4)
    s = np.zeros((sites, 6))
    s[:, 0] = r.uniform(-0.5, 0.5, sites)
    s[:, 1] = np.where(np.arange(sites) % 3 == 2, 0.0, 2.5)
    s[:, 2] = 0.4
    s[:, 3:] = r.uniform(-0.2, 1.2, (sites, 3)) * np.array(L)  # images outside of the box too
    s[0, 3:] = np.array(L) / np.array(n) * np.array([1, 2, 0])  # on a node
    return s


# below and above 2^20 values, sides 1..3 mod 4, and a flat grid
@pytest.mark.gpu
@pytest.mark.parametrize("n,mmax", [((3, 5, 7), 2), ((1, 2, 9), 3), ((17, 14, 19), 5), ((9, 23, 21), 5), ((260, 1, 17), 5)])
@pytest.mark.parametrize("origin", [True, False])
def test_tiles(oracle, n, mmax, origin):
    L = tuple(0.9 * k + 2.0 for k in n)
    sol, solv = _solute(n, L, 5), np.array(ORIGIN if origin else ORIGIN[1:])
    V = M.vext(M.SpatialGrid(n, L), M.AngularGrid(mmax, 2), sol, solv, 300.0).cpu().numpy()
    ref = oracle.vext(n, L, mmax, 2, sol, solv, 300.0)
    # rounding of the sum: some 1e-16 of its largest terms, which the cap bounds
    # only from above
    assert np.abs(V - ref).max() <= 1e-12 * np.abs(ref).max()


@pytest.mark.gpu
def test_far_coordinates():
    """A box of 1e160 A: d^2 overflows, 1/d is 0."""
    n, L = (2, 3, 3), (1e160,) * 3
    sol = np.array([[1.0, 0.0, 0.0, 3e159, 2e159, 1e159]])
    V = M.vext(M.SpatialGrid(n, L), M.AngularGrid(2, 2), sol, np.array(ORIGIN[1:]), 300.0).cpu().numpy()
    assert (V == 0.0).all()
