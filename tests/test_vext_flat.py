"""The external potential's node tiles where a grid has few nodes along y or z:
each tile of 1, 2 or 4 by 1, 2 or 4 nodes, whole and ragged."""
import numpy as np
import pytest

import mini_mdft_amd as M

torch = pytest.importorskip("torch")

SOLV = np.array([[-0.8, 3.1, 0.6, 0.0, 0.0, 0.0], [0.4, 1.2, 0.2, 0.8, 0.1, 0.6], [0.4, 0.0, 0.0, -0.8, 0.0, 0.6]])

# ny, nz of the 1 x 1 .. 4 x 4 tiles in turn, on rows long enough for 2^20 values
# and on short ones
SIDES = [(1, 1), (1, 5), (1, 7), (9, 1), (5, 5), (2, 7), (7, 1), (3, 5), (4, 7), (10, 3)]


@pytest.mark.gpu
@pytest.mark.parametrize("sides", SIDES)
@pytest.mark.parametrize("values", [2**20, 2**15])
def test_tiles(oracle, sides, values):
    ny, nz = sides
    n = (-(-values // (330 * ny * nz)), ny, nz)
    L = tuple(0.9 * k + 2.0 for k in n)
    r = np.random.default_rng(4)
    sol = np.zeros((4, 6))
    sol[:, 0] = r.uniform(-0.5, 0.5, 4)
    sol[:, 1] = [2.5, 0.0, 2.5, 2.5]
    sol[:, 2] = 0.4
    sol[:, 3:] = r.uniform(-0.2, 1.2, (4, 3)) * np.array(L)
    V = M.vext(M.SpatialGrid(n, L), M.AngularGrid(5, 2), sol, SOLV, 300.0).cpu().numpy()
    ref = oracle.vext(n, L, 5, 2, sol, SOLV, 300.0)
    # rounding of the sum: some 1e-16 of its largest terms, which the cap bounds
    # only from above
    assert np.abs(V - ref).max() <= 1e-12 * np.abs(ref).max()


@pytest.mark.gpu
def test_side_without_a_quotient():
    """A box of 1e-309 A, whose reciprocal overflows: d^2 is infinite, 1/d is 0."""
    n, L = (2, 3, 3), (1e-309,) * 3
    sol = np.array([[1.0, 0.0, 0.0, 3.0, 2.0, 1.0]])
    V = M.vext(M.SpatialGrid(n, L), M.AngularGrid(2, 2), sol, SOLV[1:2], 300.0).cpu().numpy()
    assert (V == 0.0).all()
