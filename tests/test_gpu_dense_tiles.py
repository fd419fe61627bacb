"""Tiles of the complex128 coarsest apply: blocks of 2 and 4 rows with 1, 2, 4 and 8
right-hand sides, remainders of each, and inverses of fewer columns than a block's
threads.  A block's column equals the same column alone bit for bit (one order of
additions for every tile); the sum itself is held to 8 N eps as for the other tiles."""
import numpy as np
import pytest

from problems import small_case

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


@pytest.mark.parametrize("nodes,nrhs", [((3, 3), 3), ((16, 16), 2), ((257, 5), 5), ((65, 33), 5), ((65, 33), 8),
                                        ((65, 33), 11), ((43, 41), 16), ((97, 45), 1), ((97, 45), 2), ((97, 45), 5)])
def test_tiles(nodes, nrhs):
    import helmholtz_amd as ha
    M, m, g, w = small_case(nodes, seed=6)
    hp = ha.HelmholtzParam(ha.getRegularMesh(M.domain, M.n), g, m, w, True, True)
    mg = ha.getMGparam(complex, int, 1, 1, 1, 1e-6, "Jac", 0.8, 2, 2, "V", "NoMUMPS", 0.5, 0.0)
    s = ha.getShiftedLaplacianMultigridSolver(hp, mg, 0.5, "GMRES", 2)
    N = int(np.prod(nodes))
    rng = np.random.default_rng(4)
    V = rng.standard_normal((N, nrhs)) + 1j * rng.standard_normal((N, nrhs))
    Z = ha.precondition(s, V)
    if N <= 2200:  # the inverse itself, from unit vectors
        inv = ha.precondition(s, np.eye(N, dtype=complex))
        assert np.linalg.norm(Z - inv @ V) <= 8 * N * EPS * np.linalg.norm(inv) * np.linalg.norm(V)
    for c in {0, nrhs // 2, nrhs - 1}:
        z = ha.precondition(s, V[:, [c]])[:, 0]
        assert np.array_equal(z, Z[:, c])
