"""The Krylov reductions split a right-hand side's nodes the same way however many
right-hand sides are solved together: a column of a large block equals the same column
alone bit for bit, on a fresh solver and on the solver that has just run the block
(whose work buffers hold the larger block).  Blocks so large that 16384 / columns is
less than the grid's own number of chunks; the iteration counts are equal too."""
import numpy as np
import pytest

from problems import small_case

pytestmark = pytest.mark.gpu


def make(nodes, prec, krylov, levels, tol):
    import helmholtz_amd as ha
    M, m, g, w = small_case(nodes, seed=7)
    hp = ha.HelmholtzParam(ha.getRegularMesh(M.domain, M.n), g, m, w, True, True)

    def solver():
        mg = ha.getMGparam(complex, int, levels, 1, 12, tol, "Jac", 0.8, 2, 2, "W", "NoMUMPS", 0.5, 0.0)
        mg.prec = prec
        return ha.getShiftedLaplacianMultigridSolver(hp, mg, 0.5, krylov, 5)
    return solver


@pytest.mark.parametrize("nodes,nrhs,prec,krylov,levels", [((513, 257), 40, "c128", "GMRES", 4),
                                                           ((129, 129), 300, "c128", "GMRES", 3),
                                                           ((129, 129), 300, "c128", "BiCGSTAB", 3),
                                                           ((129, 129), 600, "c64", "GMRES", 3)])
def test_column_of_a_large_block(nodes, nrhs, prec, krylov, levels):
    import helmholtz_amd as ha
    fresh = make(nodes, prec, krylov, levels, 1e-2)
    N = int(np.prod(nodes))
    rng = np.random.default_rng(11)
    B = np.asfortranarray(rng.standard_normal((N, nrhs)) + 1j * rng.standard_normal((N, nrhs)))
    s = fresh()
    X, _ = ha.solveLinearSystem(None, B, s)
    iters = s.last_stats["iters"].copy()
    for c in (0, nrhs // 2, nrhs - 1):
        alone = fresh()
        for one in (s, alone):
            x, _ = ha.solveLinearSystem(None, B[:, c], one)
            assert np.array_equal(x, X[:, c])
            assert one.last_stats["iters"][0] == iters[c]
