"""Arnoldi passes of the complex128 mode at the sizes where their sums change
shape: one RHS and a few on grids of less than, exactly and just over one chunk
of 256 nodes, more chunks than a reduction's 512, and every basis count between
the kernels' 4, 6, 8, 10, 12, 16 and 32 vectors."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# exact arithmetic: with the exact preconditioner (one level) FGMRES converges in
# one step; with none of the shift's help it takes about `inner` steps per
# restart, so every basis count up to `inner` is used
@pytest.mark.parametrize("nodes,inner,nrhs", [((9, 9), 3, 1), ((16, 16), 5, 1), ((257, 3), 7, 2), ((33, 33), 9, 1),
                                              ((33, 33), 11, 3), ((65, 33), 15, 1), ((65, 65), 31, 2),
                                              ((385, 385), 10, 1), ((17, 17, 17), 12, 2)])
def test_solution_and_residual(nodes, inner, nrhs):
    import helmholtz_amd as ha
    import scipy.sparse.linalg as spla
    from oracle import helmholtz_ref as hr
    from problems import small_case
    M, m, g, w = small_case(nodes, seed=11)
    levels = 1 if int(np.prod(nodes)) < 3000 and min(nodes) < 9 else (1 if min(nodes) < 33 and len(nodes) == 2 else 2)
    if nodes == (385, 385):
        levels = 4
    hp = ha.HelmholtzParam(ha.getRegularMesh(M.domain, M.n), g, m, w, True, True)
    mg = ha.getMGparam(complex, int, levels, 1, 200, 1e-10, "Jac", 0.8, 2, 2, "W", "NoMUMPS", 0.5, 0.0)
    s = ha.getShiftedLaplacianMultigridSolver(hp, mg, 0.5, "GMRES", inner)
    N = int(np.prod(nodes))
    rng = np.random.default_rng(2)
    B = rng.standard_normal((N, nrhs)) + 1j * rng.standard_normal((N, nrhs))
    X, s = ha.solveLinearSystem(None, B, s)
    H = hr.get_helmholtz_operator7(M, m, w, g, True, True)
    assert all(v == "converged" for v in s.last_stats["status"])
    res = np.linalg.norm(H @ X - B, axis=0) / np.linalg.norm(B, axis=0)
    # the reported residual is the true one to the rounding of one product
    assert np.all(res <= 1e-10 * (1 + 1e-3))
    assert np.allclose(res, s.last_stats["true_res"], rtol=1e-3)
    if N < 5000:
        x = spla.spsolve(H.tocsc(), B[:, 0])
        assert np.linalg.norm(X[:, 0] - x) <= 1e-7 * np.linalg.norm(x)
    # one column alone: the same bits
    s1 = ha.getShiftedLaplacianMultigridSolver(hp, mg, 0.5, "GMRES", inner)
    x1, s1 = ha.solveLinearSystem(None, B[:, 0], s1)
    assert np.array_equal(x1, X[:, 0])
