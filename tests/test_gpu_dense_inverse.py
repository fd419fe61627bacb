"""The dense coarsest inverse on the GPU against NumPy's, through a one-level
solver: its preconditioner is exactly the inverse of the shifted operator."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


# node counts on both sides of each panel width (1024, 2048, 4096 rows), of the
# unblocked form (768), and partial panels and blocks
@pytest.mark.parametrize("nodes", [(3, 3), (8, 4), (9, 7), (17, 33), (32, 24), (37, 21), (33, 31), (32, 32), (41, 25), (13, 13, 7),
                                   (64, 32), (65, 33), (9, 16, 17), (66, 64)])
def test_inverse(nodes):
    import helmholtz_amd as ha
    from oracle import helmholtz_ref as hr
    from problems import small_case
    M, m, g, w = small_case(nodes, seed=sum(nodes))
    hp = ha.HelmholtzParam(ha.getRegularMesh(M.domain, M.n), g, m, w, True, True)
    mg = ha.getMGparam(complex, int, 1, 1, 1, 1e-6, "Jac", 0.8, 2, 2, "V", "NoMUMPS", 0.5, 0.0)
    s = ha.getShiftedLaplacianMultigridSolver(hp, mg, 0.5, "GMRES", 2)
    N = int(np.prod(nodes))
    A = hr.operator_from_param(hr.HelmholtzParam(M, g + 0.5 * w, m, w, True, True), 2).toarray()
    rng = np.random.default_rng(1)
    V = rng.standard_normal((N, 6)) + 1j * rng.standard_normal((N, 6))
    Z = ha.precondition(s, V)
    # Gauss-Jordan with partial pivoting: residual of a column within a modest
    # multiple of n eps |A| |x| (the elimination's growth stays O(1) here)
    r = np.linalg.norm(A @ Z - V, axis=0)
    assert np.all(r <= 8 * N * EPS * np.linalg.norm(A, 2 if N <= 1200 else "fro") * np.linalg.norm(Z, axis=0))


@pytest.mark.parametrize("nodes,omega", [((9, 9), 14.0), ((21, 13), 30.0), ((33, 25), 40.0)])
def test_inverse_needs_pivoting(nodes, omega):
    """Frequencies far above the grid's: the diagonal is small or negative and
    rows have to be exchanged."""
    import helmholtz_amd as ha
    from oracle import helmholtz_ref as hr
    from problems import small_case
    M, m, g, w = small_case(nodes, seed=5, omega=omega)
    hp = ha.HelmholtzParam(ha.getRegularMesh(M.domain, M.n), g, m, w, True, True)
    mg = ha.getMGparam(complex, int, 1, 1, 1, 1e-6, "Jac", 0.8, 2, 2, "V", "NoMUMPS", 0.5, 0.0)
    s = ha.getShiftedLaplacianMultigridSolver(hp, mg, 0.0, "GMRES", 2)
    N = int(np.prod(nodes))
    A = hr.operator_from_param(hr.HelmholtzParam(M, g, m, w, True, True), 2).toarray()
    Z = ha.precondition(s, np.eye(N, dtype=complex))
    assert np.linalg.norm(Z - np.linalg.inv(A)) <= 64 * N * EPS * np.linalg.cond(A) * np.linalg.norm(np.linalg.inv(A))


# one row per wavefront with 1, 2 and 4 right-hand sides (remainders of 4, of 64
# and of the 256 / 512 columns loaded at a time), and the 4 x 4 tiles
@pytest.mark.parametrize("nodes,nrhs", [((3, 3), 1), ((8, 8), 1), ((21, 25), 1), ((33, 17), 1), ((33, 17), 2), ((33, 17), 3),
                                        ((33, 17), 4), ((33, 17), 9), ((23, 23), 7), ((33, 17), 35), ((65, 33), 8),
                                        ((65, 33), 9)])
def test_apply_tiles(nodes, nrhs):
    """Column c of a block does not depend on the tile it falls into: the sums run
    in one order for every tile, so each column equals the same column alone."""
    import helmholtz_amd as ha
    from problems import small_case
    M, m, g, w = small_case(nodes, seed=3)
    hp = ha.HelmholtzParam(ha.getRegularMesh(M.domain, M.n), g, m, w, True, True)
    mg = ha.getMGparam(complex, int, 1, 1, 1, 1e-6, "Jac", 0.8, 2, 2, "V", "NoMUMPS", 0.5, 0.0)
    s = ha.getShiftedLaplacianMultigridSolver(hp, mg, 0.5, "GMRES", 2)
    N = int(np.prod(nodes))
    rng = np.random.default_rng(4)
    V = rng.standard_normal((N, nrhs)) + 1j * rng.standard_normal((N, nrhs))
    Z = ha.precondition(s, V)
    inv = ha.precondition(s, np.eye(N, dtype=complex))
    assert np.linalg.norm(Z - inv @ V) <= 8 * N * EPS * np.linalg.norm(inv) * np.linalg.norm(V)
    for c in {0, nrhs // 2, nrhs - 1}:
        assert np.array_equal(ha.precondition(s, V[:, [c]])[:, 0], Z[:, c])
