"""The spread operator's marching kernels against the oracle's CSR: grids of one
and several tiles (30 x 14 owned nodes), remainders of one and two nodes, z-runs
of one, two and many planes, rows of the 2-D march, the transpose, the shift and
a complex64 input (through an adjoint solve's and a c64 solve's operator)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nodes", [(3, 3, 3), (5, 17, 3), (30, 14, 5), (31, 15, 8), (32, 16, 9), (61, 29, 16), (33, 43, 51),
                                   (3, 3), (5, 129), (64, 5), (65, 33), (257, 17)])
@pytest.mark.parametrize("beta", [(1.0, 1.0), (0.7, 0.7), (0.4, 0.85)])
def test_apply_and_adjoint(nodes, beta):
    import helmholtz_amd as ha
    from oracle import helmholtz_ref as hr
    from problems import small_case
    M, m, g, w = small_case(nodes, seed=sum(nodes))
    b = beta[0] if len(nodes) == 2 else np.array(beta)
    A = hr.get_helmholtz_operator_ho(M, m, w, g, True, True, b)
    hp = ha.HelmholtzParam(ha.getRegularMesh(M.domain, M.n), g, m, w, True, True)
    H = ha.GetHelmholtzOperatorHO(hp, b)
    N = int(np.prod(nodes))
    rng = np.random.default_rng(3)
    X = np.asfortranarray(rng.standard_normal((N, 3)) + 1j * rng.standard_normal((N, 3)))
    want = A @ X
    assert np.linalg.norm(H @ X - want) <= 1e-13 * np.linalg.norm(want)
    Hs = H + ha.GetHelmholtzShiftOP(m, w, 0.5)
    want = want + (0.5j * w * w * m)[:, None] * X
    assert np.linalg.norm(Hs @ X - want) <= 1e-13 * np.linalg.norm(want)


@pytest.mark.parametrize("nodes,levels", [((33, 41), 2), ((17, 33, 17), 2)])
@pytest.mark.parametrize("prec", ["c128", "c64"])
def test_solves_use_residual_and_transpose(nodes, levels, prec):
    import helmholtz_amd as ha
    from oracle import helmholtz_ref as hr
    from problems import small_case
    M, m, g, w = small_case(nodes, seed=8)
    b = 0.8 if len(nodes) == 2 else np.array([0.8, 0.9])
    A = hr.get_helmholtz_operator_ho(M, m, w, g, True, True, b)
    hp = ha.HelmholtzParam(ha.getRegularMesh(M.domain, M.n), g, m, w, True, True)
    H = ha.GetHelmholtzOperatorHO(hp, b)
    mg = ha.getMGparam(complex, int, levels, 1, 200, 1e-9, "Jac", 0.8, 2, 2, "W", "NoMUMPS", 0.5, 0.0)
    mg.prec = prec
    s = ha.getShiftedLaplacianMultigridSolver(hp, mg, 0.5, "GMRES", 12)
    rng = np.random.default_rng(9)
    B = rng.standard_normal((m.size, 2)) + 1j * rng.standard_normal((m.size, 2))
    for tr, Op in ((0, A), (1, A.conj().T)):
        X, s = ha.solveLinearSystem(H, B, s, tr)
        assert np.all(np.linalg.norm(Op @ X - B, axis=0) <= 1e-9 * (1 + 1e-3) * np.linalg.norm(B, axis=0))
