"""The panel form of the dense coarsest inverse, which grids of a bandwidth above 224
take (n1 > 224, in 3-D n1 n2 > 224): every panel width on both sides of its switch (8
columns up to 1024 nodes, 6 to 2048, 4 to 4096, 2 to 8192, 1 to the 10000 nodes that a
coarsest grid may have), the unblocked form (up to 768 nodes) and the first blocked one,
last panels and blocks of every width, and frequencies far above the grid's with no
shift, where rows have to be exchanged.

Columns of the inverse against the sparse operator.  Bar: the residual of a column within
8 N eps |A| |x|, as for the banded form (partial pivoting, growth of order one); |A| is
bounded by sqrt(|A|_1 |A|_inf)."""
import numpy as np
import pytest

from problems import small_case

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


@pytest.mark.parametrize("nodes,omega", [((225, 3), None), ((256, 3), 40.0), ((257, 3), 60.0), ((16, 15, 3), 30.0),
                                         ((17, 17, 3), None), ((16, 16, 4), 30.0), ((342, 3), 60.0), ((25, 9, 5), 30.0),
                                         ((256, 8), None), ((410, 5), 60.0), ((16, 16, 9), 30.0), ((256, 16), 60.0),
                                         ((683, 6), None), ((17, 17, 15), 30.0), ((25, 25, 13), None), ((512, 16), 60.0),
                                         ((2731, 3), 60.0), ((23, 23, 17), 30.0), ((250, 40), None)])
def test_panel_inverse(nodes, omega):
    import scipy.sparse.linalg as sl

    import helmholtz_amd as ha
    from oracle import helmholtz_ref as hr
    M, m, g, w = small_case(nodes, seed=sum(nodes), omega=omega)
    shift = 0.5 if omega is None else 0.0
    hp = ha.HelmholtzParam(ha.getRegularMesh(M.domain, M.n), g, m, w, True, True)
    mg = ha.getMGparam(complex, int, 1, 1, 1, 1e-6, "Jac", 0.8, 2, 2, "V", "NoMUMPS", 0.5, 0.0)
    s = ha.getShiftedLaplacianMultigridSolver(hp, mg, shift, "GMRES", 2)
    N = int(np.prod(nodes))
    A = hr.operator_from_param(hr.HelmholtzParam(M, g + shift * w, m, w, True, True), 2).tocsr()
    cols = np.unique(np.r_[0, 31, 32, N // 2, N - 33, N - 1, np.random.default_rng(2).integers(0, N, 42)])
    V = np.zeros((N, len(cols)), dtype=complex)
    V[cols, np.arange(len(cols))] = 1.0
    Z = ha.precondition(s, V)
    r = np.linalg.norm(A @ Z - V, axis=0)
    norm = np.sqrt(sl.norm(A, 1) * sl.norm(A, np.inf))
    assert np.all(r <= 8 * N * EPS * norm * np.linalg.norm(Z, axis=0))
