"""The banded elimination of the dense coarsest inverse at the edges of its blocks and
windows: fewer nodes than a block of 32 columns, one more and one less than whole
blocks, windows of every row count up to the widest (bandwidth 224 in 2-D and 3-D) and
the first bandwidth past it, which takes the panel form.

Bar: the residual of a column within 8 N eps |A| |x|, as for the panel form (partial
pivoting, growth of order one)."""
import numpy as np
import pytest

from problems import small_case

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


@pytest.mark.parametrize("nodes,omega", [((3, 5), None), ((5, 5), 14.0), ((3, 11), None), ((32, 3), 30.0), ((7, 37), None),
                                         ((97, 9), None), ((61, 21), 40.0), ((224, 5), None), ((225, 5), None),
                                         ((14, 16, 5), None), ((15, 15, 5), None), ((3, 4, 50), None)])
def test_band_inverse(nodes, omega):
    import helmholtz_amd as ha
    from oracle import helmholtz_ref as hr
    M, m, g, w = small_case(nodes, seed=sum(nodes), omega=omega)
    shift = 0.5 if omega is None else 0.0  # a large frequency without a shift has to exchange rows
    hp = ha.HelmholtzParam(ha.getRegularMesh(M.domain, M.n), g, m, w, True, True)
    mg = ha.getMGparam(complex, int, 1, 1, 1, 1e-6, "Jac", 0.8, 2, 2, "V", "NoMUMPS", 0.5, 0.0)
    s = ha.getShiftedLaplacianMultigridSolver(hp, mg, shift, "GMRES", 2)
    N = int(np.prod(nodes))
    A = hr.operator_from_param(hr.HelmholtzParam(M, g + shift * w, m, w, True, True), 2).toarray()
    Z = ha.precondition(s, np.eye(N, dtype=complex))
    r = np.linalg.norm(A @ Z - np.eye(N), axis=0)
    assert np.all(r <= 8 * N * EPS * np.linalg.norm(A, 2) * np.linalg.norm(Z, axis=0))
