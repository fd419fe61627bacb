"""Blocks past 16 MB take the marching stencil kernels, smaller ones the gathering
kernels: the same operator, node for node.

Bars: complex128 <= 1e-13 and complex64 <= 2e-6 relative against the assembled
operator (as for the gathering kernels), and every column equal bit for bit to the
same column alone, since both kernels form A x through one expression.
"""
import numpy as np
import pytest

from oracle import helmholtz_ref as hr
from problems import small_case

pytestmark = pytest.mark.gpu

import helmholtz_amd as ha  # noqa: E402

# rows of a thread: 2 (complex128) or 4 (complex64); wavefronts straddling rows (n1 < 64),
# a single row or plane beyond the last full run, grids of three nodes an axis
GRIDS = [(33, 17, 9), (64, 5, 6), (65, 3, 4), (3, 6, 4), (3, 130, 4), (129, 6, 3), (11, 3), (3, 12), (64, 33), (131, 67)]


@pytest.mark.parametrize("nodes", GRIDS)
@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("prec", ["c128", "c64"])
def test_march_matches_csr_and_gather(nodes, order, prec):
    dt, bar = (np.complex128, 1e-13) if prec == "c128" else (np.complex64, 2e-6)
    N = int(np.prod(nodes))
    nrhs = (16 << 20) // (N * np.dtype(dt).itemsize) + 2
    M, m, g, w = small_case(nodes, seed=sum(nodes))
    H = hr.get_helmholtz_operator7(M, m, w, g, True, True, order)
    Hg = ha.GetHelmholtzOperator(ha.getRegularMesh(M.domain, M.n), m, w, g, True, True, order)
    rng = np.random.default_rng(8)
    X = np.asfortranarray((rng.standard_normal((N, nrhs)) + 1j * rng.standard_normal((N, nrhs))).astype(dt))
    Y = Hg.apply(X, prec)
    for c in (0, 1, nrhs // 2, nrhs - 1):
        y = H @ X[:, c].astype(np.complex128)
        assert np.linalg.norm(Y[:, c] - y) <= bar * np.linalg.norm(y)
        assert np.array_equal(Hg.apply(np.ascontiguousarray(X[:, c]), prec).ravel(), Y[:, c])


@pytest.mark.parametrize("nodes,levels", [((33, 17, 9), 2), ((65, 33), 2)])
@pytest.mark.parametrize("prec", ["c128", "c64"])
def test_march_in_the_cycle(nodes, levels, prec):
    """Sweeps and residuals of a cycle with three sweeps (separate kernels): a column of a
    large block equals the same column alone, each from its own kind of kernel."""
    M, m, g, w = small_case(nodes, seed=11)
    hp = ha.HelmholtzParam(ha.getRegularMesh(M.domain, M.n), g, m, w, True, True)
    mg = ha.getMGparam(complex, int, levels, 1, 1, 1e-6, "Jac", 0.8, 3, 3, "W", "NoMUMPS", 0.5, 0.0)
    mg.prec = prec
    s = ha.getShiftedLaplacianMultigridSolver(hp, mg, 0.5, "GMRES", 2)
    N = int(np.prod(nodes))
    nrhs = (16 << 20) // (N * (16 if prec == "c128" else 8)) + 2
    rng = np.random.default_rng(9)
    V = rng.standard_normal((N, nrhs)) + 1j * rng.standard_normal((N, nrhs))
    Z = ha.precondition(s, V)
    for c in (0, nrhs - 1):
        z = ha.precondition(s, V[:, [c]])[:, 0]
        assert np.linalg.norm(Z[:, c] - z) <= (1e-13 if prec == "c128" else 1e-5) * np.linalg.norm(z)
