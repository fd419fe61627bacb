"""The complex64 coarsest apply on MFMA: matrices whose 2 n real columns end in a part of
a group of 16 (and in half a load of four), right-hand sides short of a tile of 16, one
and two groups in flight (few and many blocks).  A column does not depend on its block's
size (same order of additions), and the apply is within 4 (2 n) eps32 |A^-1| |r| of the
complex128 solver's."""
import numpy as np
import pytest

from problems import small_case

pytestmark = pytest.mark.gpu

import helmholtz_amd as ha  # noqa: E402


@pytest.mark.parametrize("nodes,nrhs", [((3, 3), 1), ((5, 5), 17), ((16, 16), 16), ((33, 17), 48), ((33, 17), 256),
                                        ((33, 17), 193), ((13, 13, 7), 3), ((21, 13), 31)])
def test_apply(nodes, nrhs):
    M, m, g, w = small_case(nodes, seed=4)
    hp = ha.HelmholtzParam(ha.getRegularMesh(M.domain, M.n), g, m, w, True, True)
    N = int(np.prod(nodes))
    rng = np.random.default_rng(2)
    V = (rng.standard_normal((N, nrhs)) + 1j * rng.standard_normal((N, nrhs))).astype(np.complex64)
    out = {}
    for prec in ("c64", "c128"):
        mg = ha.getMGparam(complex, int, 1, 1, 1, 1e-6, "Jac", 0.8, 2, 2, "V", "NoMUMPS", 0.5, 0.0)
        mg.prec = prec
        s = ha.getShiftedLaplacianMultigridSolver(hp, mg, 0.5, "GMRES", 2)
        out[prec] = ha.precondition(s, V)
        inv = ha.precondition(s, np.eye(N, dtype=complex)) if prec == "c128" else None
        for c in {0, nrhs // 2, nrhs - 1}:
            assert np.array_equal(ha.precondition(s, V[:, [c]])[:, 0], out[prec][:, c])
    err = np.linalg.norm(out["c64"] - out["c128"], axis=0)
    assert np.all(err <= 4 * 2 * N * np.finfo(np.float32).eps * np.linalg.norm(inv) * np.linalg.norm(V, axis=0))
