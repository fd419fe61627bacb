"""Jac-GMRES smoothing in three launches per step: one cycle against the oracle at
the sizes where its chunks change (fewer than 256 nodes, one node per thread, more
than 256 chunks of 256), every step count's basis, 2-D and 3-D, several RHS with a
zero column, and one column alone (the same bits)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nodes,pre,post", [((9, 9), 1, 2), ((17, 15), 2, 3), ((33, 17), 8, 1), ((65, 33), 2, 2),
                                            ((129, 65), 4, 2), ((385, 193), 2, 1), ((17, 9, 9), 2, 2), ((33, 17, 17), 3, 5)])
@pytest.mark.parametrize("cycle", ["V", "K"])
def test_cycle(nodes, pre, post, cycle):
    import helmholtz_amd as ha
    from oracle import helmholtz_ref as hr, slmg_ref as sr
    from problems import small_case
    M, m, g, w = small_case(nodes, seed=21, neumann=True)
    levels = 4 if nodes[0] > 300 else (3 if min(nodes) > 16 and len(nodes) == 2 else 2)
    hp = ha.HelmholtzParam(ha.getRegularMesh(M.domain, M.n), g, m, w, True, True)
    rng = np.random.default_rng(22)
    V = np.asfortranarray(rng.standard_normal((m.size, 3)) + 1j * rng.standard_normal((m.size, 3)))
    V[:, 1] = 0.0

    def solver(prec):
        mg = ha.getMGparam(complex, int, levels, 1, 10, 1e-6, "Jac-GMRES", 0.8, pre, post, cycle, "NoMUMPS", 0.5, 0.0)
        mg.prec = prec
        return ha.getShiftedLaplacianMultigridSolver(hp, mg, 0.5, "GMRES", 2)

    Z = ha.precondition(solver("c128"), V)
    hier = sr.build_hierarchy(hr.HelmholtzParam(M, g, m, w, True, True), levels, 0.5)
    zo = sr.vcycle(hier, 0, V[:, 0], 0.8, pre, post, cycle, 0, "Jac-GMRES")
    # the least-squares steps amplify rounding: the bar of the solver's own cycle test
    assert np.linalg.norm(Z[:, 0] - zo) <= 1e-10 * np.linalg.norm(zo)
    assert not np.any(Z[:, 1])
    assert np.array_equal(ha.precondition(solver("c128"), V[:, [2]])[:, 0], Z[:, 2])
    Zf = ha.precondition(solver("c64"), V)
    assert np.linalg.norm(Zf[:, 0] - zo) <= 2e-4 * np.linalg.norm(zo)
