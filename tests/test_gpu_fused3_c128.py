"""The fused 3-D legs in complex128 against the separate kernels and the oracle's
cycle, on device blocks used in place.

Bars: 1e-13 between the two forms (the parity bar of the stencil: they differ in the
rounding of diagonal-free sweeps only) and 1e-12 to the oracle (the bar of one cycle).
"""
import numpy as np
import pytest

from oracle import helmholtz_ref as hr, slmg_ref as sr
from problems import small_case

pytestmark = pytest.mark.gpu

import helmholtz_amd as ha  # noqa: E402
from helmholtz_amd import _lib  # noqa: E402
from helmholtz_amd.device import DeviceArray  # noqa: E402
from helmholtz_amd.solver import _ensure_handle  # noqa: E402


# one tile and several, tiles straddling both in-plane edges, one z-run and several
# (many right-hand sides leave one run, one right-hand side takes runs of four planes)
@pytest.mark.parametrize("nodes,nrhs", [((17, 17, 9), 1), ((33, 17, 17), 3), ((65, 49, 33), 2), ((97, 33, 25), 12),
                                        ((29, 57, 65), 1)])
@pytest.mark.parametrize("cycle", ["V", "W"])
def test_legs(nodes, nrhs, cycle):
    M, m, g, w = small_case(nodes, seed=21, neumann=True)
    hp = ha.HelmholtzParam(ha.getRegularMesh(M.domain, M.n), g, m, w, True, True)
    rng = np.random.default_rng(22)
    V = np.asfortranarray(rng.standard_normal((m.size, nrhs)) + 1j * rng.standard_normal((m.size, nrhs)))
    zs = []
    for fused in (True, False):
        mg = ha.getMGparam(complex, int, 3, 1, 1, 1e-6, "Jac", 0.8, 2, 2, cycle, "NoMUMPS", 0.5, 0.0)
        s = ha.getShiftedLaplacianMultigridSolver(hp, mg, 0.5, "GMRES", 2)
        s.MG.fused = fused
        _ensure_handle(s)
        dv, dz = DeviceArray.from_numpy(V), DeviceArray(V.shape, np.complex128)
        _lib.check(_lib.lib().hh_solver_precondition(s._handle, dv.ptr, dz.ptr, nrhs, _lib.HH_DEVICE))
        zs.append(dz.to_numpy())
        assert np.array_equal(dv.to_numpy(), V)
    assert np.linalg.norm(zs[0] - zs[1]) <= 1e-13 * np.linalg.norm(zs[1])
    hier = sr.build_hierarchy(hr.HelmholtzParam(M, g, m, w, True, True), 3, 0.5)
    for c in (0, nrhs - 1):
        zo = sr.vcycle(hier, 0, V[:, c], 0.8, 2, 2, cycle)
        assert np.linalg.norm(zs[0][:, c] - zo) <= 1e-12 * np.linalg.norm(zo)
