"""hh_solver_precondition on device blocks: where they lie, and through the Krylov
storage where V and Z overlap or Z is not aligned to a value; the same bits as
from host blocks, V left as it was."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("nodes,levels,cycle,relax", [((65, 33), 3, "W", "Jac"), ((33, 17), 2, "V", "Jac"), ((17, 9), 1, "V", "Jac"),
                                                      ((33, 33), 3, "K", "Jac-GMRES"), ((33, 17, 17), 2, "W", "Jac"),
                                                      ((9, 9), 2, "V", "Jac")])
def test_device_blocks(prec, nodes, levels, cycle, relax):
    import helmholtz_amd as ha
    from helmholtz_amd import _lib
    from helmholtz_amd.device import DeviceArray
    from problems import small_case
    M, m, g, w = small_case(nodes, seed=5)
    hp = ha.HelmholtzParam(ha.getRegularMesh(M.domain, M.n), g, m, w, True, True)
    mg = ha.getMGparam(complex, int, levels, 1, 1, 1e-6, relax, 0.8, 2, 2, cycle, "NoMUMPS", 0.5, 0.0)
    mg.prec = prec
    s = ha.getShiftedLaplacianMultigridSolver(hp, mg, 0.5, "GMRES", 1)
    N, nr = m.size, 3
    rng = np.random.default_rng(1)
    V = np.asfortranarray(rng.standard_normal((N, nr)) + 1j * rng.standard_normal((N, nr)))
    want = ha.precondition(s, V)
    dt = want.dtype
    L = _lib.lib()

    def apply(vp, zp):
        _lib.check(L.hh_solver_precondition(s._handle, vp, zp, nr, _lib.HH_DEVICE))

    dv, dz = DeviceArray.from_numpy(V), DeviceArray((N, nr), dt)
    for _ in range(2):
        apply(dv.ptr, dz.ptr)
        assert np.array_equal(dz.to_numpy(), want)
    assert np.array_equal(dv.to_numpy(), V)
    # Z over V (exactly, and shifted by a few values)
    both = DeviceArray((N * nr + 64,), np.complex128)
    for shift in (0, 16):
        _lib.check(L.hh_memcpy(both.ptr + 16 * shift, V.ctypes.data, V.nbytes, 0))
        apply(both.ptr + 16 * shift, both.ptr)
        z = np.empty_like(want, order="F")
        _lib.check(L.hh_memcpy(z.ctypes.data, both.ptr, z.nbytes, 1))
        assert np.array_equal(z, want)
    # Z half a value off its alignment
    off = DeviceArray((N * nr + 2,), np.complex128)
    half = dt.itemsize // 2
    apply(dv.ptr, off.ptr + half)
    z = np.empty_like(want, order="F")
    _lib.check(L.hh_memcpy(z.ctypes.data, off.ptr + half, z.nbytes, 1))
    assert np.array_equal(z, want)
