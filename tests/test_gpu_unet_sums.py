"""Sums over all pixels (loss, head bias gradient) at the edges of their blocks: fewer
pixels than a block's threads, one pixel past a chunk of 512, more chunks than the 512
blocks a launch takes.

Both follow from the network's own output in 64 bits.  A sum of n 32-bit terms through
blocks of at most n / 256 + 600 additions in a row is off by at most that many eps32 of
the sum of magnitudes; a term itself by 3 eps32."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nx,ny", [(1, 9, 9), (1, 17, 33), (1, 57, 9), (1, 41, 25), (17, 129, 129)])
def test_sums(n, nx, ny):
    from helmholtz_amd import learned
    rng = np.random.default_rng(nx)
    net = learned.UNet(seed=5)
    feats = rng.standard_normal((n, nx * ny, 4)).astype(np.float32)
    target = rng.standard_normal((n, nx * ny, 2)).astype(np.float32)
    y = net.forward(feats, nx, ny).astype(np.float64)
    loss, g = net.loss_grad(feats, target, nx, ny)
    d = (y - target).reshape(-1, 2)
    k = d.size
    tol = (k / 256 + 600 + 3) * np.finfo(np.float32).eps
    assert abs(loss - np.mean(d**2)) <= tol * np.mean(d**2)
    want = (2.0 * d / k).sum(axis=0)
    assert np.all(np.abs(np.asarray(g[-2:], np.float64) - want) <= tol * np.abs(2.0 * d / k).sum(axis=0))
