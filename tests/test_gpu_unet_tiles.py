"""The U-Net's convolution tiles at the sizes where they can go wrong: images
narrower or lower than a tile, one more and one less than a tile's width, single
tiles, batches that pick wide wavefronts (four pixel groups) and batches that do
not.

The reference states the network in torch on the CPU with every rounding that the
GPU makes: products summed in 64 bits, each stored activation and each stored
gradient rounded to BF16.  What is left is the order of the 32-bit sums, which now
and then moves a value to the next BF16 number or through a ReLU's zero.  The same
statement summed in 32 bits on the CPU is off from it by up to 3.1e-3 (output, in the
norm), 3.5e-2 (one pixel, of the output's rms), 4.7e-3 (gradient) and 1.3e-2 (a
layer's gradient) over these sizes and three seeds; the bars are four times that.  A
wrong tile edge is of the order of the output itself."""
import numpy as np
import pytest

from oracle import unet_ref as ur

pytestmark = pytest.mark.gpu


def rounded_network(theta, feats, target, nx, ny):
    """y, loss and gradient with the GPU's BF16 roundings."""
    torch = pytest.importorskip("torch")
    F = torch.nn.functional
    r16 = lambda x: x.float().to(torch.bfloat16).double()  # noqa: E731

    class Stored(torch.autograd.Function):  # stored in BF16, as its gradient is
        @staticmethod
        def forward(ctx, x):
            return r16(x)

        @staticmethod
        def backward(ctx, g):
            return r16(g)

    rd = Stored.apply
    th = torch.tensor(theta.astype(np.float64), requires_grad=True)
    n = feats.shape[0]
    x = torch.zeros((n, 16, ny, nx), dtype=torch.float64)
    x[:, :4] = torch.tensor(feats.astype(np.float64).reshape(n, ny, nx, 4)).permute(0, 3, 1, 2)
    ws, off = [], 0
    for ci, co in ur.SPEC:
        W = th[off:off + 9 * co * ci].reshape(3, 3, co, ci).permute(2, 3, 0, 1)
        off += 9 * co * ci
        ws.append((W, th[off:off + co]))
        off += co
    hw, hb = th[off:off + 32].reshape(2, 16), th[off + 32:off + 34]
    k1 = torch.tensor([0.25, 0.5, 0.25], dtype=torch.float64)
    kd, ku = torch.outer(k1, k1), torch.outer(2 * k1, 2 * k1)
    conv = lambda x, l: rd(torch.relu(F.conv2d(x, ws[l][0], ws[l][1], padding=1)))  # noqa: E731
    down = lambda x: rd(F.conv2d(x, kd.expand(x.shape[1], 1, 3, 3), stride=2, padding=1, groups=x.shape[1]))  # noqa: E731
    up = lambda x: rd(F.conv_transpose2d(x, ku.expand(x.shape[1], 1, 3, 3), stride=2, padding=1, groups=x.shape[1]))  # noqa: E731
    join = lambda u, s: rd(torch.cat([u, s], 1))  # noqa: E731
    s0 = conv(conv(x, 0), 1)
    s1 = conv(conv(down(s0), 2), 3)
    s2 = conv(conv(down(s1), 4), 5)
    b3 = conv(conv(down(s2), 6), 7)
    b4 = conv(conv(join(up(b3), s2), 8), 9)
    b5 = conv(conv(join(up(b4), s1), 10), 11)
    b6 = conv(conv(join(up(b5), s0), 12), 13)
    y = (torch.einsum("nchw,oc->nhwo", b6, hw) + hb).reshape(n, nx * ny, 2)
    loss = torch.mean((y - torch.tensor(target.astype(np.float64))) ** 2)
    loss.backward()
    return y.detach().numpy(), float(loss.detach()), th.grad.numpy().copy()


def case(seed, n, nx, ny):
    rng = np.random.default_rng(seed)
    feats = ur.bf16_round(rng.standard_normal((n, nx * ny, 4)).astype(np.float32))
    return feats, rng.standard_normal((n, nx * ny, 2)).astype(np.float32)


@pytest.mark.parametrize("n,nx,ny", [(1, 9, 9), (3, 17, 9), (1, 65, 9), (2, 9, 65), (1, 33, 33), (16, 65, 65),
                                     (4, 129, 129), (2, 97, 193)])
def test_tiles(n, nx, ny):
    from helmholtz_amd import learned
    net = learned.UNet(seed=11)
    theta = ur.bf16_round(net.get_params())
    net.set_params(theta)
    feats, target = case(nx + ny, n, nx, ny)
    yr, lref, gref = rounded_network(theta, feats, target, nx, ny)
    y = net.forward(feats, nx, ny)
    err = np.linalg.norm(y - yr) / np.linalg.norm(yr)
    peak = np.abs(y - yr).max() / np.sqrt(np.mean(yr**2))
    loss, g = net.loss_grad(feats, target, nx, ny)
    gerr = np.linalg.norm(g - gref) / np.linalg.norm(gref)
    print(f"{n} x {nx} x {ny}: forward {err:.2e}, largest {peak:.2e}, gradient {gerr:.2e}")
    assert err <= 1.25e-2 and peak <= 0.14
    assert loss == pytest.approx(lref, rel=1.25e-2)
    assert gerr <= 2e-2
    off = 0
    for ci, co in ur.SPEC:
        k = 9 * co * ci + co
        d = np.linalg.norm(g[off:off + k] - gref[off:off + k])
        print(f"  {ci} -> {co}: {d / np.linalg.norm(gref[off:off + k]):.2e}")
        assert d <= 5.2e-2 * np.linalg.norm(gref[off:off + k])
        off += k
    # nothing depends on what a buffer held before
    loss2, g2 = net.loss_grad(feats, target, nx, ny)
    assert np.array_equal(y, net.forward(feats, nx, ny)) and loss2 == loss and np.array_equal(g, g2)
