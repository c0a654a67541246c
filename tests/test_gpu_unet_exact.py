"""The network's gradients where every product and sum is exact (MI355X).

Each convolution copies one shifted input channel into every output channel (a
weight of 1, or of 4 behind a pooling, which makes the mean of four a sum
again), the input holds small whole numbers and the target differs from the
output of M pixels by -c, 0 or c, c = 3 M / 2^e, so that the loss's gradient
2 / (3 M) c rounds to s = 2^(1-e) in bf16.  Then every activation is a whole
number or a quarter of one below 2^8, every gradient s times a whole number
below 2^8, and every weight gradient s times a sum below 2^22: bf16 holds the
former, FP32 sums the latter without rounding in any order.  So the
convolutions' gradients must equal the FP64 ones bit for bit: a tile left out,
a halo lost or a remainder counted twice shows, which 1e-1 does not see.
(Checked on the CPU for these seeds: the largest activation is 133, gradient
13 s, sum of magnitudes 1.2e6 s.)"""
import ctypes as C
import statistics
import time

import numpy as np
import pytest

from tests.test_gpu_unet import CONVS, _flat_grads, _fp, _lib, _torch_net

pytestmark = pytest.mark.gpu


def _copying_params(rng):
    out = []
    for i, (cin, cout) in enumerate(CONVS):
        w = np.zeros((cout, 9, cin), np.float32)
        real = 2 if i == 0 else cin   # the input's other channels are zero
        w[np.arange(cout), rng.integers(0, 9, cout), np.resize(rng.permutation(real), cout)] = \
            4.0 if i in (2, 4, 6) else 1.0
        out += [w.ravel(), np.zeros(cout, np.float32)]
    wh = np.zeros((3, 32), np.float32)
    wh[np.arange(32) % 3, np.arange(32)] = 1.0
    return np.concatenate(out + [wh.ravel(), np.zeros(3, np.float32)])


def _case(H, W, B):
    """(parameters, x, target, the convolutions' gradients in FP64 with the
    loss's gradient rounded to s)"""
    import torch
    e = (3 * H * W * B).bit_length()
    c, s = 3 * H * W * B / 2.0 ** e, 2.0 ** (1 - e)
    rng = np.random.default_rng(1000 * H + W + B)
    p = _copying_params(rng)
    x = rng.integers(0, 4, (B, H, W, 2))
    k = np.where(rng.random((B, H, W, 3)) < 1 / 16, rng.choice([-1.0, 1.0], (B, H, W, 3)), 0.0)
    fwd, ws, wh, bh = _torch_net(p.astype(np.float64))
    xt = torch.zeros((B, 16, H, W), dtype=torch.float64)
    xt[:, :2] = torch.tensor(x, dtype=torch.float64).permute(0, 3, 1, 2)
    y = fwd(xt)
    t = y.detach() - torch.tensor(k).permute(0, 3, 1, 2)
    (0.5 * s * ((y - t) ** 2).sum()).backward()
    t = (y.detach() - c * torch.tensor(k).permute(0, 3, 1, 2)).permute(0, 2, 3, 1).numpy()
    x32, t32 = (np.ascontiguousarray(a.astype(np.float32)) for a in (x, t))
    assert np.array_equal(t32, t)
    return p, x32, t32, _flat_grads(ws, wh, bh)[:28]


def _grads(L, H, W, B, p, x, t):
    net = C.c_void_p()
    assert L.mcl_net_create(H, W, B, 1, C.byref(net)) == 0
    try:
        g, loss = np.zeros(p.size, np.float32), C.c_float()
        assert L.mcl_net_set_params(net, _fp(p)) == 0
        assert L.mcl_net_train_step(net, _fp(x), _fp(t), 0.0, C.byref(loss)) == 0
        assert L.mcl_net_get_grads(net, _fp(g)) == 0
        return g
    finally:
        L.mcl_net_destroy(net)


# levels 16 and 8 pixels wide and the 4- and 2-wide ones below them; 17 runs of
# 64 pixels in two splits; 64-wide levels two and six rows high
@pytest.mark.parametrize("H,W,B", [(64, 16, 3), (136, 32, 1), (64, 64, 5), (16, 512, 1), (48, 256, 1)])
def test_gradients_exact_narrow_levels(H, W, B):
    _check(H, W, B)


# five tiles in three splits; 32 x 4 tiles below; an odd tile count over many
# workgroups; three tiles a split at the 64-wide level
@pytest.mark.parametrize("H,W,B", [(40, 32, 1), (48, 96, 1), (128, 256, 3), (256, 256, 3)])
def test_gradients_exact_tiles(H, W, B):
    _check(H, W, B)


@pytest.mark.parametrize("H,W,B", [(32, 256, 15), (64, 128, 9), (256, 256, 4)])
def test_forward_bytes_do_not_depend_on_the_tile(H, W, B):
    """An image alone takes smaller tiles than in a batch; every output is the
    same chain of products."""
    print(f"[gpu-unet-exact] forward {H} x {W}, batch {B} and alone", flush=True)
    from mantle_convection_lab_amd.learn import Net
    x = np.random.default_rng(H + W).normal(size=(B, H, W, 2)).astype(np.float32)
    batch, one = Net(H, W, B, seed=3), Net(H, W, 1, seed=3)
    y = batch.forward(x)
    for b in range(B):
        assert y[b].tobytes() == one.forward(x[b: b + 1])[0].tobytes(), b
    batch.close()
    one.close()


def _check(H, W, B):
    print(f"[gpu-unet-exact] {H} x {W}, batch {B}", flush=True)
    p, x, t, want = _case(H, W, B)
    g = _grads(_lib(), H, W, B, p, x, t)
    off = 0
    for i, w in enumerate(want):
        got = g[off: off + w.size]
        off += w.size
        assert w.any()
        assert np.array_equal(got, w), (i, np.abs(got - w).max())


def test_narrow_levels_take_the_staged_weight_gradient():
    """A training step of a tall image, whose levels are 64 to 8 pixels wide,
    against the same image lying, 256 to 32: the same products.  Staged they
    differ by the tiles (1.3 times); with the 16- and 8-wide levels' weight
    gradients unstaged it was 3.9 times, and a 512 x 16 network's seven
    milliseconds."""
    from mantle_convection_lab_amd.learn import Net
    rng = np.random.default_rng(0)
    took = []
    for H, W in ((256, 64), (64, 256)):
        net = Net(H, W, 4, seed=3)
        x = rng.normal(size=(4, H, W, 2)).astype(np.float32)
        t = rng.normal(size=(4, H, W, 3)).astype(np.float32)
        ts = []
        for _ in range(20):
            t0 = time.perf_counter()
            net.train_step(x, t, 1e-3)
            ts.append(time.perf_counter() - t0)
        took.append(statistics.median(ts))
        net.close()
    print(f"[gpu-unet-exact] tall {took[0] * 1e6:.0f} us, lying {took[1] * 1e6:.0f} us", flush=True)
    assert took[0] <= 2 * took[1]
