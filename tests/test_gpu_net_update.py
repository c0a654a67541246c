"""The weight update over all layers in one launch (MI355X): two Adam steps
against the same formula in FP64 on the gradients read back, every parameter of
every layer; and a network that has stepped against one given the same
parameters, whose bf16 weights come from the other form of the kernel: equal
outputs bit for bit, gradients to the order of their FP32 sums.  The bound of
an update is relative to its terms, lr (b1 |m1| + ...) / den: ten FP32 roundings
and 1 - b2^k, whose FP32 value is off by up to 6e-5 of itself; the parameter's
own rounding comes on top."""
import ctypes as C

import numpy as np
import pytest

from tests.test_gpu_unet import CONVS, _fp, _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,B", [(16, 16, 1), (32, 48, 2)])
def test_update_all_layers(H, W, B):
    print(f"[gpu-net-update] {H} x {W}, batch {B}", flush=True)
    L = _lib()
    rng = np.random.default_rng(H + W)
    x = rng.normal(0, 1, (B, H, W, 2)).astype(np.float32)
    t = rng.normal(0, 1, (B, H, W, 3)).astype(np.float32)
    a, b = C.c_void_p(), C.c_void_p()
    assert L.mcl_net_create(H, W, B, 7, C.byref(a)) == 0
    assert L.mcl_net_create(H, W, B, 8, C.byref(b)) == 0
    try:
        n = L.mcl_net_num_params(a)
        assert n == sum(co * 9 * ci + co for ci, co in CONVS) + 99
        g, h, p, q = (np.ones(n, np.float32) for _ in range(4))
        loss = C.c_float()
        assert L.mcl_net_get_grads(a, _fp(g)) == 0 and not g.any()
        assert L.mcl_net_get_params(a, _fp(p)) == 0
        lr, b1, b2 = (float(np.float32(v)) for v in (1e-3, 0.9, 0.999))
        m1, m2, m1abs = np.zeros(n), np.zeros(n), np.zeros(n)
        for k in (1, 2):
            assert L.mcl_net_train_step(a, _fp(x), _fp(t), lr, C.byref(loss)) == 0
            assert L.mcl_net_get_grads(a, _fp(g)) == 0
            assert L.mcl_net_get_params(a, _fp(q)) == 0
            gd = g.astype(np.float64)
            m1 = b1 * m1 + (1 - b1) * gd
            m1abs = b1 * m1abs + (1 - b1) * np.abs(gd)
            m2 = b2 * m2 + (1 - b2) * gd * gd
            c1, c2 = 1 - b1 ** k, 1 - b2 ** k
            den = np.sqrt(m2 / c2) + 1e-8
            want = p - lr * (m1 / c1) / den
            bound = lr * (m1abs / c1) / den * (10 * 6e-8 + 6e-5) + 1.2e-7 * np.abs(want) + 1e-12
            assert np.all(np.abs(q - want) <= bound), (k, np.max(np.abs(q - want) / bound))
            p = q.copy()
        ya, yb = np.zeros((B, H, W, 3), np.float32), np.zeros((B, H, W, 3), np.float32)
        assert L.mcl_net_set_params(b, _fp(q)) == 0
        assert L.mcl_net_forward(a, _fp(x), _fp(ya)) == 0 and L.mcl_net_forward(b, _fp(x), _fp(yb)) == 0
        assert ya.tobytes() == yb.tobytes()
        for net, out in ((a, g), (b, h)):
            assert L.mcl_net_train_step(net, _fp(x), _fp(t), 0.0, C.byref(loss)) == 0
            assert L.mcl_net_get_grads(net, _fp(out)) == 0
        assert np.linalg.norm(g.astype(np.float64) - h) <= 1e-4 * np.linalg.norm(g.astype(np.float64))
    finally:
        L.mcl_net_destroy(a)
        L.mcl_net_destroy(b)
