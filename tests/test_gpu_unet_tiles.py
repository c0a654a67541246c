"""The tiled convolutions at the shapes where their dispatch changes (MI355X):
widths that are multiples of 16 but not of 32 at some level, levels narrower
than 16 pixels (the run-of-64 and unstaged kernels), images lower than a tile,
batches whose tile count is not a multiple of eight, and enough pixels for the
large tiles.  Bars as in test_gpu_unet.py: forward within 3e-2 of FP64 and 2e-2
of the unstaged kernels, every weight and bias gradient within 1e-1 of FP64, or
as near as the unstaged kernels' own where bf16 itself is further off (a 16 x
16 network's bottom level has 2 x 2 pixels)."""
import ctypes as C
import os

import numpy as np
import pytest

from tests.test_gpu_unet import _flat_grads, _fp, _lib, _torch_net

pytestmark = pytest.mark.gpu


def _run(L, H, W, B, x, t, direct):
    net = C.c_void_p()
    assert L.mcl_net_create(H, W, B, 5, C.byref(net)) == 0
    try:
        if direct:
            os.environ["MCL_CONV_DIRECT"] = "1"
        n = L.mcl_net_num_params(net)
        p, g, y = np.zeros(n, np.float32), np.zeros(n, np.float32), np.zeros((B, H, W, 3), np.float32)
        loss = C.c_float()
        assert L.mcl_net_get_params(net, _fp(p)) == 0
        assert L.mcl_net_forward(net, _fp(x), _fp(y)) == 0
        assert L.mcl_net_train_step(net, _fp(x), _fp(t), 0.0, C.byref(loss)) == 0
        assert L.mcl_net_get_grads(net, _fp(g)) == 0
        return p, y, g, loss.value
    finally:
        os.environ.pop("MCL_CONV_DIRECT", None)
        L.mcl_net_destroy(net)


@pytest.mark.parametrize("H,W,B", [(16, 16, 1), (32, 96, 1), (32, 256, 2), (128, 32, 3), (48, 48, 2), (128, 256, 3)])
def test_tiles_match_fp64_and_direct(H, W, B):
    import torch
    print(f"[gpu-unet-tiles] {H} x {W}, batch {B}", flush=True)
    L = _lib()
    rng = np.random.default_rng(H + W + B)
    x = np.stack([rng.uniform(0, 1, (B, H, W)), rng.uniform(-3, 0, (B, H, W))], axis=-1).astype(np.float32)
    t = rng.normal(0, 1, (B, H, W, 3)).astype(np.float32)
    p, y, g, loss = _run(L, H, W, B, x, t, False)
    _, yd, gd, _ = _run(L, H, W, B, x, t, True)
    assert np.linalg.norm(y - yd) <= 2e-2 * np.linalg.norm(yd)
    fwd, ws, wh, bh = _torch_net(p.astype(np.float64))
    xt = torch.zeros((B, 16, H, W), dtype=torch.float64)
    xt[:, :2] = torch.tensor(x, dtype=torch.float64).permute(0, 3, 1, 2)
    yt = fwd(xt)
    yref = yt.detach().permute(0, 2, 3, 1).numpy()
    assert np.linalg.norm(y - yref) <= 3e-2 * np.linalg.norm(yref)
    lt = ((yt - torch.tensor(t, dtype=torch.float64).permute(0, 3, 1, 2)) ** 2).mean()
    lt.backward()
    assert abs(loss - lt.item()) < 3e-2 * lt.item()
    off = 0
    for i, r in enumerate(_flat_grads(ws, wh, bh)):
        e, ed = (np.linalg.norm(v[off: off + r.size] - r) / max(np.linalg.norm(r), 1e-30) for v in (g, gd))
        off += r.size
        assert e < max(1e-1, 1.25 * ed), (i, e, ed)
