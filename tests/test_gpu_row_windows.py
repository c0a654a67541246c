"""The FP64 solvers' one-row-a-thread form on meshes with hanging nodes (MI355X).

One refined corner element leaves two hanging nodes and rows of at most 18
velocity and 9 temperature slots, so the form applies, and with it a wait more
after the constraint.  In a box of 16 x 3072 elements the vector window of some
workgroups fits the LDS buffer of 6144 doubles and that of others does not: all
of them must then take the same form.  A capped launch has more rows than
threads and reads the matrix; the two agree as two workgroup counts do
(iterations equal, fields to 1e-10: compensated sums)."""
import math

import numpy as np
import pytest

WINDOW, ROWS = 6144, 512


def _corner(side, nproz, **over):
    from mantle_convection_lab_amd import Input, Mesh
    from mantle_convection_lab_amd.learn import workload_keys
    base = int(round(math.log2(side)))
    keys = workload_keys(side, 1e5, 30.0, seed=3, nproz=nproz, model_height=float(nproz), precision=0, warm_start=0)
    keys.update(dict(level=base + 2, mg_min_level=min(2, base)), **over)
    inp = Input.from_keys(keys)
    mesh = Mesh(inp, depth=base)
    X = mesh.level(-1)["X"]
    spike = np.where(np.isclose(X[0], 0.0) & np.isclose(X[1], 0.0), 1e6, 0.0)
    mesh, _, refined, _ = mesh.adapt(spike, base, base + 1, 1.0, 0.0)
    assert refined == 1
    return inp, mesh


def _windows(lm, n):
    """(longest row, widths of the windows of 512 rows) of n equations, lm
    [corners][nel]."""
    per = lm.shape[0]
    r = np.repeat(lm, per, axis=0).ravel()
    c = np.tile(lm, (per, 1)).ravel()
    both = (r >= 0) & (c >= 0)
    pair = np.unique(r[both].astype(np.int64) * n + c[both])
    r, c = pair // n, pair % n
    first = np.searchsorted(r, np.arange(0, n, ROWS))
    return int(np.bincount(r).max()), np.maximum.reduceat(c, first) - np.minimum.reduceat(c, first) + 1


@pytest.mark.parametrize("side,nproz,mixed", [(32, 1, False), (16, 192, True)])
def test_corner_mesh_windows(side, nproz, mixed):
    """The meshes below are what their tests say (CPU)."""
    lv = _corner(side, nproz)[1].level(-1)
    assert lv["nh"] == 2
    for lm, n, slots in ((lv["lm"].reshape(8, -1), lv["neq"], 18), (lv["heat_lm"], lv["neqT"], 9)):
        longest, w = _windows(lm, n)
        assert longest == slots and len(w) > 1
        assert w.min() <= WINDOW
        assert (w.max() > WINDOW) == mixed


def _run(side, nproz, cap, **over):
    from mantle_convection_lab_amd import Model
    inp, mesh = _corner(side, nproz, **over)
    x, z = mesh.level(-1)["X"] / [[1.0], [nproz]]
    m = Model(inp, mesh=mesh, T0=1 - z + 0.1 * np.cos(np.pi * x) * np.sin(np.pi * z))
    m.ctx._ck(m.ctx.L.mcl_set_launch_cap(m.ctx.h, cap))
    print(f"[row-windows] {side} x {side * nproz}, cap {cap}", flush=True)
    r = [m.step() for _ in range(2)]
    out = [(q["uzawa"], q["inner"], q["heat_cg"]) for q in r], [m.field(f) for f in ("D", "P", "T")]
    m.ctx.close()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("side,nproz,cap,over", [
    (32, 1, 1, {}),
    (64, 1, 1, dict(max_citcom_cycle=8)),
    (32, 1, 2, dict(exact_dots=1, max_citcom_cycle=10)),
    (16, 192, 60, dict(max_citcom_cycle=3, max_cg_cycle=60)),
])
def test_forms_agree_with_hanging_nodes(side, nproz, cap, over):
    (n0, f0), (n1, f1) = _run(side, nproz, 0, **over), _run(side, nproz, cap, **over)
    assert n0 == n1 and all(c[1] > 50 for c in n0)   # past the first recomputed residual
    for a, b in zip(f0, f1):
        assert np.isfinite(b).all() and np.linalg.norm(a - b) <= 1e-10 * np.linalg.norm(b)
