"""What a program does with this framework, as cases that can be timed: Stokes
solves and time steps through Model / Context, batches of instances through
Batch, the learned guess's network through Net.

A case is a dict of plain values; its "kind" says which path it takes:

  stokes   one Stokes solve from rest on new fields: buoyancy, viscosity,
           assembly, the Uzawa solve, and the fields read back
  steps    a run continued from a saved state: the state is put back (T, d, p,
           the heat rates, model time), `steps` time steps follow, and the
           state is saved again
  batch    one round of independent instances by graph replay on concurrent
           lanes, each continued from its saved state
  forward  the network's output for a batch of fields
  train    the network's loss and gradients for a batch of snapshots (a caller
           that combines gradients itself takes them from here)

The box is `npx` x `npz` unit blocks of `side` x `side` elements, free slip
with T = 1 at the bottom and T = 0 at the top, viscosity exp(-ln(contrast) T).
"""
import ctypes as C
import math

import numpy as np
import torch

from mantle_convection_lab_amd import _native as N
from mantle_convection_lab_amd import amr
from mantle_convection_lab_amd.batch import Batch
from mantle_convection_lab_amd.learn import Net, default_weights_path, workload_keys
from mantle_convection_lab_amd.model import Input, Mesh, Model


def listed():
    return [
        # the reference's own kind of run: isoviscous 64 x 64, Ra 1e4, FP64 with its inner solver's caps
        dict(name="fp64_64_iso", kind="steps", side=64, npx=1, npz=1, Ra=1e4, contrast=1.0, precision=0, schur=1,
             solver="cg", warm=0, develop=0, steps=2),
        # the plain FP64 method on variable viscosity: the yardstick of every mixed solve
        dict(name="fp64_128", kind="stokes", side=128, npx=1, npz=1, Ra=1e6, contrast=1e3, precision=0, schur=1,
             solver="cg"),
        # the reference's default inner solver (Jacobi) behind the drop-in boundary
        dict(name="fp64_32_jacobi", kind="stokes", side=32, npx=1, npz=1, Ra=1e4, contrast=1.0, precision=0, schur=1,
             solver="jc", noise=0.0),
        # the smallest mesh of the batched workload: every phase is latency
        dict(name="mixed_32", kind="stokes", side=32, npx=1, npz=1, Ra=1e5, contrast=30.0, precision=1, schur=1,
             solver="cg"),
        # a 3:1 box, the wide boxes of convection studies; its rows do not divide evenly over the device
        dict(name="mixed_192x64_run", kind="steps", side=64, npx=3, npz=1, Ra=3e5, contrast=100.0, precision=1,
             schur=1, solver="cg", warm=1, develop=4, steps=4),
        # the headline workload's first solve
        dict(name="mixed_256", kind="stokes", side=256, npx=1, npz=1, Ra=1e6, contrast=1e3, precision=1, schur=1,
             solver="cg"),
        # the headline workload once the flow has settled: a run continued, the network consulted
        dict(name="mixed_256_run", kind="steps", side=256, npx=1, npz=1, Ra=1e6, contrast=1e3, precision=1, schur=1,
             solver="cg", warm=1, develop=14, steps=8, net=True),
        # the largest mesh of the batched workload
        dict(name="mixed_512", kind="stokes", side=512, npx=1, npz=1, Ra=1e6, contrast=30.0, precision=1, schur=1,
             solver="cg"),
        # an adapted quadtree with hanging nodes, aspect ratio 2
        dict(name="amr_32x16", kind="stokes", side=16, extra=2, plumes=8, Ra=1e6, contrast=1e3, precision=1),
        # a batch of small instances advanced together
        dict(name="batch_6", kind="batch", n=6, smin=32, smax=128, Ra=1e5, contrast=100.0, lanes=4),
        # the network's pass inside a guess: one 256 x 256 field
        dict(name="forward_256_b1", kind="forward", H=256, W=256, B=1),
        # the network's training at its stated batch of 32
        dict(name="train_256_b32", kind="train", H=256, W=256, B=32),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["fp64", "jacobi", "mixed", "mixed", "run", "run", "amr", "batch", "forward", "train"])
    Ra, contrast = round(_log(rng, 1e4, 3e6), 1), round(_log(rng, 1.0, 1e3), 3)
    if kind == "fp64":
        side, npx, npz = rng.choice([(16, 1, 1), (16, 3, 1), (32, 1, 1), (32, 2, 1), (32, 1, 2), (64, 1, 1),
                                     (32, 3, 2)])
        return dict(kind="stokes", side=side, npx=npx, npz=npz, Ra=Ra, contrast=contrast, precision=0, schur=1,
                    solver="cg")
    if kind == "jacobi":
        side, npx, npz = rng.choice([(8, 1, 1), (8, 3, 1), (16, 1, 1), (16, 2, 1), (16, 1, 3), (32, 1, 1)])
        return dict(kind="stokes", side=side, npx=npx, npz=npz, Ra=Ra, contrast=min(contrast, 30.0), precision=0,
                    schur=1, solver="jc", noise=0.0)
    if kind == "mixed":
        side, npx, npz = rng.choice([(32, 1, 1), (32, 3, 1), (64, 1, 1), (64, 2, 1), (64, 3, 2), (128, 1, 1),
                                     (128, 1, 2), (128, 3, 1), (256, 1, 1), (256, 2, 1)])
        return dict(kind="stokes", side=side, npx=npx, npz=npz, Ra=Ra, contrast=contrast, precision=1, schur=1,
                    solver="cg")
    if kind == "run":
        side, npx, npz = rng.choice([(32, 1, 1), (32, 4, 1), (64, 1, 1), (64, 2, 1), (128, 1, 1), (128, 2, 1),
                                     (256, 1, 1)])
        return dict(kind="steps", side=side, npx=npx, npz=npz, Ra=Ra, contrast=contrast, precision=1, schur=1,
                    solver="cg", warm=1, develop=rng.randint(4, 12), steps=rng.randint(1, 8))
    if kind == "amr":
        return dict(kind="stokes", side=16, extra=rng.randint(1, 2), plumes=rng.randint(4, 12), Ra=Ra,
                    contrast=contrast, precision=1)
    if kind == "batch":
        return dict(kind="batch", n=rng.randint(3, 6), smin=32, smax=rng.choice([64, 128]), Ra=Ra, contrast=contrast,
                    lanes=rng.randint(2, 4))
    H, W = rng.choice([32, 64, 128, 256]), rng.choice([32, 64, 128, 256])
    most = max(1, min(32, 32 * 256 * 256 // (H * W)))
    return dict(kind=kind, H=H, W=W, B=max(1, int(_log(rng, 1, most + 0.99))))


# ------------------------------------------------------------------- inputs

def _keys(case):
    # the multigrid of a wide box starts one level lower: its coarsest grid then has as few rows as the unit box's
    return workload_keys(case["side"], case["Ra"], case["contrast"], 1, nprox=case["npx"], nproz=case["npz"],
                         model_length=float(case["npx"]), model_height=float(case["npz"]),
                         precision=case["precision"], schur_mode=case["schur"], solver=case["solver"],
                         mg_min_level=2 if case["npx"] * case["npz"] <= 2 else 1, warm_start=case.get("warm", 0), zero_P=int(case["kind"] == "stokes"))


def _temperature(case, X, seed):
    """A conductive profile with a seeded perturbation: long waves, and noise
    on every node (0.01 as in the runs' initial states)."""
    rng = np.random.default_rng(seed)
    x, z = X[0] / case["npx"], X[1] / case["npz"]
    T = 1 - z
    for k in range(1, 4):
        T = T + 0.01 * rng.uniform(0.3, 1) * np.cos(np.pi * k * x) * np.sin(np.pi * z)
    T = T + case.get("noise", 0.01) * rng.uniform(-1, 1, x.size) * np.sin(np.pi * z)
    T[np.isclose(z, 0.0)], T[np.isclose(z, 1.0)] = 1.0, 0.0
    return T


_STATE = ("T", "HEAT_D", "HEAT_DDOT", "D", "P")


def _saved(m):
    return {f: m.field(f) for f in _STATE}, m.ctx.model_time()


def _restore(m, saved):
    fields, t = saved
    for f, v in fields.items():
        m.ctx.set_field(m.finest, f, v)
    m.ctx.set_model_time(t)


def _fields(m, names):
    return {f: m.field(f) for f in names}


def _net_input(case, rng):
    """Fields as the network meets them: temperature anomaly of unit RMS
    (plumes, boundary layers, noise) and log10 viscosity between -3 and 0."""
    B, H, W = case["B"], case["H"], case["W"]
    z, x = np.meshgrid((np.arange(H) + 0.5) / H, (np.arange(W) + 0.5) / W, indexing="ij")
    out = np.empty((B, H, W, 2), np.float32)
    for b in range(B):
        a = sum(rng.normal() * np.cos(np.pi * k * x + rng.uniform(0, 6)) * np.sin(np.pi * rng.integers(1, 4) * z)
                for k in range(1, 6))
        a = a + 0.1 * rng.normal(size=a.shape)
        a = a - a.mean(axis=1, keepdims=True)
        out[b, :, :, 0] = a / np.sqrt((a * a).mean())
        out[b, :, :, 1] = -3 * rng.uniform() * np.clip(1 - z + 0.05 * a, 0, 1)
    return out


def _net_target(case, rng):
    B, H, W = case["B"], case["H"], case["W"]
    z, x = np.meshgrid((np.arange(H) + 0.5) / H, (np.arange(W) + 0.5) / W, indexing="ij")
    t = np.empty((B, H, W, 3), np.float32)
    for b in range(B):
        for c in range(3):
            t[b, :, :, c] = rng.normal() * np.cos(np.pi * rng.integers(1, 4) * x) * np.sin(np.pi * z)
            t[b, :, :, c] += 0.1 * rng.normal(size=(H, W))
    return t


def _net(case, seed):
    """(network, x, t): trained weights for a forward pass (they fit any grid),
    seeded initial weights for training."""
    rng = np.random.default_rng(seed)
    net = Net(case["H"], case["W"], case["B"], seed=int(rng.integers(1, 1 << 40)))
    x = _net_input(case, rng)
    if case["kind"] == "forward":
        net.load(default_weights_path(256))
        return net, x, None
    return net, x, _net_target(case, rng)


def _batch_specs(case, seed):
    rng = np.random.default_rng(seed)
    depth = np.linspace(math.log2(case["smin"]), math.log2(case["smax"]), case["n"]).round().astype(int)
    return [(int(2 ** d), float(case["Ra"] * 10 ** rng.uniform(-0.5, 0.5)),
             float(max(1.0, case["contrast"] * 10 ** rng.uniform(-0.5, 0.5))), int(rng.integers(1, 1 << 40)))
            for d in depth]


class _State:
    """What the program keeps: released when the state is dropped."""

    def __init__(self, case, **kw):
        self.case = case
        self.__dict__.update(kw)

    def __del__(self):
        for o in ("model", "batch", "net"):
            v = getattr(self, o, None)
            if v is not None:
                (v.ctx if o == "model" else v).close()


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("forward", "train"):
        net, x, t = _net(case, seed)
        return _State(case, net=net, x=x, t=t, grads=np.empty(net.n, np.float32))
    if kind == "batch":
        b = Batch(_batch_specs(case, seed), learn_min=0)
        b.step()
        b.capture(case["lanes"])
        return _State(case, batch=b, saved=[_saved(m) for m in b.models])
    if "plumes" in case:
        keys, base = amr.c3_keys(2 * case["side"], case["extra"], Ra=case["Ra"], contrast=case["contrast"],
                                 warm_start=0, zero_P=1)
        inp = Input.from_keys(keys)
        mesh = Mesh(inp, depth=base)
        develop = lambda X: amr.developed_temperature(X, length=2.0, delta=0.05, nplumes=case["plumes"],  # noqa: E731
                                                      width=0.05)
        for _ in range(case["extra"] + 1):
            mesh, _, nr, nc = mesh.adapt(develop(mesh.level(-1)["X"]), base, base + case["extra"])
            if nr == 0 and nc == 0:
                break
        X = mesh.level(-1)["X"]
        rng = np.random.default_rng(seed)
        T = develop(X) * (1 + 0.02 * rng.uniform(-1, 1, X.shape[1]))
        return _State(case, model=Model(inp, mesh=mesh, T0=np.clip(T, 0.0, 1.0)))
    inp = Input.from_keys(_keys(case))
    mesh = Mesh(inp)
    T0 = _temperature(case, mesh.level(-1)["X"], seed)
    if kind == "stokes":
        return _State(case, model=Model(inp, mesh=mesh, T0=T0))
    net = None
    if case.get("net"):
        net = Net(case["side"] * case["npz"], case["side"] * case["npx"], 1)
        net.load(default_weights_path(256))
    m = Model(inp, mesh=mesh, T0=T0, net=net)
    for _ in range(case["develop"]):
        m.step()
    if case["develop"] == 0:
        # a run's very first step: the heat equation starts from T at rest
        lv = mesh.level(-1)
        m.ctx.set_field(m.finest, "HEAT_D", T0[lv["heat_eq_node"]])
    return _State(case, model=m, net=net, saved=_saved(m))


def run(state):
    kind = state.case["kind"]
    if kind == "forward":
        return state.net.forward(state.x)
    if kind == "train":
        loss = state.net.train_step(state.x, state.t, 0.0)
        state.net._ck(N.hip_lib().mcl_net_get_grads(state.net.h, state.grads.ctypes.data_as(C.POINTER(C.c_float))))
        return {"loss": loss, "grads": state.grads}
    if kind == "batch":
        for m, s in zip(state.batch.models, state.saved):
            _restore(m, s)
        state.batch.graph_step()
        return [_fields(m, _STATE) for m in state.batch.models]
    m = state.model
    if kind == "stokes":
        c = m.ctx
        c.buoyancy_force()
        c.viscosity()
        c.velocity_pressure_KGF_matrix()
        c.solve_velocity_pressure()
        return _fields(m, ("V", "P", "STRESS"))
    _restore(m, state.saved)
    for _ in range(state.case["steps"]):
        m.step()
    return _fields(m, _STATE)


# --------------------------------------------------------- what has to be done

CONVS = [(16, 32, 0), (32, 32, 0), (32, 64, 1), (64, 64, 1), (64, 128, 2), (128, 128, 2), (128, 256, 3), (256, 256, 3),
         (384, 128, 2), (128, 128, 2), (192, 64, 1), (64, 64, 1), (96, 32, 0), (32, 32, 0)]  # (Cin, Cout, level)


def _elements(case):
    if case["kind"] == "batch":
        d = np.linspace(math.log2(case["smin"]), math.log2(case["smax"]), case["n"]).round()
        return float((4.0 ** d).sum())
    if "plumes" in case:
        return 2.0 * case["side"] ** 2 * 4.0 ** case["extra"] * 0.5   # about half of the box at the finest level
    return float(case["side"] ** 2 * case["npx"] * case["npz"])


def work(case):
    """Network: each layer's products, its input read and its output written
    once in bf16, weights once (training: three products and twice the
    activations' traffic).  Solves and steps: the fields in and out once, and
    the matrix (18 entries a row, two rows a node) written and read once, in
    each step; the iterations that a solve needs are not known beforehand."""
    if case["kind"] in ("forward", "train"):
        M = float(case["B"] * case["H"] * case["W"])
        flops = sum(2 * 9 * ci * co * M / 4 ** l for ci, co, l in CONVS) + 2 * 96 * M
        nbytes = sum(2 * (ci + co) * M / 4 ** l + 2 * 9 * ci * co for ci, co, l in CONVS) + 20 * M
        return {"bytes": nbytes * (1 if case["kind"] == "forward" else 3), "flops": flops * (1 if case["kind"] == "forward" else 3)}
    n = _elements(case) * case.get("steps", 1)
    return {"bytes": n * (2 * 18 * 2 * (8 + 4) + 12 * 8), "flops": n * 2 * 18 * 2 * 2}


# ------------------------------------------------------- results in 64 bits

def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _exact_net(case, seed):
    net, x, t = _net(case, seed)
    params = net.params()
    net.close()
    dev = _dev()
    ws, off = [], 0
    for ci, co, _ in CONVS:
        w = params[off: off + co * 9 * ci].reshape(co, 9, ci)
        off += co * 9 * ci
        ws.append((torch.tensor(w, dtype=torch.float64, device=dev).requires_grad_(),
                   torch.tensor(params[off: off + co], dtype=torch.float64, device=dev).requires_grad_()))
        off += co
    wh = torch.tensor(params[off: off + 96].reshape(3, 32), dtype=torch.float64, device=dev).requires_grad_()
    bh = torch.tensor(params[off + 96: off + 99], dtype=torch.float64, device=dev).requires_grad_()

    def conv(i, v):  # v: (B, H, W, C)
        w, b = ws[i]
        H, W = v.shape[1:3]
        p = torch.nn.functional.pad(v, (0, 0, 1, 1, 1, 1))
        y = b
        for k in range(9):
            y = y + p[:, k // 3: k // 3 + H, k % 3: k % 3 + W].reshape(-1, v.shape[3]) @ w[:, k, : v.shape[3]].T
        return torch.relu(y).reshape(*v.shape[:3], -1)

    def pool(v):
        B, H, W, ch = v.shape
        return v.reshape(B, H // 2, 2, W // 2, 2, ch).mean(dim=(2, 4))

    def up(v):
        return v.repeat_interleave(2, dim=1).repeat_interleave(2, dim=2)

    def net64(v):
        e1 = conv(1, conv(0, v))
        e2 = conv(3, conv(2, pool(e1)))
        e3 = conv(5, conv(4, pool(e2)))
        b = conv(7, conv(6, pool(e3)))
        d3 = conv(9, conv(8, torch.cat([up(b), e3], 3)))
        d2 = conv(11, conv(10, torch.cat([up(d3), e2], 3)))
        d1 = conv(13, conv(12, torch.cat([up(d2), e1], 3)))
        return d1 @ wh.T + bh

    # one image after the other: the gradients add up, the memory does not
    ys, loss = [], 0.0
    for b in range(case["B"]):
        v = torch.zeros(1, case["H"], case["W"], 16, dtype=torch.float64, device=dev)
        v[..., :2] = torch.tensor(x[b], dtype=torch.float64, device=dev)
        y = net64(v)
        if t is None:
            ys.append(y.detach()[0].cpu())
            continue
        part = ((y[0] - torch.tensor(t[b], dtype=torch.float64, device=dev)) ** 2).sum() / t.size
        part.backward()
        loss += float(part)
    if t is None:
        return torch.stack(ys)
    grads = [g.grad.reshape(-1) for w in ws for g in w] + [wh.grad.reshape(-1), bh.grad]
    return {"loss": loss, "grads": torch.cat(grads).cpu()}


def _exact_stokes(case, seed):
    """Nodal velocity by dense Cholesky factors of the stiffness and of the
    Schur complement, from the elements' formulas; nodes x-major."""
    dev = _dev()
    nx, nz = case["side"] * case["npx"], case["side"] * case["npz"]
    length, height = float(case["npx"]), float(case["npz"])
    gx, gz = nx + 1, nz + 1
    x, z = np.meshgrid(np.arange(gx) * (length / nx), np.arange(gz) * (height / nz), indexing="ij")
    T = _temperature(case, np.stack([x.ravel(), z.ravel()]), seed)
    eta = np.exp(-math.log(case["contrast"]) * T)
    b = case["Ra"] * T
    b = b - np.tile(b.reshape(gx, gz).mean(axis=0), gx)
    ex, ez = np.meshgrid(np.arange(nx), np.arange(nz), indexing="ij")
    n0 = (ex * gz + ez).ravel()
    ien = np.stack([n0, n0 + 1, n0 + gz + 1, n0 + gz])            # corners (-,-), (-,+), (+,+), (+,-)
    hx, hz = length / nx, height / nz
    s = np.array([[-1, -1], [-1, 1], [1, 1], [1, -1]], float)
    nel = nx * nz
    Ke = np.zeros((8, 8, nel))
    Fe = np.zeros((8, nel))
    Ge = np.zeros((8, nel))
    for g in s / math.sqrt(3.0):
        Na = 0.25 * (1 + s[:, 0] * g[0]) * (1 + s[:, 1] * g[1])
        dx = 0.25 * s[:, 0] * (1 + s[:, 1] * g[1]) * 2 / hx
        dz = 0.25 * s[:, 1] * (1 + s[:, 0] * g[0]) * 2 / hz
        J = hx * hz / 4
        e = Na @ eta[ien]
        f = Na @ b[ien]
        for a in range(4):
            Ge[2 * a] -= dx[a] * J
            Ge[2 * a + 1] -= dz[a] * J
            Fe[2 * a + 1] += Na[a] * f * J
            for c in range(4):
                Ke[2 * a, 2 * c] += e * J * (2 * dx[a] * dx[c] + dz[a] * dz[c])
                Ke[2 * a, 2 * c + 1] += e * J * dz[a] * dx[c]
                Ke[2 * a + 1, 2 * c] += e * J * dx[a] * dz[c]
                Ke[2 * a + 1, 2 * c + 1] += e * J * (2 * dz[a] * dz[c] + dx[a] * dx[c])
    nno = gx * gz
    free = np.ones((nno, 2), bool)
    ix, iz = np.divmod(np.arange(nno), gz)
    free[(ix == 0) | (ix == nx), 0] = False
    free[(iz == 0) | (iz == nz), 1] = False
    num = np.full(2 * nno, -1)
    keep = np.flatnonzero(free.ravel())
    num[keep] = np.arange(keep.size)
    dof = np.stack([2 * ien[a] + d for a in range(4) for d in range(2)])
    q = torch.tensor(num[dof], device=dev)
    n = keep.size
    to = lambda v: torch.tensor(v, dtype=torch.float64, device=dev)  # noqa: E731
    K = torch.zeros(n + 1, n + 1, dtype=torch.float64, device=dev)   # the last row takes the fixed degrees of freedom
    G = torch.zeros(n + 1, nel, dtype=torch.float64, device=dev)
    F = torch.zeros(n + 1, dtype=torch.float64, device=dev)
    q = torch.where(q < 0, n, q)
    col = torch.arange(nel, device=dev)
    for i in range(8):
        F.index_put_((q[i],), to(Fe[i]), accumulate=True)
        G.index_put_((q[i], col), to(Ge[i]), accumulate=True)
        for j in range(8):
            K.index_put_((q[i], q[j]), to(Ke[i, j]), accumulate=True)
    K, G, F = K[:n, :n], G[:n], F[:n]
    L = torch.linalg.cholesky(K)
    A = torch.linalg.solve_triangular(L, G, upper=False)
    y = torch.linalg.solve_triangular(L, F[:, None], upper=False)
    S = A.T @ A
    S = S + torch.trace(S) / nel ** 2                               # the constant pressure is free: fix it
    p = torch.cholesky_solve(A.T @ y, torch.linalg.cholesky(S))
    u = torch.linalg.solve_triangular(L.T, y - A @ p, upper=True)[:, 0].cpu().numpy()
    V = np.zeros(2 * nno)
    V[keep] = u
    return {"V": np.ascontiguousarray(V.reshape(nno, 2).T).ravel(), "P": None, "STRESS": None}


def exact(case, seed):
    if case["kind"] in ("forward", "train"):
        return _exact_net(case, seed)
    if case["kind"] == "stokes" and "plumes" not in case and _elements(case) <= 2048:
        return _exact_stokes(case, seed)
    return None
