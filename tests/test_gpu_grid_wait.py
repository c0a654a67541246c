"""The grid-wide waits of the persistent kernels (MI355X) at the workgroup
counts where their layout changes: one workgroup, the edges of 8, 16 and 64
lanes, the first counts with groups (65, 66), an uneven last group, the whole
device.  A solve's results depend on the count only through the order of
compensated sums, so every count must take the same iterations and agree with
the full grid to 1e-10 (the bar of the parity tests for parallel sums)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solve(cap, precision, side, solver):
    from mantle_convection_lab_amd import Input, Model
    from mantle_convection_lab_amd.learn import workload_keys
    m = Model(Input.from_keys(workload_keys(side, 1e5, 30.0, seed=3, precision=precision, warm_start=0,
                                               solver=solver)))
    m.ctx._ck(m.ctx.L.mcl_set_launch_cap(m.ctx.h, cap))
    print(f"[grid-wait] cap {cap} precision {precision} side {side} {solver}", flush=True)
    r = m.step()
    out = (r["uzawa"], r["inner"], m.field("D"), m.field("P"), m.field("T"))
    m.ctx.close()
    return out


# the FP64 solvers keep one row a thread in registers when the grid has a
# thread for every row, else they read the matrix: the smaller caps of the
# last three cases take the second form, the uncapped run the first
@pytest.mark.parametrize("precision,side,solver,caps", [
    (1, 128, "cg", [7, 8, 9, 16, 17, 63, 64, 65, 66, 129, 255]),
    (1, 32, "cg", [1, 2]),
    (0, 64, "cg", [1, 2, 7, 15]),
    (0, 32, "cg", [1, 3]),
    (0, 16, "jc", [1]),
    (0, 32, "jc", [1, 3]),
])
def test_workgroup_counts_agree(precision, side, solver, caps):
    ref = _solve(0, precision, side, solver)
    for cap in caps:
        got = _solve(cap, precision, side, solver)
        assert got[:2] == ref[:2]
        for a, b in zip(got[2:], ref[2:]):
            assert np.linalg.norm(a - b) <= 1e-10 * np.linalg.norm(b)
