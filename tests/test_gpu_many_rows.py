"""The FP64 inner solvers with many rows a thread (MI355X): a launch cap, as the
lanes of a batch have, leaves each of the 512 threads of a workgroup 16 rows.
Both solvers read a matrix that the caches do not hold, so a workgroup's rate of
algorithmic bytes shows whether its loads wait for each other: 28 GB/s for
conjugate gradients and for Jacobi sweeps (16.5 and 15.5 with every vector entry
gathered past the caches, or one column's load after the other)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver,side,cap", [("cg", 256, 16), ("jc", 128, 4)])
def test_rate_at_sixteen_rows_a_thread(solver, side, cap):
    from mantle_convection_lab_amd import Input, Model
    from mantle_convection_lab_amd.learn import workload_keys
    m = Model(Input.from_keys(workload_keys(side, 1e5, 10.0, seed=1, precision=0, warm_start=0, zero_P=1,
                                            solver=solver, max_citcom_cycle=1, max_cg_cycle=100)))
    c = m.ctx
    c._ck(c.L.mcl_set_launch_cap(c.h, cap))
    c.buoyancy_force()
    c.viscosity()
    c.velocity_pressure_KGF_matrix()
    print(f"[many-rows] {solver} {side} on {cap} workgroups", flush=True)
    s = [c.solve_velocity_pressure() for _ in range(3)]
    nv = 2 * side * side - 2
    nnz = int(c.get_matrix(m.finest, "K")[0].sum())
    per = 12 * nnz + (11 if solver == "cg" else 3) * 8 * nv
    rate = max(per * q.inner_iterations / (q.device_ms * 1e-3) for q in s) / cap / 1e9
    print(f"[many-rows] {rate:.1f} GB/s a workgroup", flush=True)
    m.ctx.close()
    assert rate >= 20
