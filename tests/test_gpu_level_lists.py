"""Halo lists of the grid levels from LDS, rows in pairs of slots (MI355X).

The fused V-cycle phases (default) take their halo rows from lists that are
kept in LDS as far as the space goes and from memory past that; the unfused
sequence (MCL_MG_FUSE=0) uses no lists.  Both do the same operations in the
same order, so the first solves must be bit-identical: on the smallest mesh
with one grid level, on a mesh of three columns of base elements (levels whose
rows do not divide evenly among the workgroups), on one whose second level's
lists do not fit the space, and on a refined mesh (hanging nodes, rows longer
than a regular mesh's 18 slots).
"""
import math
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEYS = dict(level=6, mg_min_level=2, nprox=1, nproz=1, model_length=1.0, model_height=1.0, Rayleigh=1e6,
            A=math.log(1000.0), refT=0.0, T_ini=4, T_mantle_perturb=0.01, Q=0.0, theta=0.5, develop_mode=0,
            solver="cg", cg_precondition=1, accuracy=1e-8, citcom_solver_accu=1e-6, max_citcom_cycle=500,
            max_cg_cycle=200, schur_mode=1, top_v_bc="SV", bot_v_bc="SV", lef_v_bc="VS", rig_v_bc="VS",
            write_output=0, precision=1, warm_start=1)


def _solve(keys, refined, fuse):
    from mantle_convection_lab_amd import Input, Mesh, Model, amr
    saved = os.environ.pop("MCL_MG_FUSE", None)
    try:
        if not fuse:
            os.environ["MCL_MG_FUSE"] = "0"
        inp = Input.from_keys(keys)
        mesh = T0 = None
        if refined:
            def develop(X):
                return amr.developed_temperature(X, length=2.0, delta=0.05, nplumes=8, width=0.05)
            mesh = Mesh(inp, depth=refined)
            for _ in range(2):
                mesh = mesh.adapt(develop(mesh.level(-1)["X"]), refined, refined + 2)[0]
            T0 = develop(mesh.level(-1)["X"])
        m = Model(inp, mesh=mesh, T0=T0)
        if refined:
            m.ctx.buoyancy_force()
            m.ctx.viscosity()
            m.ctx.velocity_pressure_KGF_matrix()
            r = m.ctx.solve_velocity_pressure()
            recs = [(r.uzawa_cycles, r.inner_iterations)]
        else:
            recs = [(r["uzawa"], r["inner"]) for r in (m.step(), m.step())]
        out = m.field("D").copy(), m.field("P").copy(), recs
        m.ctx.close()
        return out
    finally:
        os.environ.pop("MCL_MG_FUSE", None)
        if saved is not None:
            os.environ["MCL_MG_FUSE"] = saved


@pytest.mark.parametrize("shape", ["level6", "3x1", "level9", "refined"])
def test_lists_and_unfused_sequence_bit_identical(shape):
    refined = 0
    if shape == "refined":
        from mantle_convection_lab_amd import amr
        keys, refined = amr.c3_keys(32, 2, Ra=1e6, contrast=1e3, warm_start=0)
    else:
        keys = {"level6": dict(KEYS), "3x1": dict(KEYS, nprox=3, model_length=3.0),
                "level9": dict(KEYS, level=9)}[shape]
    print(f"[gpu-level-lists] {shape}", flush=True)
    a, b = _solve(keys, refined, True), _solve(keys, refined, False)
    assert a[2] == b[2]
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
