"""Meshes at the edge of what mcl_mesh_upload takes (MI355X)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _mesh(depth):
    """(input, uniform mesh at that depth on the node grid of 64 x 64)"""
    from mantle_convection_lab_amd import Input, Mesh
    from mantle_convection_lab_amd.learn import workload_keys
    inp = Input.from_keys(dict(workload_keys(64, 1e4, 10.0, seed=1, precision=0, warm_start=0), mg_min_level=2))
    return inp, Mesh(inp, depth=depth)


def test_equation_at_a_node_without_elements():
    """A node of no element may carry a velocity equation: its row is empty,
    its diagonal zero, and the solve ends with the error for NaN."""
    from mantle_convection_lab_amd import _native as N
    from mantle_convection_lab_amd.model import Context, MclError
    inp, mesh = _mesh(4)
    lv, v = mesh.level(-1), mesh.views()[mesh.nlev - 1]
    keep = []

    def put(field, a, kind):
        a = np.ascontiguousarray(a)
        keep.append(a)
        setattr(v, field, a.ctypes.data_as(kind))

    pos = 40
    new = lv["node"][pos - 1] + 1
    assert new < lv["node"][pos]
    ids = np.insert(lv["id"], pos, [lv["neq"], -1], axis=1).astype(np.int32)
    put("node", np.insert(lv["node"], pos, new).astype(np.int32), N.PI)
    put("id", ids, N.PI)
    put("heat_id", np.insert(lv["heat_id"], pos, -1).astype(np.int32), N.PI)
    put("v_bc", np.insert(lv["v_bc"], pos, 0, axis=1).astype(np.int8), N.PB)
    put("v_bc_val", np.insert(lv["v_bc_val"], pos, 0.0, axis=1), N.PD)
    put("T_bc", np.insert(lv["T_bc"], pos, 0).astype(np.int8), N.PB)
    put("T_bc_val", np.insert(lv["T_bc_val"], pos, 0.0), N.PD)
    put("X", np.insert(lv["X"], pos, 0.5, axis=1), N.PD)
    v.nno, v.neq = lv["nno"] + 1, lv["neq"] + 1
    v.interp_n = v.interp_eq = N.PI()
    c = Context()
    print("[upload] an equation at a node without elements", flush=True)
    views = (N.MeshView * 1)(v)
    c.upload(views, {v.lev: dict(nel=lv["nel"], nno=v.nno, neq=v.neq, neqT=lv["neqT"])})
    c.set_control(inp.control())
    c.set_field(v.lev, "T", np.linspace(1.0, 0.0, v.nno))
    c.buoyancy_force()
    c.viscosity()
    c.velocity_pressure_KGF_matrix()
    assert c.get_field(v.lev, "F").size == v.neq and c.get_matrix(v.lev, "K")[0][lv["neq"]] == 0
    with pytest.raises(MclError, match="NaN"):
        c.solve_velocity_pressure()
    c.close()


def test_no_mesh_after_a_failed_upload():
    """A list of levels that do not nest is refused once its levels are built;
    the context then has no mesh, not the tables of the one before, and takes
    the next upload."""
    from mantle_convection_lab_amd import Model
    from mantle_convection_lab_amd import _native as N
    from mantle_convection_lab_amd.model import MclError
    inp, mesh = _mesh(3)
    finer = _mesh(4)[1]
    m, ref = Model(inp, mesh=mesh), Model(inp, mesh=mesh)
    want = ref.step()
    c = m.ctx
    good = mesh.views()
    bad = (N.MeshView * 2)(finer.views()[finer.nlev - 1], good[mesh.nlev - 1])
    print("[upload] a coarser level with nodes that the finest has not", flush=True)
    assert c.L.mcl_mesh_upload(c.h, bad, 2) == 1
    for call in (c.viscosity, c.buoyancy_force, c.velocity_pressure_KGF_matrix, c.solve_velocity_pressure,
                 c.update_temperature):
        with pytest.raises(MclError, match="no mesh"):
            call()
    with pytest.raises(MclError):
        c.get_field(m.finest, "T")
    m.ctx.close()
    m = Model(inp, mesh=mesh)
    c = m.ctx
    assert c.L.mcl_mesh_upload(c.h, bad, 2) == 1
    c.upload(good, c.levels)
    for k in range(mesh.nlev):
        c.set_field(mesh.level_struct(k).lev, "T", mesh.initial_temperature(k))
    c.set_model_time(0.0)
    got = m.step()
    assert (got["uzawa"], got["inner"]) == (want["uzawa"], want["inner"])
    assert all(np.array_equal(m.field(f), ref.field(f)) for f in ("D", "P", "T"))
    m.ctx.close()
    ref.ctx.close()
