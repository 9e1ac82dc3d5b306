"""The column waves of the fused step (levels per lane and tracers per wave
chosen from the column depth and the tracer count) against the oracle, bit for
bit, at the depths where a lane group is just full or just too short: 32, 33,
64, 65, 96, 97 and 128 interfaces, with even and odd tracer counts, one tracer
group or several in the vertical solve, and tracers of different schemes, which
keep a wave each."""
import numpy as np
import pytest

from fesom2_amd import meshgen as mg

pytestmark = pytest.mark.gpu

MIXED = [dict(), dict(hor="UPW1", ver="UPW1"), dict(lim="NON"), dict(AB_order=2, ph=0.5, pv=0.0)]


def _case(layers, ntr):
    mesh = mg.build_mesh(nx=20, ny=14, dx=20e3, jitter=0.2, seed=layers, cartesian=True, nlayers=layers, hmax=6250.0,
                         dz0=5.0 if layers > 60 else None, min_layers=4, max_layers=layers, topo="bumps",
                         bump_height=6000.0)
    return mesh, mg.build_state(mesh, seed=layers, ntr=ntr, dt=600.0, dx=20e3, kv_range=(1e-5, 1e-2))


@pytest.mark.parametrize("layers,ntr,schemes", [
    (4, 1, None), (31, 2, None), (31, 5, None), (31, 4, MIXED), (32, 3, None), (47, 11, None), (63, 2, None),
    (63, 4, MIXED), (64, 3, None), (95, 3, None), (95, 4, MIXED), (96, 2, None), (127, 1, None), (127, 21, None)])
def test_column_waves_bitwise(layers, ntr, schemes):
    from fesom2_amd import gpu
    from oracle.oracle import Oracle
    mesh, st = _case(layers, ntr)
    print(f"[gpu] {layers} layers, {ntr} tracers, 2 steps", flush=True)
    ctx = gpu.context_for(mesh, st, schemes=schemes)
    try:
        ctx.solve_tracers_ale(st.dt, 2)
        out = [ctx.tracer_download(i + 1) for i in range(ntr)]
    finally:
        ctx.close()
    v, vo = st.values.copy(), st.valuesold.copy()
    o = Oracle(mesh)
    for _ in range(2):
        o.step(st, v, vo, schemes=schemes)
    k = np.arange(1, mesh.nl)
    w = (k[None, :] >= mesh.ulevels_nod2D[:, None]) & (k[None, :] < mesh.nlevels_nod2D[:, None])
    for i, (gv, gvo) in enumerate(out):
        np.testing.assert_array_equal(gv[w], v[i][w], err_msg=f"tracer {i + 1}")
        np.testing.assert_array_equal(gvo[w], vo[i][w], err_msg=f"tracer {i + 1} valuesold")
