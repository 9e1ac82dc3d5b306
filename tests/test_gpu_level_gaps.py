"""Meshes on which the elements beside an edge share no level and leave a gap
between their ranges: the reference's segments of both reach into the gap
(oce_adv_tra_hor.F90:166-249). The fused step against the oracle, bit for bit,
with the upper element on either side of the edge, for every scheme and term,
both old levels of an AB3 tracer and 64-bit row offsets; and it is the fused
step that runs."""
import dataclasses

import numpy as np
import pytest

from fesom2_amd import meshgen as mg

pytestmark = pytest.mark.gpu

SCHEMES = [dict(), dict(hor="UPW1", ver="UPW1"), dict(lim="NON", ph=0.5, pv=0.0), dict(hor="MUSCL", AB_order=3),
           dict(ver="PPM"), dict(ver="CDIFF", i_vert_diff=False)]


def _gap_mesh(layers):
    """Five edges with a gap, alternately under their first and their second element."""
    mesh = mg.build_mesh(nx=20, ny=14, dx=20e3, jitter=0.2, seed=layers, cartesian=True, nlayers=layers, hmax=6250.0,
                         dz0=5.0 if layers > 60 else None, min_layers=4, max_layers=layers, topo="bumps",
                         bump_height=3000.0)
    nl, ul = mesh.nlevels.copy(), mesh.ulevels.copy()
    nmin, umax = mesh.nlevels_nod2D_min.copy(), mesh.ulevels_nod2D_max.copy()
    taken, gaps = np.zeros(mesh.nod2D, bool), 0
    for e in np.flatnonzero((mesh.edge_tri >= 0).all(1) & (mesh.nlevels[mesh.edge_tri].min(1) > 12)):
        a, b = mesh.edge_tri[e] if gaps % 2 == 0 else mesh.edge_tri[e][::-1]
        nodes = mesh.elem2D_nodes[[a, b]].ravel()
        if taken[mesh.elem2D_nodes[np.isin(mesh.elem2D_nodes, nodes).any(1)]].any():
            continue
        nl[a], ul[b] = 4, 8 + gaps
        nmin[mesh.elem2D_nodes[a]] = 4
        umax[mesh.elem2D_nodes[b]] = 8 + gaps
        taken[nodes] = True
        gaps += 1
        if gaps == 5:
            break
    assert gaps == 5
    return dataclasses.replace(mesh, nlevels=nl, ulevels=ul, nlevels_nod2D_min=nmin, ulevels_nod2D_max=umax)


def _check(mesh, st, schemes, nsteps=2):
    from fesom2_amd import gpu
    from oracle.oracle import Oracle
    schemes = schemes or [dict()] * st.ntr
    old = [np.ascontiguousarray(np.stack([o, 0.9 * o], -1)) if s.get("AB_order") == 3 else o
           for o, s in zip(st.valuesold, schemes)]
    ctx = gpu.context_for(mesh, st, schemes=schemes, valuesold=old)
    try:
        ctx.solve_tracers_ale(st.dt, nsteps - 1)
        ctx.profile_enable(True)
        ctx.solve_tracers_ale(st.dt, 1)
        names = set(ctx.profile())
        out = [ctx.tracer_download(i + 1) for i in range(st.ntr)]
    finally:
        ctx.close()
    v, vo = st.values.copy(), [o.copy() for o in old]
    o = Oracle(mesh)
    for _ in range(nsteps):
        o.step(st, v, vo, schemes=schemes)
    k = np.arange(1, mesh.nl)
    w = (k[None, :] >= mesh.ulevels_nod2D[:, None]) & (k[None, :] < mesh.nlevels_nod2D[:, None])
    for i, (gv, gvo) in enumerate(out):
        np.testing.assert_array_equal(gv[w], v[i][w], err_msg=f"tracer {i + 1}")
        np.testing.assert_array_equal(gvo[w], vo[i][w], err_msg=f"tracer {i + 1} valuesold")
    assert "kA_edge" in names and "k_edge_flux" not in names


@pytest.mark.parametrize("rows", ["", "wide"])
@pytest.mark.parametrize("terms", ["", "diffusion", "redi"])
@pytest.mark.parametrize("layers,ntr", [(24, 2), (31, 6), (63, 6), (70, 6), (127, 3)])
def test_level_gaps(monkeypatch, layers, ntr, terms, rows):
    monkeypatch.setenv("FGPU_STEP_ROWS", rows)
    mesh = _gap_mesh(layers)
    st = mg.build_state(mesh, seed=layers, ntr=ntr, dt=600.0, dx=20e3, kv_range=(1e-5, 1e-2))
    rng = np.random.default_rng(layers)
    if terms:
        w_e = st.w * rng.uniform(0.2, 1.0, st.w.shape)
        st = dataclasses.replace(st, w_e=w_e, w_i=st.w - w_e, use_wsplit=True,
                                 Ki=rng.uniform(20.0, 400.0, (mesh.nod2D, layers)))
    if terms == "redi":
        st = dataclasses.replace(st, redi=True, slope_tapered=rng.normal(0.0, 0.01, (mesh.nod2D, layers, 3)))
    print(f"[gpu] level gaps, {layers} layers, {ntr} tracers, terms {terms or 'none'}, rows {rows or 'as chosen'}", flush=True)
    _check(mesh, st, SCHEMES[:ntr] if ntr > 2 else None)
