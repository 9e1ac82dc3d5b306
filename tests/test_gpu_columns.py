"""The column waves of the fused step (levels per lane and tracers per wave
chosen from the column depth and the tracer count) against the oracle, bit for
bit: at the depths where a lane group is just full or just too short (32, 33,
64, 65, 96, 97 and 128 interfaces), with even and odd tracer counts, one tracer
group or several in the vertical solve, and tracers of different schemes, which
keep a wave each; with 64-bit row offsets; around a node with more edges than
the waves keep in registers; for tracers whose values reach the smallest
doubles; and on a mesh with a level gap across an edge, which steps through the
per-stage kernels."""
import dataclasses

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


def _check(mesh, st, schemes=None):
    from fesom2_amd import gpu
    from oracle.oracle import Oracle
    ctx = gpu.context_for(mesh, st, schemes=schemes)
    try:
        ctx.solve_tracers_ale(st.dt, 2)
        out = [ctx.tracer_download(i + 1) for i in range(st.ntr)]
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


@pytest.mark.parametrize("layers,ntr,schemes", [
    (4, 1, None), (31, 2, None), (31, 5, None), (31, 4, MIXED), (32, 3, None), (47, 11, None), (63, 2, None),
    (63, 4, MIXED), (64, 3, None), (95, 3, None), (95, 4, MIXED), (96, 2, None), (127, 1, None), (127, 21, None)])
def test_column_waves_bitwise(layers, ntr, schemes):
    mesh, st = _case(layers, ntr)
    print(f"[gpu] {layers} layers, {ntr} tracers, 2 steps", flush=True)
    _check(mesh, st, schemes)


@pytest.mark.parametrize("layers,ntr,schemes", [(24, 3, None), (47, 2, MIXED[:2]), (70, 3, None), (100, 1, None)])
def test_wide_row_offsets(monkeypatch, layers, ntr, schemes):
    monkeypatch.setenv("FGPU_STEP_ROWS", "wide")
    mesh, st = _case(layers, ntr)
    print(f"[gpu] 64-bit row offsets, {layers} layers, {ntr} tracers", flush=True)
    _check(mesh, st, schemes)


@pytest.mark.parametrize("layers,ntr", [(12, 2), (40, 1), (40, 5), (70, 2)])
def test_node_of_many_edges(layers, ntr):
    """A hub with 15 spokes inside two rings."""
    m, r = 15, 3e-3
    ang = 2 * np.pi * np.arange(m) / m
    ring = np.stack([np.cos(ang), np.sin(ang)], 1)
    coord = np.concatenate([[[0.0, 0.0]], r * ring, 2.2 * r * ring]) + [1.0, 0.1]
    i, j = np.arange(m), (np.arange(m) + 1) % m
    elem = np.concatenate([np.stack([0 * i, 1 + i, 1 + j], 1), np.stack([1 + i, 1 + m + i, 1 + j], 1),
                           np.stack([1 + j, 1 + m + i, 1 + m + j], 1)])
    depth = -(3000.0 + 1500.0 * np.sin(3.0 * np.arange(len(coord))))
    mesh = mg.assemble_mesh(coord, elem, L=2 * np.pi, cartesian=False, zbar=-np.linspace(0.0, 4500.0, layers + 1),
                            depth=depth, min_layers=4, max_layers=layers)
    st = mg.build_state(mesh, seed=1, ntr=ntr, dt=300.0, kv_range=(1e-5, 1e-2))
    assert np.bincount(mesh.edges.ravel()).max() == m
    print(f"[gpu] hub of {m} edges, {layers} layers, {ntr} tracers", flush=True)
    _check(mesh, st)


@pytest.mark.parametrize("layers,ntr", [(24, 2), (47, 4), (70, 2)])
def test_tiny_values(layers, ntr):
    """Values from 1e-250 down through the subnormal numbers to zero beside one of order one."""
    mesh, st = _case(layers, ntr)
    rng = np.random.default_rng(3)
    v = st.values.copy()
    v[-1] = np.where(v[-1] != 0.0, 10.0 ** -rng.uniform(250.0, 330.0, v[-1].shape), 0.0)
    v[-1][: mesh.nod2D // 4] = 1.0
    st = dataclasses.replace(st, values=v, valuesold=v.copy(), ids=np.array([301] * ntr, np.int32))
    print(f"[gpu] tiny values, {layers} layers, {ntr} tracers", flush=True)
    _check(mesh, st)


def test_level_gap_across_an_edge():
    mesh, st = _case(24, 2)
    e = int(np.flatnonzero((mesh.edge_tri >= 0).all(1) & (mesh.nlevels[mesh.edge_tri].min(1) > 12))[50])
    a, b = mesh.edge_tri[e]
    nl, ul = mesh.nlevels.copy(), mesh.ulevels.copy()
    nl[a], ul[b] = 4, 8
    nmin, umax = mesh.nlevels_nod2D_min.copy(), mesh.ulevels_nod2D_max.copy()
    nmin[mesh.elem2D_nodes[a]], umax[mesh.elem2D_nodes[b]] = 4, 8
    gap = dataclasses.replace(mesh, nlevels=nl, ulevels=ul, nlevels_nod2D_min=nmin, ulevels_nod2D_max=umax)
    print("[gpu] level gap", flush=True)
    _check(gap, st)


@pytest.mark.parametrize("path", ["fused", "staged"])
@pytest.mark.parametrize("layers,ntr,redi", [(7, 9, True), (8, 3, True), (31, 3, True), (32, 2, False), (63, 3, True),
                                             (64, 2, True), (70, 2, False), (127, 2, True)])
def test_explicit_diffusion_waves(monkeypatch, path, layers, ntr, redi):
    """The explicit diffusion terms where a lane group just holds a column, or
    takes it in two or three passes."""
    mesh, st = _case(layers, ntr)
    rng = np.random.default_rng(layers)
    Ki = rng.uniform(20.0, 400.0, (mesh.nod2D, layers))
    S = rng.normal(0.0, 0.01, (mesh.nod2D, layers, 3)) if redi else None
    st = dataclasses.replace(st, Ki=Ki, slope_tapered=S, redi=redi)
    schemes = [dict(i_vert_diff=i % 2 == 1) for i in range(ntr)]
    if path == "staged":
        monkeypatch.setenv("FGPU_STEP", "staged")
    print(f"[gpu] explicit diffusion, {layers} layers, {ntr} tracers, {path}", flush=True)
    _check(mesh, st, schemes)


EXTRAS = [dict(ver="PPM"), dict(ver="CDIFF", i_vert_diff=False), dict(ver="PPM", lim="NON"), dict(ver="CDIFF", hor="MUSCL", lim="NON"),
          dict(), dict(ver="UPW1", hor="UPW1", lim="NON")]


@pytest.mark.parametrize("split,diffusion", [(True, False), (False, True), (True, True)])
@pytest.mark.parametrize("layers,ntr", [(4, 6), (31, 4), (32, 6), (63, 6), (64, 3), (95, 1), (127, 6)])
def test_extra_schemes_and_terms(layers, ntr, split, diffusion):
    """CDIFF and PPM tracers, the split vertical velocity (implicit upwind step
    of the low-order solution, its rows in the vertical solve), Ki with Redi and
    tracers without implicit vertical diffusion."""
    mesh, st = _case(layers, ntr)
    rng = np.random.default_rng(layers)
    schemes = EXTRAS[:ntr]
    if split:
        w_e = st.w * rng.uniform(0.2, 1.0, st.w.shape)
        st = dataclasses.replace(st, w_e=w_e, w_i=st.w - w_e, use_wsplit=True)
    if diffusion:
        st = dataclasses.replace(st, Ki=rng.uniform(20.0, 400.0, (mesh.nod2D, layers)), redi=True,
                                 slope_tapered=rng.normal(0.0, 0.01, (mesh.nod2D, layers, 3)))
    print(f"[gpu] extra schemes, {layers} layers, {ntr} tracers, split {split}, diffusion {diffusion}", flush=True)
    _check(mesh, st, schemes)


@pytest.mark.parametrize("ivd,split", [(True, False), (False, False), (True, True)])
@pytest.mark.parametrize("layers", [32, 33, 40, 41, 64, 65, 127])
def test_per_tracer_calls(layers, ivd, split):
    """The per-tracer calls, by (row, level) pairs up to 32 levels and by rows of
    up to 64 levels per wave beyond, with the diffusion terms and the W split."""
    from fesom2_amd import gpu
    from oracle.oracle import Oracle
    mesh, st = _case(layers, 2)
    rng = np.random.default_rng(layers)
    st = dataclasses.replace(st, Ki=rng.uniform(20.0, 400.0, (mesh.nod2D, layers)), redi=True,
                             slope_tapered=rng.normal(0.0, 0.01, (mesh.nod2D, layers, 3)))
    if split:
        w_e = st.w * rng.uniform(0.2, 1.0, st.w.shape)
        st = dataclasses.replace(st, w_e=w_e, w_i=st.w - w_e, use_wsplit=True)
    schemes = dict(i_vert_diff=ivd)
    print(f"[gpu] per-tracer calls, {layers} layers, ivd {ivd}, split {split}", flush=True)
    ctx = gpu.context_for(mesh, st, schemes=schemes)
    o = Oracle(mesh)
    k = np.arange(1, mesh.nl)
    w = (k[None, :] >= mesh.ulevels_nod2D[:, None]) & (k[None, :] < mesh.nlevels_nod2D[:, None])
    e = mesh.edge_tri
    no2 = e[:, 1] < 0
    lo = np.where(no2, mesh.ulevels[e[:, 0]], np.minimum(mesh.ulevels[e[:, 0]], mesh.ulevels[e[:, 1]]))
    hi = np.where(no2, mesh.nlevels[e[:, 0]], np.maximum(mesh.nlevels[e[:, 0]], mesh.nlevels[e[:, 1]]))
    em = (k[None, :] >= lo[:, None]) & (k[None, :] < hi[:, None])
    try:
        ctx.init_tracers_AB(2)
        grad = ctx.work(2, "edge_up_dn_grad", (mesh.edge2D, layers, 4))
        ctx.do_oce_adv_tra(st.dt, 2)
        hor = ctx.work(2, "del_ttf_advhoriz", (mesh.nod2D, layers))
        ctx.diff_tracers_ale(st.dt, 2)
        gv, gvo = ctx.tracer_download(2)
    finally:
        ctx.close()
    v, vo = st.values[1].copy(), st.valuesold[1].copy()
    out = o.adv_stage(st, v, vo, ID=int(st.ids[1]), i_vert_diff=ivd)
    o.diff_stage(st)
    np.testing.assert_array_equal(grad[em], out["edge_up_dn_grad"][em])
    np.testing.assert_array_equal(hor[w], out["del_ttf_advhoriz"][w])
    np.testing.assert_array_equal(gv[w], v[w])
    np.testing.assert_array_equal(gvo[w], vo[w])
