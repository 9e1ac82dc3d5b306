"""Forms of the fused step's column waves against the oracle, bit for bit: AB3
tracers (two old levels, rotated) at every number of levels per lane and tracers
per wave, and the kernels for fields beyond 4 GiB (64-bit row offsets) with
every scheme and term."""
import dataclasses

import numpy as np
import pytest

from fesom2_amd import meshgen as mg

pytestmark = pytest.mark.gpu

AB3 = dict(AB_order=3)
EXTRAS = [dict(ver="PPM"), dict(ver="CDIFF", i_vert_diff=False), dict(ver="PPM", lim="NON", AB_order=3),
          dict(ver="CDIFF", hor="MUSCL", lim="NON"), dict(), dict(ver="UPW1", hor="UPW1", lim="NON")]


def _case(layers, ntr):
    mesh = mg.build_mesh(nx=20, ny=14, dx=20e3, jitter=0.2, seed=layers, cartesian=True, nlayers=layers, hmax=6250.0,
                         dz0=5.0 if layers > 60 else None, min_layers=4, max_layers=layers, topo="bumps",
                         bump_height=6000.0)
    return mesh, mg.build_state(mesh, seed=layers, ntr=ntr, dt=600.0, dx=20e3, kv_range=(1e-5, 1e-2))


def _check(mesh, st, schemes, nsteps=3):
    from fesom2_amd import gpu
    from oracle.oracle import Oracle
    k = np.arange(1, mesh.nl)
    w = (k[None, :] >= mesh.ulevels_nod2D[:, None]) & (k[None, :] < mesh.nlevels_nod2D[:, None])
    rng = np.random.default_rng(mesh.nl)
    old = []
    for o, s in zip(st.valuesold, schemes):
        older = np.where(w, o + rng.normal(0.0, 0.05, o.shape), 0.0)
        old.append(np.ascontiguousarray(np.stack([o, older], -1)) if s.get("AB_order") == 3 else o)
    ctx = gpu.context_for(mesh, st, schemes=schemes, valuesold=old)
    try:
        ctx.solve_tracers_ale(st.dt, nsteps)
        out = [ctx.tracer_download(i + 1) for i in range(st.ntr)]
    finally:
        ctx.close()
    v, vo = st.values.copy(), [o.copy() for o in old]
    o = Oracle(mesh)
    for _ in range(nsteps):
        o.step(st, v, vo, schemes=schemes)
    for i, (gv, gvo) in enumerate(out):
        np.testing.assert_array_equal(gv[w], v[i][w], err_msg=f"tracer {i + 1}")
        np.testing.assert_array_equal(gvo[w], vo[i][w], err_msg=f"tracer {i + 1} valuesold")


# layers, tracers: <1,2>, <1,1>, <2,2>, an odd last group, <2,1>; <3,2>; <2,1>
@pytest.mark.parametrize("rows", ["", "wide"])
@pytest.mark.parametrize("layers,schemes", [(31, [AB3] * 2), (31, [AB3] * 3), (47, [AB3] * 2), (47, [AB3] * 4),
                                            (63, [AB3] * 5), (70, [AB3] * 3), (95, [AB3] * 2), (100, [AB3]),
                                            (127, [AB3] * 2), (70, [AB3, dict(), AB3, dict(lim="NON")])])
def test_ab3_tracers(monkeypatch, layers, schemes, rows):
    monkeypatch.setenv("FGPU_STEP_ROWS", rows)
    mesh, st = _case(layers, len(schemes))
    print(f"[gpu] AB3, {layers} layers, {len(schemes)} tracers, rows {rows or 'as chosen'}", flush=True)
    _check(mesh, st, schemes)


@pytest.mark.parametrize("ntr", [2, 4])
@pytest.mark.parametrize("layers", [24, 47, 70, 95])
def test_far_pairs(monkeypatch, layers, ntr):
    """Tracers of one scheme, which share waves where their fields lie near each other."""
    monkeypatch.setenv("FGPU_STEP_ROWS", "wide")
    mesh, st = _case(layers, ntr)
    print(f"[gpu] far fields, {layers} layers, {ntr} tracers", flush=True)
    _check(mesh, st, [dict()] * ntr)


@pytest.mark.parametrize("split,diffusion", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("layers,ntr", [(31, 4), (63, 6), (70, 3), (127, 6)])
def test_far_schemes_and_terms(monkeypatch, layers, ntr, split, diffusion):
    monkeypatch.setenv("FGPU_STEP_ROWS", "wide")
    mesh, st = _case(layers, ntr)
    rng = np.random.default_rng(layers)
    if split:
        w_e = st.w * rng.uniform(0.2, 1.0, st.w.shape)
        st = dataclasses.replace(st, w_e=w_e, w_i=st.w - w_e, use_wsplit=True)
    if diffusion:
        st = dataclasses.replace(st, Ki=rng.uniform(20.0, 400.0, (mesh.nod2D, layers)), redi=True,
                                 slope_tapered=rng.normal(0.0, 0.01, (mesh.nod2D, layers, 3)))
    print(f"[gpu] far fields, extra schemes, {layers} layers, {ntr} tracers, split {split}, diffusion {diffusion}",
          flush=True)
    _check(mesh, st, EXTRAS[:ntr])


@pytest.mark.parametrize("ntr", [2, 3])
@pytest.mark.parametrize("layers", [31, 47, 70, 127])
def test_far_explicit_diffusion(monkeypatch, layers, ntr):
    """Pairs and single tracers with the explicit diffusion terms."""
    monkeypatch.setenv("FGPU_STEP_ROWS", "wide")
    mesh, st = _case(layers, ntr)
    rng = np.random.default_rng(layers)
    st = dataclasses.replace(st, Ki=rng.uniform(20.0, 400.0, (mesh.nod2D, layers)), redi=True,
                             slope_tapered=rng.normal(0.0, 0.01, (mesh.nod2D, layers, 3)))
    print(f"[gpu] far fields, explicit diffusion, {layers} layers, {ntr} tracers", flush=True)
    _check(mesh, st, [dict(i_vert_diff=i % 2 == 1) for i in range(ntr)])
