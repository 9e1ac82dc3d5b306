"""The library's host code on a stand-in of the HIP runtime (host_runtime.c):
device memory is host memory and no kernel runs, so these tests see the order
of calls and the handling of failed allocations, without a GPU. Each runs in a
process of its own, the stand-in loaded first."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

SETUP = """
import ctypes, os, sys
rt = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
rt.host_live_bytes.restype = ctypes.c_size_t
import numpy as np
from fesom2_amd import gpu, meshgen as mg
mesh = mg.build_mesh(nx=12, ny=10, dx=20e3, jitter=0.2, seed=0, cartesian=True, nlayers=8, hmax=4000.0, min_layers=4,
                     max_layers=8, topo="bumps", bump_height=1500.0)
st = mg.build_state(mesh, seed=0, ntr=2, dt=600.0, dx=20e3)
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("hip") / "libhost_runtime.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", so, os.path.join(HERE, "host_runtime.c")], check=True)
    return so


def _run(runtime, code, **env):
    r = subprocess.run([sys.executable, "-c", SETUP + textwrap.dedent(code), runtime], cwd=os.path.dirname(HERE),
                       env={**os.environ, **env}, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


@pytest.mark.parametrize("step", ["fused", "staged"])
def test_fills_are_done_before_the_stream_uses_them(runtime, step):
    """Buffers that start at zero are filled before anything of the context's
    stream can read or write them."""
    _run(runtime, """
        ctx = gpu.context_for(mesh, st, schemes=dict(i_vert_diff=False))
        assert rt.host_hazards() == 0, "set-up"
        n, L = mesh.nod2D, mesh.nl - 1
        ctx.set_ki(np.ones((n, L)), np.zeros((n, L, 3)), True)
        ctx.solve_tracers_ale(st.dt, 2)
        assert rt.host_hazards() == 0, "step"
        ctx.init_tracers_AB(1)
        ctx.do_oce_adv_tra(st.dt, 1)
        ctx.diff_tracers_ale(st.dt, 1)
        assert rt.host_hazards() == 0, "per-tracer calls"
        ctx.tracer_config(2, 2, AB_order=3)
        ctx.solve_tracers_ale(st.dt, 1)
        assert rt.host_hazards() == 0, "AB3"
        ctx.close()
        ctx = gpu.Context()
        ctx.mesh_init(mesh)
        ctx.set_uv(st.uv)
        ctx.vert_vel_ale(st.dt)
        assert rt.host_hazards() == 0, "vertical velocity"
        i = np.arange(100)
        ctx.ssh_set_matrix(1 + np.arange(101), 1 + i, 1.0 + i)
        ctx.ssh_solve_preconditioner(2)
        ctx.nn_init(0)
        ctx.nn_loss_grad(np.ones((1, 100)), np.ones((1, 100)))
        assert rt.host_hazards() == 0, "learned preconditioner"
        ctx.close()
        """, FGPU_STEP=step)


@pytest.mark.parametrize("slots", ["one", "all"])
def test_staged_buffers_after_a_failed_allocation(runtime, slots):
    """A call repeated after FGPU_ERR_NOMEM allocates what the failed one could
    not, whichever allocation failed, also where the buffers of the per-tracer
    calls are replaced by those of the batched per-stage step."""
    _run(runtime, f"""
        def calls(ctx):
            ctx.init_tracers_AB(1)
            if {slots == "all"}:
                ctx.solve_tracers_ale(st.dt, 1)
        ctx = gpu.context_for(mesh, st)
        base = rt.host_live_bytes()
        calls(ctx)
        want = rt.host_live_bytes() - base
        ctx.close()
        failed = 0
        for k in range(100):
            ctx = gpu.context_for(mesh, st)
            base = rt.host_live_bytes()
            rt.host_fail_in(k)
            try:
                calls(ctx)
            except gpu.FesomGpuError as e:
                assert "hipMalloc" in str(e)
                failed += 1
            else:
                assert rt.host_fail_left() >= 0
                rt.host_fail_in(-1)
                break
            ctx.init_tracers_AB(1)
            calls(ctx)
            assert rt.host_live_bytes() - base == want, k
            ctx.close()
        assert failed == {9 if slots == "one" else 11}
        """, FGPU_STEP="staged")


def test_tracers_after_a_failed_allocation(runtime):
    """fgpu_tracers_init releases the former tracers first: after it has failed
    there are none, and a repeated call sets them up."""
    _run(runtime, """
        ctx = gpu.context_for(mesh, st)
        for k in range(11):
            rt.host_fail_in(k)
            try:
                ctx.tracers_init(3)
                raise AssertionError(k)
            except gpu.FesomGpuError as e:
                assert "hipMalloc" in str(e)
            for call in (lambda: ctx.solve_tracers_ale(st.dt, 1), lambda: ctx.init_tracers_AB(1),
                         lambda: ctx.tracer_config(1, 1), lambda: ctx.tracer_content(1),
                         lambda: ctx.tracer_upload(1, st.values[0], st.valuesold[0])):
                try:
                    call()
                    raise AssertionError(k)
                except gpu.FesomGpuError as e:
                    assert "tracers not initialised" in str(e), (k, e)
        ctx.tracers_init(2)
        for i in range(2):
            ctx.tracer_config(i + 1, i + 1)
            ctx.tracer_upload(i + 1, st.values[i], st.valuesold[i])
        ctx.solve_tracers_ale(st.dt, 1)
        ctx.close()
        """)


def test_ssh_matrix_after_a_failed_allocation(runtime):
    """A matrix of another size after one that could not be allocated gets
    arrays of its own size."""
    _run(runtime, """
        def diagonal(ctx, n):
            ctx.ssh_set_matrix(1 + np.arange(n + 1), 1 + np.arange(n), np.ones(n))
        ctx = gpu.Context()
        base = rt.host_live_bytes()
        diagonal(ctx, 2000)
        want = rt.host_live_bytes() - base
        ctx.close()
        for k in range(19):
            ctx = gpu.Context()
            base = rt.host_live_bytes()
            rt.host_fail_in(k)
            try:
                diagonal(ctx, 50)
                raise AssertionError(k)
            except gpu.FesomGpuError as e:
                assert "hipMalloc" in str(e)
            diagonal(ctx, 2000)
            assert rt.host_live_bytes() - base == want, k
            ctx.close()
        """)


def test_contexts_share_the_download_threads(runtime):
    """The threads of large downloads come once, whatever the number of
    contexts, and end with the last context that has used them."""
    _run(runtime, """
        def threads():
            return len(os.listdir("/proc/self/task"))
        big = mg.build_mesh(nx=93, ny=60, dx=20e3, jitter=0.2, seed=0, cartesian=True, nlayers=47, hmax=4000.0,
                            min_layers=4, max_layers=47, topo="bumps", bump_height=1500.0)
        bst = mg.build_state(big, seed=0, ntr=1, dt=600.0, dx=20e3)
        base = threads()
        ctx = [gpu.context_for(big, bst) for _ in range(3)]
        assert threads() == base
        n = []
        for c in ctx:
            v, vo = c.tracer_download(1)
            assert np.array_equal(v, bst.values[0]) and np.array_equal(vo, bst.valuesold[0])
            n.append(threads() - base)
        assert n[0] > 0 and n == [n[0]] * 3, n
        ctx[1].close()
        ctx[0].close()
        assert threads() - base == n[0]
        assert np.array_equal(ctx[2].tracer_download(1)[0], bst.values[0])
        ctx[2].close()
        assert threads() == base
        c = gpu.context_for(big, bst)
        assert np.array_equal(c.tracer_download(1)[0], bst.values[0])
        c.close()
        assert threads() == base
        """)


def test_vertical_after_a_failed_allocation(runtime):
    """fgpu_set_vertical repeated after FGPU_ERR_NOMEM has every array, those of
    the implicit diffusion's levels among them."""
    _run(runtime, """
        ctx = gpu.Context()
        ctx.mesh_init(mesh)
        want = rt.host_live_bytes()
        ctx.close()
        failed = 0
        for k in range(200):
            ctx = gpu.Context()
            rt.host_fail_in(k)
            try:
                ctx.mesh_init(mesh)
            except gpu.FesomGpuError as e:
                assert "hipMalloc" in str(e)
                if ctx.nl:   # the mesh is there, its vertical geometry is not
                    failed += 1
                    ctx.set_vertical(mesh)
                    assert rt.host_live_bytes() == want, k
            else:
                rt.host_fail_in(-1)
                break
            ctx.close()
        assert failed == 12
        """)


@pytest.mark.parametrize("nx,ny,layers", [(64, 64, 64), (65, 63, 64), (64, 66, 64), (87, 100, 63), (128, 96, 127), (70, 50, 121)])
def test_download_in_pieces(runtime, nx, ny, layers):
    """Fields around a whole number of slots and pieces come back whole, several at once too."""
    _run(runtime, f"""
        m = mg.build_mesh(nx={nx}, ny={ny}, dx=20e3, jitter=0.2, seed=0, cartesian=True, nlayers={layers}, hmax=4000.0,
                          min_layers=4, max_layers={layers}, topo="bumps", bump_height=1500.0)
        s = mg.build_state(m, seed=0, ntr=1, dt=600.0, dx=20e3)
        rng = np.random.default_rng(0)
        v, vo = rng.normal(size=(2, m.nod2D, {layers}))
        c = gpu.context_for(m, s)
        c.tracer_upload(1, v, vo)
        for _ in range(3):
            gv, gvo = c.tracer_download(1)
            assert np.array_equal(gv, v) and np.array_equal(gvo, vo)
        c.vert_vel_ale(s.dt)
        w = c.vert_vel_download()
        assert np.array_equal(w["w"], s.w) and np.array_equal(w["w_i"], s.w_i) and np.array_equal(w["hnode_new"], m.hnode_new)
        c.close()
        """)


@pytest.mark.parametrize("nx,ny", [(8, 6), (38, 36), (53, 27), (67, 61), (151, 113)])
def test_mesh_set_up_in_parts(runtime, nx, ny):
    """The up- and downwind triangles are the oracle's, whatever number of parts the edges are searched in."""
    _run(runtime, f"""
        from oracle.oracle import Oracle
        m = mg.build_mesh(nx={nx}, ny={ny}, dx=20e3, jitter=0.2, seed=1, cartesian=True, nlayers=4, hmax=4000.0,
                          min_layers=3, max_layers=4, topo="bumps", bump_height=1500.0)
        s = mg.build_state(m, seed=0, ntr=1, dt=600.0, dx=20e3)
        c = gpu.context_for(m, s)
        assert np.array_equal(c.edge_up_dn_tri(m.edge2D) - 1, Oracle(m).edge_up_dn_tri)   # 0: no such triangle
        c.close()
        """)
