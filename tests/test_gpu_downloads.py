"""Downloads below and above the size from which they go through pinned slots in
pieces, and from several threads at once."""
import threading

import numpy as np
import pytest

from fesom2_amd import meshgen as mg

pytestmark = pytest.mark.gpu


def _context(nx, layers, seed):
    from fesom2_amd import gpu
    mesh = mg.build_mesh(nx=nx, ny=60, dx=20e3, jitter=0.2, seed=1, cartesian=True, nlayers=layers, hmax=4000.0,
                         min_layers=4, max_layers=layers, topo="bumps", bump_height=3000.0)
    st = mg.build_state(mesh, seed=seed, ntr=2, dt=600.0, dx=20e3)
    rng = np.random.default_rng(seed)
    v, vo = rng.normal(size=(2, mesh.nod2D, layers)), rng.normal(size=(2, mesh.nod2D, layers))
    ctx = gpu.context_for(mesh, st)
    for i in range(2):
        ctx.tracer_upload(i + 1, v[i], vo[i])
    return ctx, v, vo


# bytes of a tracer and its old level: 3.9, 4.2, 6.0 and 35 MB
@pytest.mark.parametrize("nx,layers", [(87, 47), (93, 47), (89, 71), (300, 121)])
def test_download_returns_the_fields(nx, layers):
    print(f"[gpu] downloads {nx} x 60 nodes, {layers} layers", flush=True)
    ctx, v, vo = _context(nx, layers, nx)
    try:
        for _ in range(2):
            for i in range(2):
                gv, gvo = ctx.tracer_download(i + 1)
                np.testing.assert_array_equal(gv, v[i])
                np.testing.assert_array_equal(gvo, vo[i])
    finally:
        ctx.close()


def test_downloads_from_several_threads():
    print("[gpu] downloads from four threads, two contexts", flush=True)
    cases = [_context(100, 60, s) for s in (1, 2)]
    wrong = []

    def work(ctx, v, vo, i):
        for _ in range(5):
            gv, gvo = ctx.tracer_download(i + 1)
            if not (np.array_equal(gv, v[i]) and np.array_equal(gvo, vo[i])):
                wrong.append(i)

    try:
        threads = [threading.Thread(target=work, args=(*c, i)) for c in cases for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        for c in cases:
            c[0].close()
    assert not wrong
