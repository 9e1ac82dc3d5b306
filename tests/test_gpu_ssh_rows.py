"""SSH solves on matrices of any row length (shorter and longer than the entries
that the iteration keeps in its own layout) and of sizes around a wave, a block
and more rows than threads; and small matrices, solved in one kernel, against
the kernels per iteration."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _matrix(n, longest, seed):
    """Symmetric, diagonally dominant; CSR with the diagonal first. Row 0 of a
    larger matrix is coupled to ``longest`` others."""
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    i = np.arange(n)
    pairs = [np.stack([i[:-1], i[1:]], 1)] if n > 1 else []
    if n > 8:
        pairs.append(rng.integers(0, n, (2 * n, 2)))
        pairs.append(np.stack([np.zeros(min(longest, n - 1), int), 1 + rng.permutation(n - 1)[:longest]], 1))
    a = sp.csr_matrix((n, n))
    if pairs:
        p = np.concatenate(pairs)
        p = np.unique(np.sort(p[p[:, 0] != p[:, 1]], 1), axis=0)
        off = sp.coo_matrix((-rng.uniform(0.1, 1.0, len(p)), (p[:, 0], p[:, 1])), shape=(n, n)).tocsr()
        a = (off + off.T).tocsr()
    a.sort_indices()
    diag = np.asarray(abs(a).sum(1)).ravel() + rng.uniform(0.05, 0.5, n)
    rowptr, colind, val = [1], [], []
    for r in range(n):
        s = slice(a.indptr[r], a.indptr[r + 1])
        colind += [r + 1, *(a.indices[s] + 1)]
        val += [diag[r], *a.data[s]]
        rowptr.append(len(colind) + 1)
    return np.array(rowptr), np.array(colind), np.array(val), a + sp.diags(diag)


@pytest.mark.parametrize("variant", [2, 1])
@pytest.mark.parametrize("n,longest", [(1, 0), (2, 0), (9, 7), (63, 8), (64, 40), (65, 9), (1000, 300), (4097, 8),
                                       (140000, 20)])
def test_solve_any_row_length(n, longest, variant):
    from fesom2_amd import gpu
    rowptr, colind, val, a = _matrix(n, longest, n + variant)
    b = np.random.default_rng(n).normal(size=n)
    print(f"[gpu] {n} rows, longest {np.diff(rowptr).max()}, preconditioner {variant}", flush=True)
    ctx = gpu.Context()
    try:
        ctx.ssh_set_matrix(rowptr, colind, val)
        ctx.ssh_solve_preconditioner(variant)
        runs = [ctx.ssh_solve_cg(np.zeros(n), b, 1e-10) for _ in range(2)]
    finally:
        ctx.close()
    x, st = runs[0]
    assert st["converged"]
    np.testing.assert_array_equal(x, runs[1][0])
    # the stopping rule on the residual, plus what its recurrence and the product here can drift by
    scale = np.sqrt(np.mean((abs(a) @ abs(x)) ** 2))
    bound = 1e-10 * np.sqrt(np.mean(b * b)) + (2 * st["iters"] + np.diff(rowptr).max()) * 2.3e-16 * scale
    assert np.sqrt(np.mean((b - a @ x) ** 2)) <= bound


@pytest.mark.parametrize("loop", ["classic", "single", "sparse"])
@pytest.mark.parametrize("n", [1, 64, 1000, 1024, 1025, 1793, 2048, 2049, 3072, 3073])
def test_one_kernel_solve_bitwise(monkeypatch, n, loop):
    """The same iterates whether the solve runs in one kernel or, from an
    iteration cap above 20,000 on, in one or more kernels per iteration."""
    from fesom2_amd import gpu
    if loop == "classic":
        monkeypatch.setenv("FGPU_SSH_CG", "classic")
    rowptr, colind, val, _ = _matrix(n, 30, n)
    rng = np.random.default_rng(n)
    b, x0 = rng.normal(size=n), 0.1 * rng.normal(size=n)
    print(f"[gpu] {n} rows, {loop}", flush=True)
    ctx = gpu.Context()
    try:
        ctx.ssh_set_matrix(rowptr, colind, val)
        ctx.ssh_solve_preconditioner(1 if loop == "sparse" else 2)
        for tol, cap in ((1e-10, 2000), (1e-10, 3), (1e-2, 2000)):
            x, st = ctx.ssh_solve_cg(x0, b, tol, cap)
            if cap < 2000 and not st["converged"]:
                continue
            y, su = ctx.ssh_solve_cg(x0, b, tol, 20001)
            np.testing.assert_array_equal(x, y)
            assert {k: st[k] for k in st if k != "ms"} == {k: su[k] for k in su if k != "ms"}
    finally:
        ctx.close()


@pytest.mark.parametrize("n,longest", [(2, 0), (63, 8), (64, 40), (65, 9), (1000, 300), (140000, 20)])
def test_learned_any_row_length(n, longest):
    """The network on full and partial tiles and rows of any length against its
    CPU reference, to that reference's bf16 tolerance, and the flexible CG with
    the untrained network, also on more rows than threads."""
    from fesom2_amd import gpu
    from oracle import mpnn_ref as nn
    rowptr, colind, val, a = _matrix(n, longest, n)
    rng = np.random.default_rng(n)
    b = rng.normal(size=n)
    print(f"[gpu] learned, {n} rows, longest {np.diff(rowptr).max()}", flush=True)
    ctx = gpu.Context()
    try:
        ctx.ssh_set_matrix(rowptr, colind, val)
        ctx.ssh_solve_preconditioner(2)
        ctx.nn_init(0)
        x, st = ctx.ssh_solve_learned(np.zeros(n), b, 1e-10)
        if n <= 1000:
            p = nn.init_params(4)
            p["w_out"] = rng.normal(0, 0.2, nn.C).astype(np.float32)
            ctx.nn_set_weights(nn.flatten(p))
            ctx.N2 = n   # as mesh_init sets it: the wrapper's output size
            z = ctx.nn_apply(b)
            ref, _ = nn.forward(nn.Graph(rowptr - 1, colind - 1, val), p, b)
            assert np.linalg.norm(z - ref) < 2e-2 * np.linalg.norm(ref)
    finally:
        ctx.close()
    assert st["converged"]
    scale = np.sqrt(np.mean((abs(a) @ abs(x)) ** 2))
    bound = 1e-10 * np.sqrt(np.mean(b * b)) + (2 * st["iters"] + np.diff(rowptr).max()) * 2.3e-16 * scale
    assert np.sqrt(np.mean((b - a @ x) ** 2)) <= bound
