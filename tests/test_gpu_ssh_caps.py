"""Small matrices are solved in one kernel. Padded with zeros beyond eight
entries per row on average, the same matrix takes the kernels per iteration,
whose sums the zeros do not change: x and every statistic have to agree bit for
bit, at the iteration cap too."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rows(n, seed, pad):
    """CSR, 1-based, the diagonal first; `pad` zeros on the diagonal at the end of each row."""
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    p = np.concatenate([np.stack([np.arange(n - 1), np.arange(1, n)], 1), rng.integers(0, n, (2 * n, 2))])
    p = np.unique(np.sort(p[p[:, 0] != p[:, 1]], 1), axis=0)
    off = sp.coo_matrix((-rng.uniform(0.1, 1.0, len(p)), (p[:, 0], p[:, 1])), shape=(n, n)).tocsr()
    a = (off + off.T).tocsr()
    a.sort_indices()
    diag = np.asarray(abs(a).sum(1)).ravel() + rng.uniform(0.05, 0.5, n)
    rowptr, colind, val = [1], [], []
    for r in range(n):
        s = slice(a.indptr[r], a.indptr[r + 1])
        colind += [r + 1, *(a.indices[s] + 1), *[r + 1] * pad]
        val += [diag[r], *a.data[s], *[0.0] * pad]
        rowptr.append(len(colind) + 1)
    return np.array(rowptr), np.array(colind), np.array(val)


@pytest.mark.parametrize("loop", ["classic", "single", "sparse"])
@pytest.mark.parametrize("n", [1, 64, 1000, 1025, 2048, 3072])
def test_one_kernel_solve_at_any_cap(monkeypatch, n, loop):
    from fesom2_amd import gpu
    if loop == "classic":
        monkeypatch.setenv("FGPU_SSH_CG", "classic")
    rng = np.random.default_rng(n)
    b, x0 = rng.normal(size=n), 0.1 * rng.normal(size=n)
    print(f"[gpu] {n} rows, {loop}", flush=True)
    runs = []
    for pad in (0, 9):
        rowptr, colind, val = _rows(n, n, pad)
        assert (len(val) > 8 * n) == (pad > 0)
        ctx = gpu.Context()
        try:
            ctx.ssh_set_matrix(rowptr, colind, val)
            ctx.ssh_solve_preconditioner(1 if loop == "sparse" else 2)
            runs.append([ctx.ssh_solve_cg(x0, b, tol, cap) for tol, cap in ((1e-10, 1), (1e-10, 3), (1e-13, 17), (1e-10, 2000))])
        finally:
            ctx.close()
    for (x, st), (y, su) in zip(*runs):
        np.testing.assert_array_equal(x, y)
        assert {k: st[k] for k in st if k != "ms"} == {k: su[k] for k in su if k != "ms"}
    if n > 1:
        assert [st["converged"] for _, st in runs[0]] == [False, False, False, True]
        assert [st["iters"] for _, st in runs[0][:3]] == [1, 3, 17]
