"""The Jacobi SVD round at the edges of its row chunks: fewer rows than a
workgroup's 32, ragged rows, more rows than a Gram chunk, rank deficiency."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(1, 1), (3, 2), (33, 5), (40, 33), (127, 31), (129, 64), (257, 96), (1030, 70), (70, 530)])
@pytest.mark.parametrize("rank", [None, 1])
def test_svd_row_chunks(ctx, m, n, rank):
    rng = np.random.default_rng(m * 7 + n)
    A = rng.standard_normal((m, n))
    if rank is not None:
        A = np.outer(rng.standard_normal(m), rng.standard_normal(n))
    U, s, Vt = ctx.svd(A)
    k = min(m, n)
    # orthogonality and backward error: a few roundings per rotation sweep, the
    # bound of the library's other SVD tests
    tol = 1e-13 * max(m, n) ** 0.5
    assert np.abs(U.T @ U - np.eye(k)).max() < tol and np.abs(Vt @ Vt.T - np.eye(k)).max() < tol
    assert np.linalg.norm((U * s) @ Vt - A) < 1e-13 * np.linalg.norm(A) * max(1, k) ** 0.5
    assert np.all(s[:-1] >= s[1:])
    assert np.abs(s - np.linalg.svd(A, compute_uv=False)).max() < 1e-13 * s[0] * k ** 0.5
