"""Jacobi SVD: the one-launch iteration of up to 32 columns at the edges of its
rows, and the rotations from reciprocal square roots (128 columns and more) on
spectra whose Gram entries span most of the exponent range."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


def _check(ctx, A):
    m, n = A.shape
    k = min(m, n)
    Q, s, Vt = ctx.svd(A)
    ref = np.linalg.svd(A, compute_uv=False)
    # each column meets a few hundred rotations (ten sweeps), every one with a
    # few roundings, whose errors add like a random walk; the rest is the products
    tol = 64 * U * max(m, n) ** 0.5 * 8
    assert np.abs(s - ref).max() <= tol * ref[0]
    assert np.linalg.norm((Q * s) @ Vt - A) <= tol * np.linalg.norm(ref)
    assert np.abs(Q.T @ Q - np.eye(k)).max() <= 2 * tol
    assert np.abs(Vt @ Vt.T - np.eye(k)).max() <= 2 * tol


# one pair of column blocks: 1 to 32 columns, rows to both sides of 256, either
# orientation, orthogonal columns (no rotation), one and two sweeps' parity
@pytest.mark.parametrize("m,n", [(1, 1), (2, 1), (32, 32), (33, 31), (16, 200), (256, 32), (257, 32), (20, 256), (300, 7)])
@pytest.mark.parametrize("kind", ["random", "orthogonal", "graded"])
def test_one_pair(ctx, m, n, kind):
    rng = np.random.default_rng(100 * m + n)
    A = rng.standard_normal((m, n))
    k = min(m, n)
    if kind == "orthogonal":
        A = np.linalg.qr(A if m >= n else A.T)[0]
        A = A if m >= n else A.T
    elif kind == "graded":
        if m >= n:
            A *= 10.0 ** -np.linspace(0, 12, n)
        else:
            A *= (10.0 ** -np.linspace(0, 12, m))[:, None]
    _check(ctx, A)


def test_zero_matrix(ctx):
    Q, s, Vt = ctx.svd(np.zeros((12, 9)))
    assert np.all(s == 0.0)
    assert np.abs(Q.T @ Q - np.eye(9)).max() <= 64 * U and np.abs(Vt @ Vt.T - np.eye(9)).max() <= 64 * U


@pytest.mark.parametrize("m,n", [(3, 2), (20, 20), (160, 150)])
def test_infinity_refused(ctx, m, n):
    A = np.ones((m, n))
    A[m // 2, n // 2] = np.inf
    with pytest.raises(Exception, match="non-finite"):
        ctx.svd(A)


# q >= 128: equal norms (45 degree rotations), steep decay, scales near both ends
@pytest.mark.parametrize("m,n", [(128, 128), (161, 129), (130, 300), (512, 200)])
@pytest.mark.parametrize("kind", ["random", "decay", "duplicates", "tiny", "huge"])
def test_many_columns(ctx, m, n, kind):
    rng = np.random.default_rng(m + n)
    A = rng.standard_normal((m, n))
    k = min(m, n)
    if kind == "decay":
        a, _, b = np.linalg.svd(A, full_matrices=False)
        A = (a * 10.0 ** -np.linspace(0, 60, k)) @ b
    elif kind == "duplicates":
        A[:, n // 2:] = A[:, :n - n // 2]
    elif kind == "tiny":
        A *= 1e-290
    elif kind == "huge":
        A *= 1e290
    _check(ctx, A)


# the completion of a zero column: in a square matrix no unit vector need have a
# large part outside the other columns' span
@pytest.mark.parametrize("m,n", [(2, 2), (32, 32), (40, 40), (100, 100), (50, 32), (20, 60)])
def test_zero_column(ctx, m, n):
    rng = np.random.default_rng(m + 3 * n)
    A = rng.standard_normal((m, n))
    if m >= n:
        A[:, n // 2] = 0.0
    else:
        A[m // 2] = 0.0
    _check(ctx, A)
