"""CholeskyQR where the diagonal factorisation's 16-column panels begin and end: one
column, panels and blocks with remainders, a pivot that fails in the last panel."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 96, 97, 129])
def test_matches_numpy(ctx, n):
    m = n + 40
    A = np.random.default_rng(n).standard_normal((m, n))
    Q, R, ok, shifted = ctx.cholqr_test(A)
    assert ok and not shifted
    q, r = np.linalg.qr(A)
    s = np.sign(np.diag(r))
    # well conditioned (cond < 1e2): the factors differ by cond times the rounding
    # of the Gram matrix, the second pass leaves Q orthonormal to rounding
    assert np.abs(Q.T @ Q - np.eye(n)).max() < 1e-13
    assert np.abs(np.tril(R, -1)).max() == 0.0
    assert np.abs(Q @ R - A).max() < 1e-13 * np.abs(A).max() * np.sqrt(m)
    assert np.abs(R - s[:, None] * r).max() < 1e-11 * np.abs(r).max()
    assert np.abs(Q - q * s).max() < 1e-10


@pytest.mark.parametrize("n", [17, 64, 80])
def test_failing_pivot_takes_the_shift(ctx, n):
    A = np.random.default_rng(n).standard_normal((n + 30, n))
    A[:, -1] = A[:, 0]  # the last pivot is zero up to rounding
    Q, R, ok, _ = ctx.cholqr_test(A)
    assert ok
    assert np.abs(Q.T @ Q - np.eye(n)).max() < 1e-11
    assert np.abs(Q @ R - A).max() < 1e-12 * np.abs(A).max() * np.sqrt(n + 30)
