"""The Lanczos step kernels at the sizes where their chunks, vector groups and
partial sums change: capped solves against the same restarted Lanczos in NumPy."""
import numpy as np
import pytest

import tensornetworks_amd as tn

pytestmark = pytest.mark.gpu


def _symmetric(rng, Dw, D):
    F = rng.uniform(-1.0, 1.0, (Dw, D, D))
    return 0.5 * (F + F.transpose(0, 2, 1))


def _restarted_lanczos(apply, x, steps, cycles):
    for _ in range(cycles):
        V = [x / np.linalg.norm(x)]
        T = np.zeros((steps, steps))
        for j in range(steps):
            w = apply(V[j])
            for _ in range(2):
                c = np.array([v @ w for v in V])
                w = w - np.array(V).T @ c
                T[j, j] += c[j]
            b = np.linalg.norm(w)
            if j + 1 < steps:
                T[j, j + 1] = T[j + 1, j] = b
                V.append(w / b)
        e, Z = np.linalg.eigh(T)
        x = np.array(V).T @ Z[:, 0]
    return e[0]


# padded lengths 2048, 8192 (last with 512-entry chunks), 9216, 131072 (last with
# 4096-entry chunks and split vector groups), 147456 (long vectors); steps past the
# line between one launch and four (2048 with 16 vectors, 6144 with 5)
@pytest.mark.parametrize("d,D1,D2,steps", [(2, 32, 32, 9), (2, 32, 32, 24), (3, 64, 32, 9), (2, 64, 64, 8), (2, 64, 64, 33), (3, 90, 31, 17),
                                           (2, 256, 256, 26), (2, 288, 256, 5), (2, 288, 256, 4)])
def test_capped_solve_matches_numpy(ctx, d, D1, D2, steps):
    rng = np.random.default_rng(100 * D1 + D2 + steps)
    W = rng.uniform(-1.0, 1.0, (2, 2, d, d))
    W = 0.5 * (W + W.transpose(0, 1, 3, 2))
    L, R = _symmetric(rng, 2, D1), _symmetric(rng, 2, D2)
    x0 = rng.standard_normal((D2, D1, d))  # psi[m + d*(i1 + D1*i2)]

    def apply(v):
        x = v.reshape(D2, D1, d).transpose(1, 2, 0)
        T = [(x.reshape(D1 * d, D2) @ R[w].T).reshape(D1, d, D2) for w in range(2)]
        y = 0.0
        for w in range(2):
            m = sum(np.einsum("mn,anb->amb", W[w, v2], T[v2]) for v2 in range(2))
            y = y + (L[w] @ m.reshape(D1, d * D2)).reshape(D1, d, D2)
        return y.transpose(2, 0, 1).ravel()

    ctx.site_bind(np.ascontiguousarray(W), np.ascontiguousarray(L.transpose(2, 1, 0)).ravel(),
                  np.ascontiguousarray(R.transpose(2, 1, 0)).ravel(), d, D1, D2, tn.TN_FP64)
    ev, x, nmv, _ = ctx.eig_lowest(x0.ravel(), tol=0.0, maxit=steps, nev=1)
    assert 4 * steps < nmv <= 5 * steps  # one solve and four restarts (the last may meet an invariant space)
    ref = _restarted_lanczos(apply, x0.ravel(), steps, 5)
    # the same Krylov spaces: the Ritz values differ by the rounding of 5*steps
    # products and passes, 2^-53 |H| each (|H| about |e0|)
    tol = 5 * steps * 2.0 ** -53 * abs(ref) * 32
    assert abs(ev[0] - ref) <= tol, (ev[0], ref)
    assert abs(np.linalg.norm(x) - 1.0) <= 1e-13
    assert abs(x @ apply(x) - ev[0]) <= tol


# one site in one launch, three kernels per apply; one- and two-site sweeps; refined
@pytest.mark.parametrize("L,d,D,kw", [(4, 2, 4, {}), (6, 3, 40, {}), (4, 2, 4, {"reorth": 1}),
                                      (6, 2, 8, {"precision": tn.TN_FP32, "refine": 1, "refine_precision": tn.TN_FP64,
                                                 "refine_tol": 1e-12})])
@pytest.mark.parametrize("two", [False, True])
def test_timed_applies_are_the_counted_ones(ctx, L, d, D, kw, two):
    # an apply that was queued ahead of the convergence test and not used goes
    # neither into the counts nor into the times
    opts = tn.SweepOpts.default(eig_tol=1e-11, **kw)
    ch = tn.Chain(ctx, tn.xxz_mpo(L, 0.5 * (d - 1)), D)
    ch.initialize(1, 5)
    ch.normalize_qr(1)
    ch.load_caches(opts)
    st = tn.SweepStats()
    before = ctx.heff_timings()
    for direction in (0, 1):
        if two:
            ch.sweep2(direction, D, 0.0, opts, st)
        else:
            ch.sweep(direction, opts, st)
    assert st.n_matvec > 0 and st.heff_ms > 0
    assert ctx.heff_timings() - before == st.n_matvec
