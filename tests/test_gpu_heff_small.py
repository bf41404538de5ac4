"""The one-launch Heff apply of small FP64 sites and the one-launch Lanczos
step of short vectors, at the edges of what they cover."""
import numpy as np
import pytest

import tensornetworks_amd as tn
from devmem import DeviceArray

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


def _flat(F):  # (bra, w, ket) -> F[w + Dw*(i + D*j)]
    return np.ascontiguousarray(F.transpose(2, 0, 1)).ravel()


def _heff(W, L, R, x):
    T = np.einsum("anb,cwb->anwc", x, R, optimize=True)
    T = np.einsum("anwc,vwmn->vamc", T, W, optimize=True)
    return np.einsum("eva,vamc->emc", L, T, optimize=True)


# padded bonds 32 and 64 in every combination (a left bond of 32 takes the one
# launch), the next larger ones (three kernels), one to eight channels, d from 2
# to 5, a table too large for the launch
@pytest.mark.parametrize("d,D1,D2,Dw", [(2, 1, 2, 5), (2, 8, 8, 5), (3, 32, 33, 5), (3, 64, 64, 5), (4, 33, 32, 3),
                                        (4, 64, 64, 6), (2, 64, 65, 5), (2, 65, 64, 5), (5, 20, 20, 4), (2, 40, 31, 1),
                                        (2, 17, 64, 2), (3, 64, 20, 6), (4, 30, 30, 8)])
@pytest.mark.parametrize("left,right", [(None, None), (0, 1), (1, 0), (0, None), (None, 1)])
def test_apply_matches_numpy(ctx, d, D1, D2, Dw, left, right):
    if Dw == 1 and (left is not None or right is not None):
        pytest.skip("an identity channel needs a second one")
    rng = np.random.default_rng(D1 * 100 + D2 + Dw)
    W = rng.uniform(-1.0, 1.0, (Dw, Dw, d, d))
    W[np.abs(W) < 0.4] = 0.0
    L, R = rng.uniform(-1.0, 1.0, (D1, Dw, D1)), rng.uniform(-1.0, 1.0, (D2, Dw, D2))
    if left is not None:  # first or last channel the identity
        L[:, -left, :] = np.eye(D1)
    if right is not None:
        R[:, -right, :] = np.eye(D2)
    x = rng.uniform(-1.0, 1.0, (D1, d, D2))
    ctx.site_bind(np.ascontiguousarray(W), _flat(L), _flat(R), d, D1, D2, tn.TN_FP64)
    xf = np.ascontiguousarray(x.transpose(2, 0, 1)).ravel()
    ref = _heff(W, L, R, x)
    # one rounding per term of the three nested sums
    bound = (D1 * Dw + D2 + Dw * d + 8) * U * _heff(np.abs(W), np.abs(L), np.abs(R), np.abs(x))

    def close(y):
        assert np.all(np.abs(y.reshape(D2, D1, d).transpose(1, 2, 0) - ref) <= bound)

    close(ctx.heff_apply(xf))
    xd, yd = DeviceArray(xf.size), DeviceArray(xf.size)
    for call in (ctx.heff_apply_device, ctx.heff_apply_device_noalloc):
        xd.upload(xf)
        yd.upload(np.full(xf.size, np.nan))
        call(xd.address, yd.address, xf.size)
        close(yd.download())
        assert np.array_equal(xd.download(), xf)
        call(xd.address, xd.address, xf.size)  # in place
        close(xd.download())


# padded bonds of 32 (vectors of 2048 entries, one launch) and of 64 and 96 (four);
# partial re-orthogonalisation scales in the next step, full in the same one
@pytest.mark.parametrize("D", [20, 40, 64, 65])
@pytest.mark.parametrize("reorth", [0, 1])
def test_sweep_energy_matches_dense(ctx, D, reorth):
    from tensornetworks_amd.models import mpo_contract, xxz_mpo
    Ws = xxz_mpo(8, 0.5, Jz=0.7, hz=0.3)
    e = np.linalg.eigvalsh(mpo_contract(Ws))[0]
    ch = tn.Chain(ctx, Ws, D)
    ch.initialize(1, 11)
    ch.normalize(1)
    o = tn.SweepOpts.default(eig_tol=1e-12, reorth=reorth, max_krylov=40)
    ch.load_caches(o)
    for _ in range(3):
        st = ch.sweep(0, o)
        st = ch.sweep(1, o)
    ch.close()
    # D >= 16 represents the ground state of 8 sites exactly; the Lanczos
    # residual is 1e-12
    assert abs(st.energy - e) < 1e-11
