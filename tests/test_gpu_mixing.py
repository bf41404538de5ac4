"""The MPO stage and the layout changes at the edges of their dispatch: tables
that fit the LDS copy and tables that do not, few and many workgroups, ragged
bonds, against a NumPy contraction."""
import numpy as np
import pytest

import tensornetworks_amd as tn
from devmem import DeviceArray

pytestmark = pytest.mark.gpu


def _flat(F):  # (bra, w, ket) -> F[w + Dw*(i + D*j)]
    return np.ascontiguousarray(F.transpose(2, 0, 1)).ravel()


def _heff(W, L, R, x):
    T = np.einsum("anb,cwb->anwc", x, R, optimize=True)
    T = np.einsum("anwc,vwmn->vamc", T, W, optimize=True)
    return np.einsum("eva,vamc->emc", L, T, optimize=True)


def _left(W, L, A):
    T = np.einsum("eva,anb->evnb", L, A, optimize=True)
    T = np.einsum("evnb,vwmn->emwb", T, W, optimize=True)
    return np.einsum("emc,emwb->cwb", A, T, optimize=True)


def _right(W, R, A):
    T = np.einsum("anb,cwb->anwc", A, R, optimize=True)
    T = np.einsum("anwc,vwmn->avmc", T, W, optimize=True)
    return np.einsum("emc,avmc->eva", A, T, optimize=True)


# Dw = 5, d = 3: 15 outputs, 225 entries (in LDS); Dw = 8, d = 3: 576 entries and
# Dw = 23, d = 3: 69 outputs (global memory)
@pytest.mark.parametrize("Dw,d,D1,D2", [(5, 3, 31, 33), (8, 3, 40, 20), (23, 3, 9, 12), (1, 2, 65, 64), (2, 2, 200, 260)])
@pytest.mark.parametrize("prec,u", [(tn.TN_FP64, 2.0 ** -53), (tn.TN_FP32, 2.0 ** -24)])
def test_dense_tables(ctx, Dw, d, D1, D2, prec, u):
    rng = np.random.default_rng(Dw * 1000 + D1)
    W = np.ascontiguousarray(rng.uniform(-1.0, 1.0, (Dw, Dw, d, d)))
    L, R = rng.uniform(-1.0, 1.0, (D1, Dw, D1)), rng.uniform(-1.0, 1.0, (D2, Dw, D2))
    x = rng.uniform(-1.0, 1.0, (D1, d, D2))
    ctx.site_bind(W, _flat(L), _flat(R), d, D1, D2, prec)
    xf = np.ascontiguousarray(x.transpose(2, 0, 1)).ravel()
    # one rounding per term of the three nested sums (operands rounded once each)
    n = D1 * Dw + D2 + Dw * d + 8
    size = _heff(np.abs(W), np.abs(L), np.abs(R), np.abs(x))
    y = ctx.heff_apply(xf).reshape(D2, D1, d).transpose(1, 2, 0)
    assert np.all(np.abs(y - _heff(W, L, R, x)) <= n * u * size)
    # the device-pointer call changes the layout on the device
    xd, yd = DeviceArray(xf.size), DeviceArray(xf.size)
    xd.upload(xf)
    ctx.heff_apply_device(xd.address, yd.address, xf.size)
    assert np.array_equal(yd.download().reshape(D2, D1, d).transpose(1, 2, 0), y)
    for direction, D, ref, size in ((0, D2, _left(W, L, x), _left(np.abs(W), np.abs(L), np.abs(x))),
                                    (1, D1, _right(W, R, x), _right(np.abs(W), np.abs(R), np.abs(x)))):
        F = ctx.env_update(direction, xf, D * D * Dw).reshape(D, D, Dw).transpose(1, 2, 0)
        n = (D1 + D2) * d + Dw * d + D1 + D2 + 8
        assert np.all(np.abs(F - ref) <= n * u * size)
