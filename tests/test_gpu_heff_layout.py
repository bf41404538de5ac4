"""Device-pointer apply at reduced precision: the layout pass that also forms the
low-precision operand against the host apply, which converts in passes of its own."""
import numpy as np
import pytest

import tensornetworks_amd as tn
from devmem import DeviceArray

pytestmark = pytest.mark.gpu


# one entry, tiles of 32 with remainders on either side, whole tiles, a longer second
# side; two calls on different inputs, the second shows what the first left behind
@pytest.mark.parametrize("d,D1,D2", [(2, 1, 1), (2, 33, 31), (3, 32, 64), (3, 21, 130), (5, 65, 40)])
@pytest.mark.parametrize("precision", [tn.TN_FP32, tn.TN_BF16, tn.TN_BF16X3])
def test_same_bits_as_host_apply(ctx, d, D1, D2, precision):
    rng = np.random.default_rng(d * 1000 + D1 * 10 + D2)
    Dw = 3
    W = rng.uniform(-1.0, 1.0, (Dw, Dw, d, d))
    L, R = rng.uniform(-1.0, 1.0, Dw * D1 * D1), rng.uniform(-1.0, 1.0, Dw * D2 * D2)
    ctx.site_bind(np.ascontiguousarray(W), L, R, d, D1, D2, precision)
    xd, yd = DeviceArray(d * D1 * D2), DeviceArray(d * D1 * D2)
    for scale in (1e3, 1.0):
        x = scale * rng.uniform(-1.0, 1.0, d * D1 * D2)
        ref = ctx.heff_apply(x)
        assert np.all(np.isfinite(ref))
        # the allocation-free apply takes no k-split and no fused first stage: its
        # sums have another order, so it is held to FP32 (BF16: operand) rounding
        u = 2.0 ** -8 if precision == tn.TN_BF16 else 2.0 ** -22
        tol = 4 * u * np.sqrt(D1 * D2 * d * Dw) * scale * max(D1, D2) * Dw
        for call, same in ((ctx.heff_apply_device, True), (ctx.heff_apply_device_noalloc, False)):
            xd.upload(x)
            call(xd.address, yd.address, x.size)
            y = yd.download()
            assert np.array_equal(y, ref) if same else np.abs(y - ref).max() <= tol
            call(xd.address, xd.address, x.size)  # in place
            assert np.array_equal(xd.download(), y)
