"""FP64 / FP32 GEMM tiles: fewer K steps than LDS stages, every operand layout,
one bit pattern from every tile, and the built-in k-split."""
import numpy as np
import pytest

import tensornetworks_amd as tn

pytestmark = pytest.mark.gpu


def _product(ctx, tin, akm, bkm, M, N, K, tile, seed=5, ksplit=1):
    rng = np.random.default_rng(seed)
    A, B = rng.uniform(-1.0, 1.0, (M, K)), rng.uniform(-1.0, 1.0, (K, N))
    if tin == tn.TN_FP32:
        A, B = A.astype(np.float32).astype(np.float64), B.astype(np.float32).astype(np.float64)
    C = ctx.gemm_test(A if akm else np.ascontiguousarray(A.T), np.ascontiguousarray(B.T) if bkm else B, tin, 0, akm,
                      bkm, M, N, K, 1, tile, ksplit)[0]
    u = 2.0 ** -53 if tin == tn.TN_FP64 else 2.0 ** -24
    # K roundings of sums bounded by |A| |B|, and the final one
    bound = (K + 1) * u * (np.abs(A) @ np.abs(B))
    assert np.all(np.abs(C - A @ B) <= bound + 2.0 ** -53 * K * (np.abs(A) @ np.abs(B))), (tin, akm, bkm, tile, K)
    return C


@pytest.mark.parametrize("tin", [tn.TN_FP64, tn.TN_FP32])
@pytest.mark.parametrize("akm,bkm", [(True, True), (True, False), (False, False), (False, True)])
@pytest.mark.parametrize("K", [32, 64, 96, 160, 448])
def test_every_tile_gives_the_same_bits(ctx, tin, akm, bkm, K):
    M, N = 128, 256
    ref = _product(ctx, tin, akm, bkm, M, N, K, 7)
    deep = 32 if tin == tn.TN_FP64 else 64  # the K multiple the deep codes ask for
    for tile in range(0, 11):
        if tile >= 8 and K % deep:
            with pytest.raises(tn.TnError):
                _product(ctx, tin, akm, bkm, M, N, K, tile)
            continue
        assert np.array_equal(_product(ctx, tin, akm, bkm, M, N, K, tile), ref), tile


# numbers of tiles that are no multiple of the eight XCDs (117, 35, 961), and more
# than 768 of 128x64 and 64x128, whose FP32 form then changes
@pytest.mark.parametrize("tin", [tn.TN_FP64, tn.TN_FP32])
@pytest.mark.parametrize("M,N,tile", [(288, 416, 7), (320, 448, 4), (1984, 3968, 3), (3968, 1984, 2), (3968, 3968, 1)])
def test_any_number_of_tiles(ctx, tin, M, N, tile):
    C = _product(ctx, tin, True, True, M, N, 96, tile)
    assert np.array_equal(C, _product(ctx, tin, True, True, M, N, 96, 7 if tile != 7 else 0))


@pytest.mark.parametrize("tin", [tn.TN_FP64, tn.TN_FP32])
@pytest.mark.parametrize("akm,bkm", [(True, True), (True, False), (False, False), (False, True)])
@pytest.mark.parametrize("M,N,K", [(32, 32, 16), (64, 32, 48), (96, 160, 112), (128, 128, 16)])
def test_odd_multiples_of_sixteen(ctx, tin, akm, bkm, M, N, K):
    for tile in (0, 7):
        _product(ctx, tin, akm, bkm, M, N, K, tile)


@pytest.mark.parametrize("D1,D2,d", [(30, 30, 2), (320, 64, 2), (64, 320, 3), (288, 224, 2)])
@pytest.mark.parametrize("prec,u", [(tn.TN_FP64, 2.0 ** -53), (tn.TN_FP32, 2.0 ** -24)])
def test_heff_with_built_in_split(ctx, D1, D2, d, prec, u):
    # stage 3 sums over (w, a'): split over K for the wide left environments
    rng = np.random.default_rng(D1 + D2)
    W = np.ascontiguousarray(rng.uniform(-1.0, 1.0, (3, 3, d, d)))
    L, R = rng.uniform(-1.0, 1.0, (D1, 3, D1)), rng.uniform(-1.0, 1.0, (D2, 3, D2))
    x = rng.uniform(-1.0, 1.0, (D1, d, D2))

    def contract(W, L, R, x):
        T = np.einsum("anb,cwb->anwc", x, R, optimize=True)
        T = np.einsum("anwc,vwmn->vamc", T, W, optimize=True)
        return np.einsum("eva,vamc->emc", L, T, optimize=True)

    ctx.site_bind(W, np.ascontiguousarray(L.transpose(2, 0, 1)).ravel(),
                  np.ascontiguousarray(R.transpose(2, 0, 1)).ravel(), d, D1, D2, prec)
    y = ctx.heff_apply(np.ascontiguousarray(x.transpose(2, 0, 1)).ravel()).reshape(D2, D1, d).transpose(1, 2, 0)
    ref = contract(W, L, R, x)
    size = contract(np.abs(W), np.abs(L), np.abs(R), np.abs(x))
    # one rounding per term of the three nested sums
    assert np.all(np.abs(y - ref) <= (D2 + 3 * d + 3 * D1 + 8) * u * size)


@pytest.mark.parametrize("M,N,K", [(32, 64, 128), (192, 256, 256), (256, 192, 512), (320, 448, 1280), (1024, 384, 1024),
                                   (192, 128, 448), (96, 32, 32)])
def test_split_bf16_built_in_tile(ctx, M, N, K):
    # tile 0: the built-in tile of the split product, with and without a k-split
    rng = np.random.default_rng(M + N + K)
    A, B = rng.uniform(-1.0, 1.0, (M, K)), rng.uniform(-1.0, 1.0, (K, N))
    ref, size = A @ B, np.abs(A) @ np.abs(B)
    for ksplit in (1, 2, 4):
        if ksplit > 1 and K % (64 * ksplit):
            continue
        C = ctx.gemm_test(A, np.ascontiguousarray(B.T), tn.TN_BF16X3, 0 if ksplit > 1 else 1, True, True, M, N, K, 1,
                          0, ksplit)[0]
        # 24-bit operands, six products and one FP32 rounding per k
        assert np.all(np.abs(C - ref) <= (7 * K + 8) * 2.0 ** -24 * size)


@pytest.mark.parametrize("tile", [0, 1, 4, 7])
def test_rows_too_far_apart_for_32_bit_offsets(ctx, tile):
    # 128 rows of 34 MB: the last row of a 128-row tile starts 4.3e9 bytes after its
    # first.  Only the two ends of the rows are not zero, so the sums (in increasing
    # k) are those of the ends alone, bit for bit.
    M, K = 128, 4259840
    rng = np.random.default_rng(3)
    ends = rng.uniform(-1.0, 1.0, (M, 64))
    A = np.zeros((M, K))  # pages that are never written stay unallocated
    A[:, :32] = ends[:, :32]
    A[:, -32:] = ends[:, 32:]
    C = ctx.gemm_test(A, A, tn.TN_FP64, tn.TN_FP64, True, True, M, M, K, 1, tile)[0]
    ref = ctx.gemm_test(ends, ends, tn.TN_FP64, tn.TN_FP64, True, True, M, M, 64, 1, 7)[0]
    assert np.array_equal(C, ref)
