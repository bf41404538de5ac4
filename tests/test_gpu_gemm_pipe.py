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


def _pad(D):
    return (D + 31) // 32 * 32


def _heff(W, L, R, x):
    T = np.einsum("anb,cwb->anwc", x, R, optimize=True)
    T = np.einsum("anwc,vwmn->vamc", T, W, optimize=True)
    return np.einsum("eva,vamc->emc", L, T, optimize=True)


def _flat(F):  # (bra, w, ket) -> F[w + Dw*(i + D*j)]
    return np.ascontiguousarray(F.transpose(2, 0, 1)).ravel()


# (d, Dw, D1, D2) and the k-split of stage 3 (sum over (w, a')) in FP64, FP32 and
# split bf16: none, by two and by four
@pytest.mark.parametrize("d,Dw,D1,D2,splits", [(2, 3, 30, 30, (1, 1, 1)), (2, 3, 320, 64, (1, 1, 1)),
                                               (3, 3, 64, 320, (1, 1, 1)), (2, 3, 288, 224, (1, 1, 1)),
                                               (3, 4, 160, 96, (2, 2, 1)), (2, 4, 128, 64, (4, 4, 4)),
                                               (2, 4, 320, 224, (4, 4, 4)), (2, 4, 250, 20, (4, 4, 4))])
@pytest.mark.parametrize("k,prec", enumerate([tn.TN_FP64, tn.TN_FP32, tn.TN_BF16X3]))
def test_heff_with_built_in_split(ctx, d, Dw, D1, D2, splits, k, prec):
    D1p, D2p = _pad(D1), _pad(D2)
    assert tn.gemm_plan(prec, True, True, D1p, d * D2p, Dw * D1p, split=True)[1] == splits[k]
    rng = np.random.default_rng(D1 + D2)
    W = np.ascontiguousarray(rng.uniform(-1.0, 1.0, (Dw, Dw, d, d)))
    L, R = rng.uniform(-1.0, 1.0, (D1, Dw, D1)), rng.uniform(-1.0, 1.0, (D2, Dw, D2))
    x = rng.uniform(-1.0, 1.0, (D1, d, D2))
    ctx.site_bind(W, _flat(L), _flat(R), d, D1, D2, prec)
    y = ctx.heff_apply(np.ascontiguousarray(x.transpose(2, 0, 1)).ravel()).reshape(D2, D1, d).transpose(1, 2, 0)
    ref = _heff(W, L, R, x)
    size = _heff(np.abs(W), np.abs(L), np.abs(R), np.abs(x))
    # one rounding per term of the three nested sums; split bf16: six products and
    # one rounding per term
    u = 2.0 ** -53 if prec == tn.TN_FP64 else 2.0 ** -24
    terms = 7 if prec == tn.TN_BF16X3 else 1
    assert np.all(np.abs(y - ref) <= (terms * (D2 + Dw * D1) + Dw * d + 8 * terms) * u * size)


# FP64 environments: left with its last sum (a, m) split, right with its first (b')
@pytest.mark.parametrize("direction,d,Dw,D1,D2,split", [(0, 2, 4, 250, 20, 4), (0, 2, 4, 320, 20, 2), (1, 2, 4, 20, 640, 2),
                                                        (1, 2, 3, 20, 512, 4)])
def test_environment_with_built_in_split(ctx, direction, d, Dw, D1, D2, split):
    D1p, D2p = _pad(D1), _pad(D2)
    shape = (D2p, Dw * D2p, D1p * d) if direction == 0 else (D1p * d, Dw * D2p, D2p)
    assert tn.gemm_plan(tn.TN_FP64, direction == 1, direction == 1, *shape, split=True)[1] == split
    rng = np.random.default_rng(D1 + 3 * D2)
    W = np.ascontiguousarray(rng.uniform(-1.0, 1.0, (Dw, Dw, d, d)))
    L, R = rng.uniform(-1.0, 1.0, (D1, Dw, D1)), rng.uniform(-1.0, 1.0, (D2, Dw, D2))
    A = rng.uniform(-1.0, 1.0, (D1, d, D2))

    def update(W, L, R, A):
        if direction == 0:
            T = np.einsum("eva,anb->evnb", L, A, optimize=True)
            T = np.einsum("evnb,vwmn->emwb", T, W, optimize=True)
            return np.einsum("emc,emwb->cwb", A, T, optimize=True)
        T = np.einsum("anb,cwb->anwc", A, R, optimize=True)
        T = np.einsum("anwc,vwmn->avmc", T, W, optimize=True)
        return np.einsum("emc,avmc->eva", A, T, optimize=True)

    ctx.site_bind(W, _flat(L), _flat(R), d, D1, D2, tn.TN_FP64)
    D = D2 if direction == 0 else D1
    F = ctx.env_update(direction, np.ascontiguousarray(A.transpose(2, 0, 1)).ravel(), D * D * Dw)
    F = F.reshape(D, D, Dw).transpose(1, 2, 0)
    size = update(np.abs(W), np.abs(L), np.abs(R), np.abs(A))
    n = (D1 if direction == 0 else D2) * (1 + d) + Dw * d + 8  # terms of the three nested sums
    assert np.all(np.abs(F - update(W, L, R, A)) <= n * 2.0 ** -53 * size)


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
