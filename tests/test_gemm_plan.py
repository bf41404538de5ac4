"""Built-in choice of the GEMM tile, k-split and copy offsets (host logic)."""
import pytest

import tensornetworks_amd as tn

TILE = {1: (128, 128), 2: (128, 64), 3: (64, 128), 4: (64, 64), 5: (32, 64), 6: (64, 32), 7: (32, 32)}


@pytest.mark.parametrize("tin,es", [(tn.TN_FP64, 8), (tn.TN_FP32, 4)])
@pytest.mark.parametrize("akm,bkm", [(True, True), (True, False), (False, False), (False, True)])
@pytest.mark.parametrize("M,N,K", [(32, 32, 64), (128, 128, 64), (3072, 4096, 64), (1024, 64, 96)])
def test_copy_offsets_fit_their_register(tin, es, akm, bkm, M, N, K):
    # the largest byte offset of a copy within a tile stays below 2^32 unless the
    # plan says that the offsets are 64-bit ones
    def largest(kmajor, rows, ld):
        k = 128 // es
        return ((rows - 1) * ld + k - 1) * es if kmajor else ((k - 1) * ld + rows - 1) * es

    seen = set()
    for e in range(12, 34):
        for ld in (2 ** e - 32, 2 ** e, 2 ** e + 32, 3 * 2 ** (e - 1)):
            for lda, ldb in ((ld, 4096), (4096, ld), (ld, ld)):
                tile, ks, wide = tn.gemm_plan(tin, akm, bkm, M, N, K, lda, ldb)
                bm, bn = TILE[tile]
                far = max(largest(akm, bm, lda), largest(bkm, bn, ldb))
                assert wide or far < 2 ** 32, (lda, ldb, tile)
                assert not wide or far >= 2 ** 31, (lda, ldb, tile)  # and not long before
                assert ks == 1
                seen.add(wide)
    assert seen == {0, 1}


def test_plan_refuses_bad_shapes():
    for bad in ((33, 32, 32), (32, 40, 32), (32, 32, 8), (0, 32, 32)):
        with pytest.raises(tn.TnError):
            tn.gemm_plan(tn.TN_FP64, True, True, *bad)
