"""Every tile shape of the long-M GEMM has a GPU case with each epilogue it takes
(dtree_gemm_long_tile is host code: without a GPU it answers for 256 CUs)."""
import test_gpu_gemm_long as t
from dtree_hip import _native as N

EPILOGUES = (N.EPI_STORE_F32, N.EPI_RESIDUAL, N.EPI_SWIGLU, N.EPI_STORE_BF16)
F16 = {(64, 64), (64, 128), (128, 128), (256, 128), (256, 192), (256, 256), (256, 320), (256, 384)}
Q4 = {(128, 128), (128, 256), (256, 192), (256, 256)}
WORK = [(rows, n) for rows in range(128, 4097, 128) for n in (64, 256, 1024, 2560, 4096, 6144, 9728, 12352, 19456, 24576)]


def test_the_lists_name_the_chosen_tiles():
    for rows, n, tile, tile_res in t.SHAPES:
        for epi in EPILOGUES:
            assert t._tile(rows, n, 64, epi, N.W_TILED_F16) == (tile_res if epi == N.EPI_RESIDUAL else tile), (rows, n)
    for rows, n, tile in t.TAILS:
        assert t._tile(rows, n, 192, N.EPI_STORE_F32, N.W_TILED_F16) == tile, (rows, n)
    for rows, n, k, tile in t.Q4_SHAPES + t.Q4_TAILS:
        assert t._tile(rows, n, k, N.EPI_STORE_F32, N.W_Q4G64) == tile, (rows, n, k)


def test_every_tile_has_a_case():
    # the tiles that any work can choose are the ones listed above ...
    for epi in EPILOGUES:
        chosen = {t._tile(r, n, 256, epi, N.W_TILED_F16) for r, n in WORK}
        assert chosen == (F16 if epi != N.EPI_RESIDUAL else {x for x in F16 if x[1] <= 256})
        assert {t._tile(r, n, 256, epi, N.W_Q4G64) for r, n in WORK} == Q4
    assert {t._tile(r, n, 192, N.EPI_STORE_F32, N.W_Q4G64) for r, n in WORK} == Q4 - {(128, 128)}
    # ... and each has a case, a last tile of fewer rows (from 256 rows on; the
    # smaller ones divide the padding) and of fewer columns
    assert {s[2] for s in t.SHAPES} == F16 and {s[3] for s in t.SHAPES} == {x for x in F16 if x[1] <= 256}
    assert {x for r, n, x, _ in t.SHAPES if r % x[0]} == {x for x in F16 if x[0] == 256}
    assert {x for r, n, x in t.TAILS if n % x[1] or x[1] == 64} == F16
    assert {s[3] for s in t.Q4_SHAPES} == Q4 and {s[3] for s in t.Q4_TAILS} == Q4 - {(128, 128)}
    assert {x for r, n, _, x in t.Q4_SHAPES if r % x[0]} == {x for x in Q4 if x[0] == 256}
