"""Which tiles a product is given, on both sides of the lines (csrc/gemm_mfma.hip); without a GPU the plans are made for 256 compute units."""
import pytest

PANEL = 1000000


@pytest.fixture(scope="module")
def mfma():
    from llmengine.ops import build, mfma
    if build.built_library() is None:
        pytest.skip("no built library")
    if mfma.compute_units() != 256:
        pytest.skip("the lines are drawn for 256 compute units")
    return mfma


# one round of narrow tiles through registers that fills the chip, and the sizes beside it
@pytest.mark.parametrize("M,N,K,panel", [(112, 12288, 2048, False), (128, 16384, 4096, False), (96, 12288, 2048, True), (112, 11264, 2048, True),
                                         (129, 12288, 2048, False), (256, 12288, 2048, False), (257, 12288, 2048, True), (192, 11264, 2048, True),
                                         (193, 11264, 2048, False), (256, 9216, 2048, True), (200, 14336, 2048, True), (100, 16400, 2048, False),
                                         (1800, 12288, 4096, False), (1500, 3072, 2048, True)])
def test_squares_keep_the_tiles_that_are_faster(mfma, M, N, K, panel):
    assert (mfma.gemm_bf16_chosen("squared", M, N, K) > PANEL) == panel


def test_stored_products_beside_them_are_as_they_were(mfma):
    assert mfma.gemm_bf16_chosen("stored", 249, 12288, 2048) > PANEL and mfma.gemm_bf16_chosen("stored", 112, 12288, 2048) > PANEL
    with pytest.raises(Exception):
        mfma.gemm_bf16_chosen("parts", 100, 64, 512, 0)


# two tiles of one area in as many rounds, or a round less in a tile that is no faster: the narrow one (or 256 x 256); and where the wide one wins
@pytest.mark.parametrize("kind,M,N,K,tile", [("added", 1779, 3072, 8192, PANEL + 192128), ("added", 1528, 3072, 8192, PANEL + 160128),
                                             ("stored", 3120, 6160, 2048, PANEL + 160128), ("stored", 2641, 6160, 3072, PANEL + 192128),
                                             ("gated", 540, 16384, 3072, PANEL + 144128), ("added", 3213, 3072, 3072, 256256),
                                             ("added", 2048, 3072, 8192, PANEL + 128192), ("rotating", 2048, 3072, 2048, PANEL + 128192),
                                             ("gated", 430, 16384, 2048, PANEL + 128256), ("stored", 1200, 6160, 2048, PANEL + 128256)])
def test_wide_panels_where_they_are_faster(mfma, kind, M, N, K, tile):
    assert mfma.gemm_bf16_chosen(kind, M, N, K, 1 if kind == "added" else 0, 64 if kind == "rotating" else 0) == tile
