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
