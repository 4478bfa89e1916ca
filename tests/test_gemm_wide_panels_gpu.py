"""Tiles of 192 and 256 columns (csrc/gemm_panel.hip), from 160 rows on in slabs of 32 k."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
PANEL = 1000000
TILES = [(96, 192), (128, 192), (160, 192), (192, 192), (128, 256), (192, 256)]


@pytest.fixture(scope="module")
def ops():
    from llmengine import ops
    return ops


def _pair(M, N, K, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(M, K, generator=g).to(torch.bfloat16), (torch.randn(N, K, generator=g) * 0.05).to(torch.bfloat16)


# one row, a tile's edges in rows and columns, k of one to seven slabs of 32 (fewer than the ring holds) and of many; what lies behind
# the last row and column joins no sum
@pytest.mark.parametrize("M,N,K", [(1, 16, 32), (97, 208, 64), (161, 320, 160), (193, 448, 224), (385, 528, 2080)])
@pytest.mark.parametrize("rows,cols", TILES)
def test_wide_panels(ops, M, N, K, rows, cols):
    """Stored and added sums against 64 bits (32-bit sums of bfloat16 products: 2e-5), and the bits of the tile through registers, which
    adds k in the same order; gated ones in whole pairs of columns only."""
    a, w = _pair(M + 9, N + 16, K, 21)
    ref = a[:M].double() @ w[:N].double().T
    a[M:], w[N:] = float("nan"), float("inf")
    ad, wb, tile = a.to(DEV)[:M], ops.block_weight(w.to(DEV))[:N // 16], PANEL + 1000 * rows + cols
    base = torch.randn(M, N, generator=torch.Generator().manual_seed(22))
    for accumulate in (False, True):
        got, other = base.clone().to(DEV), base.clone().to(DEV)
        ops.gemm_bf16(ad, wb, got, accumulate, tile=tile)
        ops.gemm_bf16(ad, wb, other, accumulate, tile=128, ksplit=1)
        want = ref + base.double() if accumulate else ref
        assert float((got.cpu().double() - want).norm() / want.norm()) < 2e-5 and torch.equal(got, other)
    if N % 32:
        return
    got, other = (torch.zeros(M, N // 2, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    ops.gemm_bf16(ad, wb, other, gated=True, tile=128)
    if cols == 256:
        ops.gemm_bf16(ad, wb, got, gated=True, tile=tile)
        assert torch.equal(got, other)
    else:
        with pytest.raises(ops.KernelError):
            ops.gemm_bf16(ad, wb, got, gated=True, tile=tile)


@pytest.mark.parametrize("T,n_q,n_kv,hd,tiles", [(2050, 8, 2, 64, TILES[:5]), (200, 10, 1, 64, TILES[:5]), (300, 3, 1, 128, TILES[4:5])])
def test_wide_panels_rotate_as_the_others(ops, T, n_q, n_kv, hd, tiles):
    g, page, K = torch.Generator().manual_seed(23), 16, 544
    x, w = _pair(T, (n_q + 2 * n_kv) * hd, K, 24)
    x, w = x.to(DEV), ops.block_weight(w.to(DEV))
    cos, sin = (torch.rand(T + 5, hd // 2, generator=g).to(DEV) for _ in range(2))
    blocks = (T + 5 + page - 1) // page
    positions, seq = torch.arange(5, T + 5, dtype=torch.int32, device=DEV), torch.zeros(T, dtype=torch.int32, device=DEV)
    table = torch.randperm(blocks, generator=g).view(1, blocks).to(torch.int32).to(DEV)

    def run(tile):
        q = torch.zeros(T, n_q * hd, dtype=torch.bfloat16, device=DEV)
        k = torch.zeros(blocks, n_kv, page, hd, dtype=torch.bfloat16, device=DEV)
        v = torch.zeros(blocks, n_kv, hd, page, dtype=torch.bfloat16, device=DEV)
        ops.mfma.gemm_qkv_rope(x, w, cos, sin, positions, seq, table, q, k, v, n_q, n_kv, hd, tile=tile)
        return q, k, v
    want = run(128)
    for rows, cols in [(0, 0)] + tiles:
        got = run(PANEL + 1000 * rows + cols if rows else 0)
        assert all(torch.equal(a, b) for a, b in zip(got, want)), (rows, cols)


def _chosen_on_256_units(ops, want, *args):
    """That the sizes still mean what the test takes them for (the plans are drawn for 256 compute units)."""
    got = ops.mfma.gemm_bf16_chosen(*args)
    assert got == want or ops.mfma.compute_units() != 256, (args, got)


# sizes at which each of these tiles is the chosen one, stored and added, or gated (two of them hold pairs), at the least k that they are chosen for
# and above; and sizes just outside, where the tiles through registers (0), 256 x 256 or narrower panels are
@pytest.mark.parametrize("M,N,K,gated,tile", [
    (329, 12288, 2048, False, PANEL + 96192), (403, 12288, 2048, False, PANEL + 128192),
    (2300, 3072, 2048, False, PANEL + 160192), (1800, 4608, 2048, False, PANEL + 192192), (390, 16384, 2048, False, PANEL + 128256),
    (514, 16384, 2048, False, PANEL + 192256), (218, 28672, 512, True, PANEL + 128256), (390, 12288, 512, True, PANEL + 128256),
    (292, 28672, 2048, True, PANEL + 192256), (1287, 6144, 1024, True, PANEL + 192256),
    (1924, 3072, 1024, False, 0), (2119, 4096, 1024, False, 256256), (2048, 3072, 544, False, 0), (2995, 3072, 512, False, 256256), (1400, 16384, 512, True, 256256), (1000, 3072, 8192, False, PANEL + 112128)])
def test_the_chosen_wide_panel_adds_in_the_order_of_the_others(ops, M, N, K, gated, tile):
    a, w = _pair(M, N, K, 25)
    ad, wb = a.to(DEV), ops.block_weight(w.to(DEV))
    _chosen_on_256_units(ops, tile, "gated" if gated else "stored", M, N, K)
    for accumulate in (False, True):
        if gated and accumulate:
            continue
        got, want = (torch.zeros(M, N // 2 if gated else N, dtype=torch.bfloat16 if gated else torch.float32, device=DEV) for _ in range(2))
        ops.gemm_bf16(ad, wb, got, accumulate, gated=gated, ksplit=1 if accumulate else 0)
        ops.gemm_bf16(ad, wb, want, accumulate, gated=gated, tile=128, ksplit=1 if accumulate else 0)
        assert torch.equal(got, want), accumulate


# shares of k that end inside the others' slabs, a short last one, and empty ones (eight of five slabs of 64 k)
@pytest.mark.parametrize("M,N,K,n", [(200, 400, 288, 8), (193, 208, 1056, 3), (97, 272, 2080, 2), (385, 528, 544, 3), (129, 256, 4128, 8)])
@pytest.mark.parametrize("rows,cols", TILES)
def test_parts_of_a_sum_in_wide_panels(ops, M, N, K, n, rows, cols):
    """The parts add up to the product (32-bit sums of bfloat16 products: 2e-5), each is there, and run after run they are the same bits."""
    a, w = _pair(M, N, K, 27)
    ref = a.double() @ w.double().T
    ad, wb = a.to(DEV), ops.block_weight(w.to(DEV))
    parts = [torch.full((n, M, N), float("nan"), device=DEV) for _ in range(2)]
    for p in parts:
        ops.mfma.gemm_parts(ad, wb, p, tile=1000 * rows + cols)
    assert torch.equal(parts[0], parts[1])
    assert float((parts[0].cpu().double().sum(0) - ref).norm() / ref.norm()) < 2e-5


@pytest.mark.parametrize("M,N,K,n,tile", [(1000, 3072, 8192, 2, PANEL + 128192), (800, 4096, 14336, 2, PANEL + 160192)])
def test_the_chosen_wide_panel_of_a_sum_in_parts(ops, M, N, K, n, tile):
    _chosen_on_256_units(ops, tile, "parts", M, N, K, n)
    assert ops.mfma.compute_units() != 256 or ops.mfma.entry("llme_gemm_parts_plan")(M, N, K, 0) == n
    a, w = _pair(M, N, K, 28)
    ref = a.double() @ w.double().T
    ad, wb, parts = a.to(DEV), ops.block_weight(w.to(DEV)), torch.full((n, M, N), float("nan"), device=DEV)
    ops.mfma.gemm_parts(ad, wb, parts)
    assert float((parts.cpu().double().sum(0) - ref).norm() / ref.norm()) < 2e-5


# (0: the chosen tile is no panel)
@pytest.mark.parametrize("M,N,K,tile", [(65, 48, 512, PANEL + 32064), (200, 528, 2080, PANEL + 32064), (273, 12288, 512, 0), (1500, 3072, 544, 0),
                                        (249, 12288, 1024, 0),
                                        (325, 12288, 1024, 0), (329, 12288, 2048, PANEL + 96192), (1287, 6144, 1024, PANEL + 192192)])
def test_squared_rectifier_behind_the_panels(ops, M, N, K, tile):
    """The squared positive part, stored in bfloat16: every tile and the chosen one give the bits of the square of the stored sum."""
    _chosen_on_256_units(ops, tile, "squared", M, N, K)
    a, w = _pair(M, N, K, 26)
    ad, wb = a.to(DEV), ops.block_weight(w.to(DEV))
    p = torch.empty(M, N, device=DEV)
    ops.gemm_bf16(ad, wb, p, tile=128)
    want = torch.clamp(p, min=0.0).square().to(torch.bfloat16)
    got = torch.zeros_like(want)
    ops.gemm_squared_relu(ad, wb, got, None)
    assert torch.equal(got, want)
    m = ops.mfma
    for rows, cols in TILES + [(32, 64), (96, 64), (48, 128), (144, 128)]:
        got.zero_()
        m.check(m.entry("llme_gemm_bf16")(m.ptr(ad), m.ptr(wb), m.ptr(got), 1, M, N, K, 0, 5, 0, 0, PANEL + 1000 * rows + cols, 1, -1,
                                          m.stream()), "squared")
        assert torch.equal(got, want), (rows, cols)
