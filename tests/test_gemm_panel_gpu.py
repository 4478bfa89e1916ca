"""Products whose rows are a tile or two high (csrc/gemm_panel.hip) and the norm that joins the parts of a sum."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
PANEL = 1000000
TILES = [(16 * m, 64) for m in range(2, 7)] + [(16 * m, 128) for m in range(3, 13)]


@pytest.fixture(scope="module")
def ops():
    from llmengine import ops
    return ops


def _pair(M, N, K, seed):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(M, K, generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g) * 0.05).to(torch.bfloat16)
    return a, w, a.double() @ w.double().T


def _rel(got, want):
    return float((got - want).norm() / want.norm())


# rows around a tile's edges, columns that end inside a tile, k of less than a slab, of one, ending in a part of one and of many
@pytest.mark.parametrize("M,N,K", [(1, 32, 32), (17, 64, 64), (33, 96, 160), (48, 160, 2048), (150, 288, 4128), (193, 2048, 288), (401, 320, 1056)])
@pytest.mark.parametrize("rows,cols", TILES)
def test_panel_tiles(ops, M, N, K, rows, cols):
    """Every tile: stored, added and gated sums against 64 bits (32-bit sums of bfloat16 products: 2e-5 as for the other tiles,
    5e-3 rounded, 8e-3 behind an activation), and the same bits as the tile through registers makes of them."""
    a, w, ref = _pair(M, N, K, 5)
    ad, wb, tile = a.to(DEV), ops.block_weight(w.to(DEV)), PANEL + 1000 * rows + cols
    out = torch.full((M, N), float("nan"), device=DEV)
    ops.gemm_bf16(ad, wb, out, tile=tile)
    assert _rel(out.cpu().double(), ref) < 2e-5
    other = torch.empty_like(out)
    ops.gemm_bf16(ad, wb, other, tile=128)
    assert torch.equal(out, other)
    base = torch.randn(M, N, generator=torch.Generator().manual_seed(6))
    acc, other = base.clone().to(DEV), base.clone().to(DEV)
    ops.gemm_bf16(ad, wb, acc, accumulate=True, tile=tile)
    assert _rel(acc.cpu().double(), ref + base.double()) < 2e-5
    ops.gemm_bf16(ad, wb, other, accumulate=True, tile=128, ksplit=1)
    assert torch.equal(acc, other)
    gated, other = (torch.empty(M, N // 2, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    ops.gemm_bf16(ad, wb, gated, gated=True, tile=tile)
    ops.gemm_bf16(ad, wb, other, gated=True, tile=128)
    assert torch.equal(gated, other)
    gu = ref.view(M, N // 32, 2, 16)
    gate = gu[:, :, 0]
    want = (gate * torch.sigmoid(gate) * gu[:, :, 1]).reshape(M, N // 2)
    assert _rel(gated.cpu().double(), want) < 8e-3


@pytest.mark.parametrize("M,N,K", [(65, 4096, 512), (65, 16, 512), (70, 128, 2048), (150, 16384, 1024), (273, 3072, 2048), (528, 640, 544), (1040, 2048, 1024)])
def test_the_chosen_tile_adds_in_the_order_of_the_others(ops, M, N, K):
    """What a product of more than 64 rows stores, adds with a fixed order or gates does not depend on the tile that is chosen for its
    sizes: the bits of the tile through registers, at sizes on both sides of every rule."""
    a, w, _ = _pair(M, N, K, 12)
    ad, wb = a.to(DEV), ops.block_weight(w.to(DEV))
    for accumulate, gated in ((False, False), (True, False), (False, True)):
        if gated and N % 32:
            continue
        got, want = (torch.zeros(M, N // 2 if gated else N, dtype=torch.bfloat16 if gated else torch.float32, device=DEV) for _ in range(2))
        ops.gemm_bf16(ad, wb, got, accumulate, gated=gated, ksplit=1 if accumulate else 0)
        ops.gemm_bf16(ad, wb, want, accumulate, gated=gated, tile=128, ksplit=1 if accumulate else 0)
        assert torch.equal(got, want), (accumulate, gated)


# the chosen tile at sizes whose k ends inside a slab, with and without biases and a limit
@pytest.mark.parametrize("T,FF,K,bias,limit", [(70, 256, 544, True, 0.0), (150, 208, 1056, False, 1.5), (273, 2048, 512, True, 2.0)])
def test_panel_tiles_gate_with_biases_and_clamps(ops, T, FF, K, bias, limit):
    """The gated epilogue that adds biases and clamps, behind every tile: against 64 bits (5e-3 as for the other tiles), and the bits
    of the tile through registers."""
    x, w, ref = _pair(T, 2 * FF, K, 13)
    both = torch.randn(2 * FF, generator=torch.Generator().manual_seed(14)).to(torch.bfloat16)
    ref = ref + (both.double() if bias else 0.0)
    g, u = (ref.view(T, FF // 16, 2, 16)[:, :, i].reshape(T, FF) for i in (0, 1))
    alpha = 1.702 if limit else 1.0
    if limit:
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
        assert (g == limit).any() and (u == -limit).any()
    want = g * torch.sigmoid(alpha * g) * (u + 1 if limit else u)
    xd, wb, bd = x.to(DEV), ops.block_weight(w.to(DEV)), both.to(DEV) if bias else None
    mfma = ops.mfma

    def run(tile):
        out = torch.zeros(T, FF, dtype=torch.bfloat16, device=DEV)
        mfma.check(mfma.entry("llme_gemm_bf16_gated_extra")(mfma.ptr(xd), mfma.ptr(wb), mfma.ptr(out), T, 2 * FF, K, mfma.ptr(bd) if bias else None,
                                                            limit, alpha, tile, 1, -1, mfma.stream()), "gemm_gated_extra")
        return out
    other, chosen = run(128), torch.zeros(T, FF, dtype=torch.bfloat16, device=DEV)
    assert _rel(other.cpu().double(), want) < 5e-3
    assert ops.gemm_gated_extra(xd, wb, chosen, 16, bd, limit, alpha) and torch.equal(chosen, other)
    for rows, cols in TILES + [(128, 256), (192, 256)]:
        assert torch.equal(run(PANEL + 1000 * rows + cols), other), (rows, cols)


def test_panel_reads_zeros_behind_the_last_row_and_the_end_of_k(ops):
    """What lies behind the operands' edges (the next rows' weights, here infinities and NaN) joins no sum."""
    M, N, K = 20, 48, 96
    a, w, ref = _pair(M + 30, N + 16, K, 7)
    a[M:], w[N:] = float("nan"), float("inf")
    ad, wb = a.to(DEV), ops.block_weight(w.to(DEV))
    for rows, cols in TILES:
        out = torch.zeros(M, N, device=DEV)
        ops.gemm_bf16(ad[:M], wb[:N // 16], out, tile=PANEL + 1000 * rows + cols)
        assert _rel(out.cpu().double(), ref[:M, :N]) < 2e-5, (rows, cols)


@pytest.mark.parametrize("M,N,K,n", [(17, 64, 1024, 2), (45, 2048, 2048, 4), (150, 160, 4128, 8), (273, 272, 288, 5), (600, 96, 512, 3)])
def test_parts_of_a_sum(ops, M, N, K, n):
    """The parts add up to the product (also where the last share of k is empty), and run after run they are the same bits."""
    a, w, ref = _pair(M, N, K, 8)
    ad, wb = a.to(DEV), ops.block_weight(w.to(DEV))
    parts = [torch.full((n, M, N), float("nan"), device=DEV) for _ in range(2)]
    for p in parts:
        ops.mfma.gemm_parts(ad, wb, p)
    assert _rel(parts[0].cpu().double().sum(0), ref) < 2e-5 and torch.equal(parts[0], parts[1])


@pytest.mark.parametrize("T,H,n", [(1, 4, 1), (17, 100, 2), (40, 2048, 3), (33, 3072, 8), (19, 4096, 5), (18, 8192, 9)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_parts_norm(ops, T, H, n, dtype):
    g = torch.Generator().manual_seed(9)
    h, parts = torch.randn(T, H, generator=g), torch.randn(n, T, H, generator=g)
    weight = (1 + 0.1 * torch.randn(H, generator=g)).to(dtype)
    hd, x = h.clone().to(DEV), torch.empty(T, H, dtype=torch.bfloat16, device=DEV)
    ops.mfma.parts_norm(hd, parts.to(DEV), weight.to(DEV), 1e-5, x)
    s = h.double() + parts.double().sum(0)
    want = weight.double() * s / torch.sqrt((s * s).mean(-1, keepdim=True) + 1e-5)
    assert _rel(hd.cpu().double(), s) < 1e-6 and _rel(x.cpu().double(), want) < 5e-3


@pytest.mark.parametrize("hd,n_q,n_kv", [(16, 8, 4), (64, 8, 2), (128, 4, 2)])
@pytest.mark.parametrize("T", [17, 100, 273])
def test_panel_tiles_rotate_as_the_others(ops, hd, n_q, n_kv, T):
    """The rotating epilogue behind every tile that holds whole heads, and behind the chosen one: the bits of the tile through
    registers."""
    g, page, K = torch.Generator().manual_seed(10), 16, 544
    x = torch.randn(T, K, generator=g).to(torch.bfloat16).to(DEV)
    w = ops.block_weight((0.05 * torch.randn((n_q + 2 * n_kv) * hd, K, generator=g)).to(torch.bfloat16).to(DEV))
    ang = torch.arange(T + 5, dtype=torch.float64)[:, None] / (10000.0 ** (torch.arange(hd // 2, dtype=torch.float64) * 2 / hd))[None, :]
    cos, sin = torch.cos(ang).float().to(DEV), torch.sin(ang).float().to(DEV)
    blocks = (T + 5 + page - 1) // page
    positions, seq = torch.arange(5, T + 5, dtype=torch.int32, device=DEV), torch.zeros(T, dtype=torch.int32, device=DEV)
    table = torch.randperm(blocks, generator=g).view(1, blocks).to(torch.int32).to(DEV)

    def run(tile):
        made = [torch.zeros(T, n_q * hd, dtype=torch.bfloat16, device=DEV), torch.zeros(blocks, n_kv, page, hd, dtype=torch.bfloat16, device=DEV),
                torch.zeros(blocks, n_kv, hd, page, dtype=torch.bfloat16, device=DEV)]
        ops.gemm_qkv_rope(x, w, cos, sin, positions, seq, table, *made, n_q, n_kv, hd, tile=tile)
        return made
    want = run(128)
    for tile in [0] + [PANEL + 1000 * rows + cols for rows, cols in TILES if cols % hd == 0]:
        for a, b in zip(want, run(tile)):
            assert torch.equal(b, a), tile


# pieces of 16 bytes past the end of k, columns that end inside a tile, one row of tiles and several
@pytest.mark.parametrize("M,N,K", [(17, 64, 20), (33, 100, 2052), (81, 48, 64), (149, 272, 288), (300, 2048, 1024), (40, 3076, 68), (1100, 300, 100)])
def test_panel_tiles_of_32_bit_operands(ops, M, N, K):
    """32-bit operands with a row-major W: stored and added (by the kernel that launch_generic takes for the sizes, of both) and in parts
    (always the panel), against 64 bits (32-bit sums of up to 2,052 products, some eight additions of which are of long partial
    sums: 1e-6)."""
    g = torch.Generator().manual_seed(11)
    a, w = torch.randn(M, K, generator=g), 0.05 * torch.randn(N, K, generator=g)
    ref = a.double() @ w.double().T
    ad, wd = a.to(DEV), w.to(DEV)
    for accumulate in (False, True):
        out = torch.full((M, N), 1.0 if accumulate else float("nan"), device=DEV)
        ops.gemm_generic(ad, wd, out, accumulate)
        assert _rel(out.cpu().double(), ref + (1.0 if accumulate else 0.0)) < 1e-6
    for n in (2, 5):
        for rows, cols in [(0, 0)] + TILES:
            parts = torch.full((n, M, N), float("nan"), device=DEV)
            ops.mfma.gemm_parts(ad, wd, parts, tile=1000 * rows + cols)
            assert _rel(parts.cpu().double().sum(0), ref) < 1e-6, (n, rows, cols)


@pytest.mark.parametrize("M", [1, 2, 3, 8, 13, 16])
@pytest.mark.parametrize("N,K", [(32, 60), (64, 1028), (9000, 64), (8224, 1024)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_32_bit_products_of_few_rows_with_the_norm_inside(ops, M, N, K, dtype):
    """Whole columns and k in four, plain over chosen rows and gated, against 64 bits."""
    g = torch.Generator().manual_seed(12)
    h, w = torch.randn(M + 3, K, generator=g), 0.05 * torch.randn(N, K, generator=g)
    weight = (1 + 0.1 * torch.randn(K, generator=g)).to(dtype)
    rows = torch.randperm(M + 3, generator=g)[:M].to(torch.int32)

    def normed(x):
        x = x.double()
        return weight.double() * x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5)
    out = torch.full((M, N), float("nan"), device=DEV)
    ops.gemv_norm(h.to(DEV), weight.to(DEV), 1e-5, w.to(DEV), out, rows=rows.to(DEV))
    assert _rel(out.cpu().double(), normed(h[rows.long()]) @ w.double().T) < 1e-6
    if N % 32 == 0:
        gated = torch.full((M, N // 2), float("nan"), device=DEV)
        ops.gemv_norm(h[:M].contiguous().to(DEV), weight.to(DEV), 1e-5, w.to(DEV), gated, gated=True)
        gu = (normed(h[:M]) @ w.double().T).view(M, N // 32, 2, 16)
        want = (gu[:, :, 0] * torch.sigmoid(gu[:, :, 0]) * gu[:, :, 1]).reshape(M, N // 2)
        assert _rel(gated.cpu().double(), want) < 2e-6


@pytest.mark.parametrize("dtype,tol", [("fp32", 1e-5), ("bf16", 2e-2)])
def test_a_step_whose_sums_stay_in_parts(ops, monkeypatch, dtype, tol):
    """A prompt of rows enough that the sums into the stream are left in parts for the norms: the logits of the same model whose sums
    have a fixed order, where no sum is (1e-5 and 2e-2 as the engine's other tests allow between orders of sums). The last
    layer's down-proj, behind which no block's norm stands, adds into the stream itself."""
    from llmengine import Engine
    cfg = {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "hidden_size": 1024, "intermediate_size": 2048, "num_hidden_layers": 3,
           "num_attention_heads": 16, "num_key_value_heads": 4, "head_dim": 64, "vocab_size": 512, "max_position_embeddings": 1024,
           "rms_norm_eps": 1e-5, "rope_theta": 10000.0, "tie_word_embeddings": True}
    launched, wanted = ops.mfma._launch_parts, []
    monkeypatch.setattr(ops.mfma, "_launch_parts", lambda *a, **k: wanted.append(a[2].shape) or launched(*a, **k))
    prompt = [(7 * i * i + 3 * i) % 512 for i in range(150)]
    logits = []
    for fixed in (True, False):
        engine = Engine.from_random(cfg, 3, dtype, std=0.05, norm_std=0.05, deterministic=fixed)
        logits.append(torch.as_tensor(engine.forward_logits(prompt)).double())
        assert len(wanted) == (0 if fixed else 5), wanted            # (o-proj three times, down-proj twice)
    assert _rel(logits[1], logits[0]) < tol


def test_a_block_on_its_own_leaves_the_stream_whole(ops):
    """A program that runs one block of a model itself, after passes of the whole model in which that block handed its last sum on in
    parts: the stream behind it holds the whole sum, as before the first pass (the two differ by the order of 32-bit sums)."""
    from llmengine import Engine
    cfg = {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "hidden_size": 1024, "intermediate_size": 2048, "num_hidden_layers": 2,
           "num_attention_heads": 16, "num_key_value_heads": 4, "head_dim": 64, "vocab_size": 512, "max_position_embeddings": 1024,
           "rms_norm_eps": 1e-5, "rope_theta": 10000.0, "tie_word_embeddings": True}
    engine = Engine.from_random(cfg, 3, "fp32", std=0.05, norm_std=0.05)
    model, left = engine.model, []
    whole = model.forward

    def forward(step, caches, rows):
        h = step.buffer("test.hidden", (step.num_tokens, model.hidden_size), torch.float32)
        model.embedding.forward(step.tokens, h, step)
        model.layers[0].forward(h, step, caches[model.schedule[0].cache_id], True)
        left.append(h.double())
        return whole(step, caches, rows)
    model.forward = forward
    for _ in range(2):
        engine.forward_logits([(7 * i * i + 3 * i) % 512 for i in range(150)])
    assert _rel(left[1], left[0]) < 1e-5


def test_parts_and_blocks_whose_forward_was_replaced_see_the_whole_stream(ops):
    """A block and a mixer whose `forward` a program has replaced (to look at what they make) run as they were given, with a whole stream
    in front of and behind them, in a step whose other sums stay in parts."""
    from llmengine import Engine
    cfg = {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "hidden_size": 1024, "intermediate_size": 2048, "num_hidden_layers": 4,
           "num_attention_heads": 16, "num_key_value_heads": 4, "head_dim": 64, "vocab_size": 512, "max_position_embeddings": 1024,
           "rms_norm_eps": 1e-5, "rope_theta": 10000.0, "tie_word_embeddings": True}
    prompt, seen, logits = [(7 * i * i + 3 * i) % 512 for i in range(150)], [], []
    for fixed in (True, False):
        engine = Engine.from_random(cfg, 3, "fp32", std=0.05, norm_std=0.05, deterministic=fixed)
        block, mixer = engine.model.layers[1], engine.model.layers[2].mixer
        block_forward, mixer_forward, states = block.forward, mixer.forward, []

        def watched_block(h, *args):
            states.append(h.double())
            block_forward(h, *args)
            states.append(h.double())

        def watched_mixer(x, step, cache, out, accumulate, *args):
            mixer_forward(x, step, cache, out, accumulate, *args)
            states.append(out.double())
        block.forward, mixer.forward = watched_block, watched_mixer
        logits.append(torch.as_tensor(engine.forward_logits(prompt)).double())
        seen.append(states)
    assert len(seen[0]) == len(seen[1]) == 3
    for whole, got in zip(*seen):
        assert _rel(got, whole) < 1e-5
    assert _rel(logits[1], logits[0]) < 1e-5
