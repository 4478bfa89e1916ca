"""The prompt attention kernel's turns over stretches of 64 keys (csrc/attention_prefill.hip): scores a stretch ahead, operands
straight into LDS, halves outside an item's keys replaced by the nearest one inside."""
import math

import pytest
import torch

import test_kernels_gpu as kernel_tests

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    from llmengine import ops
    return ops


# one stretch, two, an odd number, more than the 64 whose pages one look at the table brings; rows that end in either half of a block
@pytest.mark.parametrize("hd,n_q,n_kv", [(64, 4, 1), (64, 3, 3), (128, 4, 1), (128, 2, 1)])
@pytest.mark.parametrize("page,window", [(16, 0), (64, 0), (32, 100)])
@pytest.mark.parametrize("half", [False, True])
def test_turns(ops, hd, n_q, n_kv, page, window, half):
    lens, news = [2, 63, 64, 65, 129, 4230, 4129], [2, 63, 64, 33, 129, 70, 3]
    out, ref, plan = kernel_tests._attn_case(ops, lens, news, n_q, n_kv, hd, page, window=window, seed=71, prefill_splits=1,
                                             tuning=ops.mfma.attention_tuning(shared=3 if half else 2))
    assert plan["prefill_splits"] == 1 and bool(plan["tuning"] & ops.mfma.TUNING_HALF_ROWS) == half
    assert not out.isnan().any()
    assert kernel_tests._rel(out, ref) < 8e-3              # bfloat16 in and out, 32-bit sums


@pytest.mark.parametrize("hd,n_q,n_kv", [(64, 1, 1), (64, 4, 1), (128, 1, 1), (128, 2, 1)])
@pytest.mark.parametrize("half", [False, True])
def test_values_of_unseen_blocks_reach_no_row(ops, hd, n_q, n_kv, half):
    """An infinite value at a key: rows that see nothing of the key's block of 32, before it or (a window of 40) behind it, are what they are
    without it."""
    T, page, at, window = 230, 16, 110, 40
    g = torch.Generator().manual_seed(72)
    k, v = torch.randn(T, n_kv, hd, generator=g), torch.randn(T, n_kv, hd, generator=g)
    q = torch.randn(T, n_q * hd, generator=g).to(torch.bfloat16).to(DEV)
    blocks = (T + page - 1) // page
    i32 = dict(dtype=torch.int32, device=DEV)
    plan = ops.mfma.plan_attention([T], [0], n_q, n_kv, hd, tuning=ops.mfma.attention_tuning(shared=3 if half else 2))
    assert plan["prefill_splits"] == 1 and bool(plan["tuning"] & ops.mfma.TUNING_HALF_ROWS) == half

    def run(values):
        kc = torch.zeros(blocks * page, n_kv, hd)
        vc = torch.zeros(blocks * page, n_kv, hd)
        kc[:T], vc[:T] = k, values
        kc = kc.view(blocks, page, n_kv, hd).permute(0, 2, 1, 3).contiguous().to(torch.bfloat16).to(DEV)
        vc = vc.view(blocks, page, n_kv, hd).permute(0, 2, 3, 1).contiguous().to(torch.bfloat16).to(DEV)
        out = torch.zeros_like(q)
        ops.mfma.attention_bf16(q, kc, vc, out, torch.tensor([0, T], **i32), torch.tensor([0], **i32),
                                torch.arange(blocks, **i32).view(1, blocks), n_q, n_kv, hd, 1.0 / math.sqrt(hd), window, plan)
        return out

    spoilt = v.clone()
    spoilt[at] = float("inf")
    want, got = run(v), run(spoilt)
    first, last = at // 32 * 32, at // 32 * 32 + 31
    # a wavefront's rows are 16 or 32: what it shares with a row that sees the block is left out
    untouched = [r for r in range(T) if r // 32 * 32 + 31 < first or r // 32 * 32 - window + 1 > last]
    assert untouched[0] == 0 and untouched[-1] == T - 1
    assert torch.equal(got[untouched], want[untouched]) and not got[untouched].isnan().any()
    assert got[at].isinf().all() and got[at + window - 1].isinf().all()


@pytest.mark.parametrize("hd,n_q,n_kv", [(64, 8, 2), (64, 3, 3), (128, 8, 2), (128, 3, 3)])
@pytest.mark.parametrize("window", [0, 1, 7, 64, 65, 200])
@pytest.mark.parametrize("half", [False, True])
def test_turns_behind_a_window_and_beside_decoded_tokens(ops, hd, n_q, n_kv, window, half):
    """Items of whole and of half the rows whose keys are not cut: first stretches that no row of a wavefront sees yet, decoded tokens in
    the same launch."""
    out, ref, plan = kernel_tests._attn_case(ops, [300, 70, 1, 190, 333], [140, 70, 1, 2, 1], n_q, n_kv, hd, 16, window=window, seed=73,
                                             tuning=ops.mfma.attention_tuning(shared=3 if half else 2))
    assert plan["prefill_splits"] == 1 and plan["n_decode"] == 2 and bool(plan["tuning"] & ops.mfma.TUNING_HALF_ROWS) == half
    assert not out.isnan().any() and kernel_tests._rel(out, ref) < 8e-3      # bfloat16 in and out, 32-bit sums
