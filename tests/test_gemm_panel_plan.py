"""The plans of products whose rows are a tile or two high (csrc/gemm_panel.hip), which the host makes: no device."""
import time
import types

import pytest
import torch

from llmengine import ops
from llmengine.ops import mfma


def _seconds(plan, sizes, calls=600):
    best = float("inf")
    for _ in range(7):
        t = time.perf_counter()
        for _ in range(calls // len(sizes)):
            for s in sizes:
                plan(*s)
        best = min(best, time.perf_counter() - t)
    return best


def test_a_models_plans_are_kept_side_by_side():
    """A step asks for the plans of its layers' products in turn, layer after layer: they are estimated once. (An estimate takes several
    times a call that finds its plan; the best of several runs of each, so that a busy machine does not decide.)"""
    plan = mfma.entry("llme_gemm_parts_plan")
    one = _seconds(plan, [(273, 2048, 2048, 0)])
    for rows in (273, 150):
        step = [(rows, n, k, wide) for n, k in ((3072, 2048), (2048, 2048), (16384, 2048), (2048, 8192)) for wide in (0, 1)]
        assert _seconds(plan, step) < 1.6 * one


def test_only_steps_whose_products_are_ever_cut_hand_parts_on():
    """The rows from which and up to which a step's blocks ask for parts are those for which the plan names any."""
    sizes = [(2048, 8192), (2048, 2048), (4096, 14336), (256, 8192), (8192, 8192)]
    for dtype, rows in ((torch.bfloat16, (1, 16, 64, 65, 700, 1024, 1025, 2000, 2048)), (torch.float32, (1, 16, 17, 700, 1024, 1025, 2000))):
        step = types.SimpleNamespace(act_dtype=dtype, fixed_order=False, choices=ops.KernelChoices())
        for T in rows:
            cut = any(mfma.parts_plan(T, N, K, dtype == torch.float32) for N, K in sizes)
            assert mfma.sums_may_stay_in_parts(step, torch.empty(T, 2048)) == cut, (dtype, T)


def test_what_a_norm_cannot_join_is_not_left_in_parts():
    """A norm's weight that the joining kernel does not take (unaligned, strided, of another type) and operands that a product refuses:
    the sublayer adds into the stream itself, and says what it refuses itself."""
    h = torch.zeros(100, 256)
    step = types.SimpleNamespace(act_dtype=torch.bfloat16, fixed_order=False, choices=ops.KernelChoices(),
                                 buffer=lambda *a: pytest.fail("parts were asked for"))

    def adds(weight):
        return mfma.sum_for(types.SimpleNamespace(fused_rms=lambda: weight if weight is None else (weight, 1e-5)), h, step)
    whole = torch.ones(257)
    assert isinstance(adds(torch.ones(256)), mfma.LeftSum) and isinstance(adds(torch.ones(256, dtype=torch.bfloat16)), mfma.LeftSum)
    for weight in (None, whole[1:], torch.ones(512)[::2], whole, torch.ones(256, dtype=torch.float16), torch.ones(1, 256)):
        assert adds(weight) is True
    step.act_dtype = torch.float32
    assert adds(torch.ones(256, dtype=torch.bfloat16)) is True
    a, w = torch.zeros(100, 8192), torch.zeros(256, 8192)
    assert mfma.parts_plan(100, 256, 8192, True) > 1
    left = adds(torch.ones(256))
    for bad_a, bad_w, out in ((a, torch.zeros(8192, 256).T, h), (torch.zeros(8192, 100).T, w, h), (a, w.to(torch.bfloat16), h), (a[:, :4096], w, h),
                              (a, w, torch.zeros(100, 256)), (a[:50], w, h[:50]), (a, w, h[:])):
        assert not mfma.product_in_parts(left, bad_a, bad_w, out, step) and left.parts is None
    assert not mfma.product_in_parts(True, a, w, h, step) and not mfma.product_in_parts(False, a, w, h, step)
