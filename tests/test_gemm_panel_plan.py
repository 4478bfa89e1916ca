"""The plans of products whose rows are a tile or two high (csrc/gemm_panel.hip), which the host makes: no device."""
import time

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
