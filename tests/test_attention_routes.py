"""Which way a step's q/k/v product goes: cut over k into a cleared sum with the rotation behind it, or with the rotation and the
cache write in its epilogue. On the CPU, with the operations replaced by a record of their calls."""
import types

import pytest
import torch

from llmengine import ops
from llmengine.parts import Attention
from llmengine.parts.base import LayerCache, PositionEncoding

LAYER_MB = 122              # of the 1B sizes


class Tables(PositionEncoding):
    def __init__(self, rotary_dim):
        self.tables = (torch.ones(16384, rotary_dim // 2), torch.zeros(16384, rotary_dim // 2), rotary_dim)

    def rotary_tables(self):
        return self.tables


class Turned(PositionEncoding):
    """An encoding that transforms q and k itself."""
    def apply(self, q, k, positions):
        pass


def _attention(hd, position, layer_mb=LAYER_MB):
    attn = Attention(64, 4, 2, hd, position=position)
    attn.w_qkv = torch.zeros(8 * hd, 64, dtype=torch.bfloat16)
    attn.w_o = torch.zeros(64, 4 * hd, dtype=torch.bfloat16)
    attn.layer_bytes = None if layer_mb is None else layer_mb * 10 ** 6
    return attn


def _step(new_lens, ctx_lens, choices=None):
    T, held = sum(new_lens), {}

    def buffer(name, shape, dtype):
        need = torch.Size(shape).numel()
        if name not in held or held[name].numel() < need:
            held[name] = torch.empty(need, dtype=dtype)
        return held[name][:need].view(shape)
    return types.SimpleNamespace(num_tokens=T, num_seqs=len(new_lens), new_lens=list(new_lens), ctx_lens=list(ctx_lens), act_dtype=torch.bfloat16,
                                 max_position=max(ctx_lens) + max(new_lens), positions=None, seq_idx=None, block_tables={"full": None},
                                 buffer=buffer, extra={}, choices=choices, fixed_order=False)


def _run(monkeypatch, attn, step, calls=None):
    calls = [] if calls is None else calls
    for name in ("gemm", "gemm_qkv_rope", "rope_kv_write", "clear", "attention_project"):
        monkeypatch.setattr(ops, name, lambda *a, _name=name, **k: calls.append(_name + (" add" if k.get("accumulate") else "")))
    monkeypatch.setattr(ops.mfma, "attention_decode_rope", lambda *a, **k: calls.append("attention_decode_rope") or True)
    hd, T = attn.head_dim, step.num_tokens
    cache = LayerCache(paged={"k": torch.zeros(1, 2, 16, hd, dtype=torch.bfloat16), "v": torch.zeros(1, 2, hd, 16, dtype=torch.bfloat16)},
                       state={}, page_size=16, group="full")
    attn.forward(torch.zeros(T, 64, dtype=torch.bfloat16), step, cache, torch.zeros(T, 64), True)
    return calls


def _route(monkeypatch, attn, step):
    calls = _run(monkeypatch, attn, step)
    return "epilogue" if "gemm_qkv_rope" in calls else "sum" if "gemm add" in calls else "stored"


PROMPT, MIXED = ([45], [0]), ([20] + [1] * 10, [0] * 11)


@pytest.mark.parametrize("hd", [16, 32, 64])
@pytest.mark.parametrize("lens", [PROMPT, MIXED, ([17], [0]), ([64], [0])])
def test_short_prompts_of_layers_that_the_host_outlasts_rotate_in_the_epilogue(monkeypatch, hd, lens):
    assert _route(monkeypatch, _attention(hd, Tables(hd)), _step(*lens)) == "epilogue"


@pytest.mark.parametrize("lens", [PROMPT, MIXED, ([1] * 20, [5] * 20)])
@pytest.mark.parametrize("hd,rotary_dim", [(64, 32), (64, 0), (64, -1), (48, 48), (32, 16), (24, 24)])
def test_what_the_epilogue_cannot_rotate_keeps_the_sum(monkeypatch, lens, hd, rotary_dim):
    """Part of a head rotated, nothing rotated, an encoding of its own, head sizes that the epilogue does not take: the product would
    be stored uncut, and a launch would be saved nowhere."""
    position = Tables(rotary_dim) if rotary_dim > 0 else Turned() if rotary_dim < 0 else None
    assert _route(monkeypatch, _attention(hd, position), _step(*lens)) == "sum"


@pytest.mark.parametrize("hd,layer_mb,lens", [(64, 200, PROMPT), (64, 428, MIXED), (64, None, PROMPT), (128, LAYER_MB, PROMPT),
                                              (64, LAYER_MB, ([20] + [1] * 20, [0] + [15000] * 20))])
def test_layers_that_keep_the_chip_busy_keep_the_sum(monkeypatch, hd, layer_mb, lens):
    """Wide layers, heads of 128, and keys and values that take as long to read."""
    assert _route(monkeypatch, _attention(hd, Tables(hd), layer_mb), _step(*lens)) == "sum"


def test_choices_decide(monkeypatch):
    attn = _attention(64, Tables(64))
    assert _route(monkeypatch, attn, _step(*PROMPT, choices=ops.KernelChoices(launch_bound_layer_bytes=0))) == "sum"
    assert _route(monkeypatch, attn, _step(*PROMPT, choices=ops.KernelChoices(fast_gemm=False))) == "sum"


def test_more_rows_and_decoding_as_before(monkeypatch):
    assert _route(monkeypatch, _attention(64, Tables(64), 428), _step([65], [0])) == "epilogue"
    assert "attention_decode_rope" in _run(monkeypatch, _attention(64, Tables(64)), _step([1] * 20, [100] * 20))


@pytest.mark.parametrize("lens", [([1] * 20, [100] * 20), ([1] * 33, [7] * 33)])
def test_layers_with_and_without_rotation_share_the_cleared_sum(monkeypatch, lens):
    """What one layer's kernels leave zero is zero for the next, whichever of them it is: a step clears once."""
    step, calls = _step(*lens), []
    for position in (Tables(64), None, Tables(64), Tables(32), Tables(64)):
        _run(monkeypatch, _attention(64, position), step, calls)
    assert calls.count("gemm add") == 5 and calls.count("attention_decode_rope") == 3 and calls.count("rope_kv_write") == 2
    assert calls.count("clear") == 1 and calls[0] == "clear"


def test_a_model_tells_its_mixers_what_a_layer_weighs():
    from llmengine.models.llama import build_llama
    from llmengine.config.llama import LlamaConfig
    from llmengine.parts import Placement
    from llmengine.weights import random_state
    from tiny_models import TINY_B
    model = build_llama(LlamaConfig.from_dict(TINY_B))
    model.load_params(None, Placement(torch.device("cpu"), torch.bfloat16))
    per_layer = 2 * sum(t.numel() for n, t in random_state(TINY_B, 0, torch.bfloat16, 0.1, 1.0, 0.1) if ".layers.0." in n)
    assert per_layer > 0 and all(layer.mixer.layer_bytes == per_layer for layer in model.layers)
