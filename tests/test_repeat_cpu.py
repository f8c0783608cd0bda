"""Which steps are launched by making the second layer's launches again: the rule, without a device."""

from types import SimpleNamespace

import pytest
import torch

from rapid_llm_amd.config.qwen3 import Qwen3Config
from rapid_llm_amd.models.causal_lm import CausalLM
from rapid_llm_amd.models.qwen3 import build_qwen3_spec

BODY = dict(
    architectures=["Qwen3ForCausalLM"], model_type="qwen3", num_hidden_layers=5, hidden_size=64, num_attention_heads=4,
    num_key_value_heads=2, head_dim=16, intermediate_size=128, vocab_size=97, rope_theta=10000.0, rms_norm_eps=1e-6,
    tie_word_embeddings=True, max_position_embeddings=128, hidden_act="silu", attention_bias=False,
)


def _model(dtype=torch.bfloat16, **change):
    model = CausalLM(build_qwen3_spec(Qwen3Config.from_dict({**BODY, **change})))
    for block in model.blocks:
        for norm in (block.mixer_norm, block.feed_forward_norm):
            norm.dtype, norm.weight = dtype, torch.empty(norm.size, device="meta")
        for linear in (block.mixer.qkv, block.mixer.o, block.feed_forward.gate_up, block.feed_forward.down):
            linear.weight = torch.empty((linear.out_features, linear.in_features), dtype=dtype, device="meta")
    caches = [SimpleNamespace(group_id=0, page_size=16, owns_pages=True, pages={"k": None, "v": None}, states={}) for _ in range(5)]
    return model, caches


def _alike(model, caches, tokens=5, static=()):
    return model._alike(SimpleNamespace(num_tokens=tokens, static=dict(static)), caches)


def test_layers_of_one_model_are_alike():
    model, caches = _model()
    assert _alike(model, caches)
    assert not _alike(model, caches, static={"decode_only_tokens": 1}) and not _alike(model, caches, tokens=1 << 20)
    model.blocks[4].feed_forward.limit = 7.0
    assert not _alike(model, caches)


@pytest.mark.parametrize("layer", [0, 1, 4])
@pytest.mark.parametrize("where", ["mixer", "mixer_norm", "feed_forward_norm", "feed_forward", "block", "product", "kind"])
def test_a_layer_with_a_function_of_its_own_is_called(where, layer):
    """What somebody puts in the place of a part's or a product's own method runs in every step."""
    model, caches = _model()
    block = model.blocks[layer]
    if where == "product":
        block.mixer.qkv.product = lambda x, out_dtype=None: x
    elif where == "kind":
        block.feed_forward.down = SimpleNamespace(weight=None, bias=None)
    else:
        target = block if where == "block" else getattr(block, where)
        target.forward = target.forward
    assert not _alike(model, caches)


@pytest.mark.parametrize("where", ["mixer", "mixer_norm", "feed_forward", "block"])
def test_a_class_whose_forward_was_replaced_is_called(where, monkeypatch):
    model, caches = _model()
    kind = type(model.blocks[0] if where == "block" else getattr(model.blocks[0], where))
    inner = kind.forward
    monkeypatch.setattr(kind, "forward", lambda self, *args: inner(self, *args))
    assert not _alike(model, caches)


def test_steps_whose_temporary_tensors_are_large_are_not_repeated():
    """The noted layer keeps them all: a float32 step of a large model lets its layers give them back one by one."""
    from rapid_llm_amd.models.causal_lm import REPEAT_MAX_BYTES, REPEAT_MAX_TOKENS

    large = dict(hidden_size=5120, num_attention_heads=64, num_key_value_heads=8, head_dim=128, intermediate_size=25600)
    model, caches = _model(torch.float32, **large)
    assert _alike(model, caches, 17) and not _alike(model, caches, REPEAT_MAX_TOKENS)
    small = dict(hidden_size=1024, num_attention_heads=16, num_key_value_heads=8, head_dim=128, intermediate_size=3072)
    for dtype, tokens in ((torch.float32, 512), (torch.bfloat16, 192)):
        assert _alike(*_model(dtype, **small), tokens)
    # gate and up, the widest, is the most that is left alive: its result alone is within the bound
    rows = max(m for m in range(1, REPEAT_MAX_TOKENS) if _alike(model, caches, m))
    assert 4 * rows * 2 * 25600 < REPEAT_MAX_BYTES


def test_steps_with_library_products_are_told_beforehand():
    """Their layers are not looked at; what float32 layers and few rows launch is all this package's."""
    small = dict(hidden_size=1024, num_attention_heads=16, num_key_value_heads=8, head_dim=128, intermediate_size=3072)
    model, caches = _model(**small)
    for tokens, library in ((1, False), (16, False), (17, False), (64, False), (192, False), (193, True), (512, True), (2048, True)):
        assert model.blocks[0].calls_library(tokens) == library and _alike(model, caches, tokens) != library
    assert not _model(torch.float32, **small)[0].blocks[0].calls_library(2048)
    wide = dict(hidden_size=4096, num_attention_heads=32, num_key_value_heads=8, head_dim=128, intermediate_size=12288)
    model, _ = _model(**wide)
    assert not model.blocks[0].calls_library(64) and model.blocks[0].calls_library(65)  # (queries, keys and values)
