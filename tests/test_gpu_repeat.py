"""Steps whose layers behind the second are launched from the second's notes: bit for bit what the layers'
own code launches, in every kind of step, and only where the layers are alike."""

import pytest
import torch

from tiny_configs import random_tokens

pytestmark = pytest.mark.gpu

BASE = dict(
    architectures=["Qwen3ForCausalLM"], model_type="qwen3", num_hidden_layers=5, hidden_size=256, num_attention_heads=4,
    num_key_value_heads=2, head_dim=64, intermediate_size=512, vocab_size=277, rope_theta=30000.0, rms_norm_eps=1e-5,
    tie_word_embeddings=False, max_position_embeddings=1024, hidden_act="silu", attention_bias=False,
)
# request -> its portions: single tokens eager and few rows of a prompt (norms inside the products), tens of rows (runs
# of K), a hundred and more, single tokens beside portions, a portion of a long prompt (its keys in runs)
STEPS = [{"a": 5}, {"a": 1, "b": 11}, {"a": 1, "b": 1}, {"c": 40, "a": 1}, {"d": 150, "b": 30, "c": 1},
         {"e": 640}, {"e": 130, "a": 1, "b": 1}]


def _run(runner, most, monkeypatch):
    from rapid_llm_amd import StepEntry
    from rapid_llm_amd.kernels import ops
    from rapid_llm_amd.models import causal_lm

    ran = []
    real = ops.repeat_launches
    monkeypatch.setattr(causal_lm, "REPEAT_MAX_TOKENS", most)
    monkeypatch.setattr(ops, "repeat_launches", lambda *a: ran.append(real(*a)) or ran[-1])
    done, logits = {}, []
    for i, step in enumerate(STEPS):
        entries = []
        for rid, n in step.items():
            tokens = random_tokens(n, runner.vocab_size, 100 * i + ord(rid))
            entries.append(StepEntry(rid, tokens, [n - 1]))
            done[rid] = done.get(rid, 0) + n
        logits.append(runner.step(entries, use_graph=False).clone())
    for rid in done:
        runner.finish(rid)
    monkeypatch.setattr(ops, "repeat_launches", real)
    return logits, ran


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("change", [{}, {"head_dim": 48, "num_attention_heads": 6, "hidden_size": 200},
                                    {"head_dim": 128, "num_hidden_layers": 4, "num_attention_heads": 12, "intermediate_size": 2048}],
                         ids=["d64", "d48", "d128"])
def test_repeated_layers_are_the_layers(dtype, change, monkeypatch):
    from rapid_llm_amd import EngineConfig, ModelRunner

    engine = EngineConfig(dtype=dtype, max_seq_len=1024, page_size=16, num_pages=200, max_num_seqs=8)
    runner = ModelRunner({**BASE, **change}, engine, load_format="random", weight_norm_std=0.1)
    want, none = _run(runner, 0, monkeypatch)
    got, ran = _run(runner, 2048, monkeypatch)
    # (a step with a product of the library's is launched by the layers; float32 has none, and the widths of the
    # last shape keep to this package's products up to 192 rows)
    least = 7 if dtype == "float32" else 6 if runner.config.head_dim == 128 else 3
    assert not none and ran == [True] * len(ran) and len(ran) >= least
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    # weights that are other tensors now are the ones that are read
    runner.model.blocks[3].feed_forward.down.weight = torch.zeros_like(runner.model.blocks[3].feed_forward.down.weight)
    want, got = _run(runner, 0, monkeypatch)[0], _run(runner, 2048, monkeypatch)[0]
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_layers_that_differ_are_not_repeated(monkeypatch):
    from rapid_llm_amd import EngineConfig, ModelRunner

    body = {**BASE, "sliding_window": 40, "layer_types": ["full_attention"] * 4 + ["sliding_attention"]}
    runner = ModelRunner(body, EngineConfig(dtype="bfloat16", max_seq_len=1024, page_size=16, num_pages=200, max_num_seqs=8),
                         load_format="random")
    assert _run(runner, 2048, monkeypatch)[1] == []
    few = ModelRunner({**BASE, "num_hidden_layers": 3}, EngineConfig(dtype="bfloat16", max_seq_len=1024, page_size=16, num_pages=200, max_num_seqs=8),
                      load_format="random")
    assert _run(few, 2048, monkeypatch)[1] == []


@pytest.mark.parametrize("where", ["mixer", "mixer_norm", "feed_forward_norm", "feed_forward", "block", "class", "product"])
def test_a_forward_put_in_the_place_of_a_layers_own_is_called(where, monkeypatch):
    """A timer or a hook around one layer's part, its block, its product or a part's class: called in every step."""
    from rapid_llm_amd import EngineConfig, ModelRunner, StepEntry
    from rapid_llm_amd.parts.mlp import SwiGLU

    runner = ModelRunner(BASE, EngineConfig(dtype="bfloat16", max_seq_len=1024, page_size=16, num_pages=200, max_num_seqs=8),
                         load_format="random", weight_norm_std=0.1)
    block, calls = runner.model.blocks[3], []
    target, name = {"block": (block, "forward"), "class": (SwiGLU, "forward"), "product": (block.feed_forward.down, "deferred")}.get(
        where, (getattr(block, where, None), "forward"))
    inner = getattr(target, name)
    step = lambda: runner.step([StepEntry("a", [5, 6, 7, 8, 9], [4])], use_graph=False).clone()
    want = step()
    runner.finish("a")
    monkeypatch.setattr(target, name, lambda *args, **kw: calls.append(0) or inner(*args, **kw))
    assert torch.equal(step(), want) and len(calls) == (5 if where == "class" else 1)


def test_every_layer_is_timed(monkeypatch):
    """Regions around parts count every layer of every step, prompts and single tokens."""
    from collections import Counter

    from rapid_llm_amd import EngineConfig, ModelRunner, StepEntry
    from rapid_llm_amd.engine.timeline import Timeline, instrument

    runner = ModelRunner(BASE, EngineConfig(dtype="bfloat16", max_seq_len=1024, page_size=16, num_pages=200, max_num_seqs=8),
                         load_format="random")
    timeline = Timeline()
    instrument(runner, timeline)
    runner.step([StepEntry("a", [5, 6, 7, 8, 9], [4])])
    for token in (3, 4, 5):
        runner.step([StepEntry("a", [token], [0])])
    seen = Counter((r.phase, r.name) for r in timeline.collect())
    for name in ("mixer norm (RMSNorm)", "mixer (GQAAttention)", "feed-forward norm (RMSNorm)", "feed-forward (SwiGLU)"):
        assert seen["steps with prompt portions", name] == 5 and seen["decode steps", name] == 15


@pytest.fixture
def biased():
    """BASE with biases on every projection: a down projection's is added by the norm behind, float32 too."""
    import dataclasses

    from rapid_llm_amd.config.qwen3 import Qwen3Config
    from rapid_llm_amd.config.registry import register_architecture, unregister_architecture
    from rapid_llm_amd.models.qwen3 import build_qwen3_spec

    def spec(cfg):
        whole = build_qwen3_spec(cfg)
        more = lambda part, **kw: dataclasses.replace(part, params={**part.params, **kw})
        return dataclasses.replace(whole, layers=tuple(
            dataclasses.replace(layer, mixer=more(layer.mixer, qkv_bias=True, o_bias=True),
                                feed_forward=more(layer.feed_forward, bias=True)) for layer in whole.layers))

    register_architecture("BiasedQwen3", Qwen3Config, spec)
    yield {**BASE, "architectures": ["BiasedQwen3"], "model_type": "BiasedQwen3"}
    unregister_architecture("BiasedQwen3")


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_repeated_layers_with_biases_and_products_cut_into_launches(biased, dtype, monkeypatch):
    """What a layer leaves is then read from several of its rows on."""
    from rapid_llm_amd import EngineConfig, ModelRunner
    from rapid_llm_amd.kernels import ops

    runner = ModelRunner(biased, EngineConfig(dtype=dtype, max_seq_len=1024, page_size=16, num_pages=200, max_num_seqs=8),
                         load_format="random", weight_norm_std=0.1)
    gen = torch.Generator(device="cuda").manual_seed(3)
    for name, t in runner.params.items():
        if "bias" in name:
            t.normal_(0.0, 0.1, generator=gen)
    monkeypatch.setattr(ops, "f32_wide", lambda m, n, k, units: 96 if m > 64 and k % 32 == 0 else 0)
    monkeypatch.setattr(ops, "_F32_MOST_PIECES", 1 << 20)
    assert ops._f32_piece_rows(640, 512) == 512  # the long portion's down projection: two launches
    want, _ = _run(runner, 0, monkeypatch)
    got, ran = _run(runner, 2048, monkeypatch)
    assert len(ran) >= (7 if dtype == "float32" else 3) and all(ran)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_weights_inside_a_unit_of_16_bytes_are_every_layers_own(monkeypatch):
    """Down projections over long sums whose rows begin inside a unit of 16 bytes."""
    from rapid_llm_amd import EngineConfig, ModelRunner

    runner = ModelRunner({**BASE, "intermediate_size": 8192},
                         EngineConfig(dtype="bfloat16", max_seq_len=1024, page_size=16, num_pages=200, max_num_seqs=8),
                         load_format="random", weight_norm_std=0.1)
    for block in runner.model.blocks:
        down = block.feed_forward.down
        room = torch.empty(down.weight.numel() + 1, dtype=down.weight.dtype, device="cuda")
        room[1:].view_as(down.weight).copy_(down.weight)
        down.weight = room[1:].view_as(down.weight)
        assert down.weight.data_ptr() % 16
    want, _ = _run(runner, 0, monkeypatch)
    got, _ = _run(runner, 2048, monkeypatch)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("how,dtype", [("odd", "bfloat16"), ("odd", "float32"), ("apart", "float32")])
def test_a_layer_whose_weight_lies_otherwise(how, dtype, monkeypatch):
    """One layer's product begins inside a unit of 16 bytes (float32: or has its rows apart): its launches are its own."""
    from rapid_llm_amd import EngineConfig, ModelRunner

    runner = ModelRunner({**BASE, "hidden_size": 1024, "intermediate_size": 3072},
                         EngineConfig(dtype=dtype, max_seq_len=1024, page_size=16, num_pages=200, max_num_seqs=8),
                         load_format="random", weight_norm_std=0.1)
    gate_up = runner.model.blocks[3].feed_forward.gate_up
    rows, k = gate_up.weight.shape
    room = torch.empty((rows + 1) * (k + 4), dtype=gate_up.weight.dtype, device="cuda")
    other = room[1 : 1 + rows * k].view(rows, k) if how == "odd" else room.view(rows + 1, k + 4)[:rows, :k]
    gate_up.weight = other.copy_(gate_up.weight)
    want, _ = _run(runner, 0, monkeypatch)
    got, ran = _run(runner, 2048, monkeypatch)
    assert not any(ran)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_what_a_noted_layer_kept_is_given_back_before_the_end_of_the_step(dtype, monkeypatch):
    """Behind the last layer no more is allocated than where every layer makes its own launches, and the step's most is
    what the estimate says beyond that."""
    from rapid_llm_amd import EngineConfig, ModelRunner, StepEntry
    from rapid_llm_amd.kernels import ops
    from rapid_llm_amd.models import causal_lm

    body = {**BASE, "hidden_size": 1024, "num_attention_heads": 16, "num_key_value_heads": 8, "head_dim": 128, "intermediate_size": 3072}
    runner = ModelRunner(body, EngineConfig(dtype=dtype, max_seq_len=1024, page_size=16, num_pages=200, max_num_seqs=8),
                         load_format="random")
    norm, at_end = runner.model.final_norm, []
    inner = norm.forward
    monkeypatch.setattr(norm, "forward", lambda *args, **kw: at_end.append(torch.cuda.memory_allocated()) or inner(*args, **kw))
    tokens, most = random_tokens(180, runner.vocab_size, 1), []
    for limit in (0, 2048):
        monkeypatch.setattr(causal_lm, "REPEAT_MAX_TOKENS", limit)
        for _ in range(2):
            torch.cuda.reset_peak_memory_stats()
            runner.step([StepEntry("a", tokens, [179])])
            runner.finish("a")
        most.append(torch.cuda.max_memory_allocated())
    weights = [t for t in runner.model.blocks[0].own_tensors() if t.dim() == 2]
    kept = sum(ops.product_bytes(180, w) for w in weights)
    # (a block may be up to 1 MB larger than what lies in it, and a few are alive at the end)
    assert at_end[3] - at_end[1] <= 4 << 20 < kept / 2
    assert most[1] - most[0] <= 1.5 * kept
