"""Where the many-row product stored as bfloat16 runs, and that a layer's answer to "is this the library's?" is what it does."""

import random
import threading

from types import SimpleNamespace

import pytest
import torch

from rapid_llm_amd.config.qwen3 import Qwen3Config
from rapid_llm_amd.kernels import ops
from rapid_llm_amd.models.causal_lm import CausalLM
from rapid_llm_amd.models.qwen3 import build_qwen3_spec


@pytest.mark.parametrize("units", [64, 256, 304])
def test_plans_are_what_the_kernel_takes(units):
    rng = random.Random(units)
    for _ in range(3000):
        m, n, k = rng.randint(1, 9000), 8 * rng.randint(1, 1600), 64 * rng.randint(1, 200)
        plan = ops.block_plain_plan(m, n, k, units)
        if plan is None:
            continue
        assert m > ops.ROWS_MAX_ROWS and plan[:2] in ops._BLOCK_TILES and plan[2] == 1
        tiles = ops._block_tiles(m, n, "plain", plan)
        assert 2 * tiles >= units  # half of the chip at least
        assert (m + 256) * k * 2 <= 0x7FFFFFFF and (n + 256) * k * 2 <= 0x7FFFFFFF
    assert ops.block_plain_plan(2048, 6140, 4096, units) is None and ops.block_plain_plan(2048, 6144, 4100, units) is None


def test_two_rounds_of_large_tiles_that_three_quarters_of_the_units_have():
    """Measured inside prompt steps: the library's products are the faster ones there, level or slower on both sides."""
    for n, k in ((4096, 2048), (4096, 4096), (4096, 12288)):
        for m in (5889, 6000, 6144):
            assert ops._block_plan(m, n, k, "plain", 256)[:2] == (4, 4) and ops.block_plain_plan(m, n, k, 256) is None
            assert ops.library_takes(m, n, k)
        assert ops.block_plain_plan(6145, n, k, 256) is not None and ops.block_plain_plan(5500, n, k, 256) is not None
    assert ops.block_plain_plan(6000, 2048, 2048, 256) is not None  # (one round)


def test_small_models_library_products():
    layers = {"0.6b": ((4096, 1024), (1024, 2048), (1024, 3072)), "1.7b": ((4096, 2048), (2048, 2048), (2048, 6144))}

    def library(m, n, k, folded):
        if folded and ((m <= ops.mid_max_rows(n, k) and ops.mid_runs(n, k, 256) > 0) or ops.block_pays(m, n, k, 256)):
            return False
        return ops.library_takes(m, n, k)

    with ops.own_products():
        for m in range(17, 1274):
            assert not any(library(m, n, k, i > 0) for i, (n, k) in enumerate(layers["0.6b"])), m
        for m in range(17, 321):
            assert not any(library(m, n, k, i > 0) for i, (n, k) in enumerate(layers["1.7b"])), m
    assert library(512, 6144, 2560, False) and not library(2048, 6144, 4096, False)
    # the choice is a thread's own and ends with the block
    assert library(300, *layers["0.6b"][1], True)
    seen = []
    with ops.own_products():
        thread = threading.Thread(target=lambda: seen.append(library(300, *layers["0.6b"][1], True)))
        thread.start()
        thread.join()
    assert seen == [True]


def test_a_step_keeps_to_own_products_only_if_every_layer_can():
    """A later layer of another kind may need the library's product, or make more than its matrices' launches: the step
    then waits for the host anyway, and every product is the one that is faster on the device."""
    body = dict(
        architectures=["Qwen3ForCausalLM"], model_type="qwen3", num_hidden_layers=4, hidden_size=1024, num_attention_heads=16,
        num_key_value_heads=8, head_dim=128, intermediate_size=3072, vocab_size=97, rope_theta=10000.0, rms_norm_eps=1e-6,
        tie_word_embeddings=True, max_position_embeddings=128, hidden_act="silu", attention_bias=False,
    )
    runtime = SimpleNamespace(device=torch.device("meta"), dtype=torch.bfloat16, max_seq_len=128, page_size=16)

    def model(change=None):
        m = CausalLM(build_qwen3_spec(Qwen3Config.from_dict(body)))
        if change is not None:
            change(m.blocks[2])
        params = {s.name: torch.empty(s.shape, dtype=torch.float32 if s.role == "vector" else torch.bfloat16, device="meta") for s in m.param_specs()}
        m._positions.clear()  # (their tables are made on the device)
        m.bind(params, runtime)
        return m

    def own(m, tokens):
        return m._own_products(SimpleNamespace(num_tokens=tokens))

    plain = model()
    assert len(plain._kinds) == 1 and own(plain, 300) and not own(plain, 16) and not own(plain, 4000)

    def wide(block):  # an intermediate size that the library's product is needed for
        ff = type(block.feed_forward)(1024, 20000, "model.layers.2.mlp.", name="layers.2.ff")
        block.feed_forward = ff

    def hooked(block):
        block.mixer.forward = block.mixer.forward

    mixed = model(wide)
    assert len(mixed._kinds) == 2
    assert any(b.calls_library(300) for b in mixed._kinds) and not own(mixed, 300)
    assert not own(model(hooked), 300)
