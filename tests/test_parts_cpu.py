"""What parts decide on the host, without a device."""

import pytest
import torch

from rapid_llm_amd.parts.linear import Linear


def _bound(in_features, out_features, dtype):
    linear = Linear(in_features, out_features)
    linear.bind(torch.zeros(out_features, in_features, dtype=dtype))
    return linear


def test_a_product_takes_unscaled_rows_only_if_its_few_row_kernel_runs():
    """A norm leaves its factor to the product behind it only where that product's kernel can
    apply it: bfloat16 weights and a width the kernel's 16-byte reads divide.  A width of 70
    behind an output projection of width 96 once reached the library product with rows that
    nobody had scaled."""
    assert _bound(96, 70, torch.bfloat16).takes_scaled_rows()
    assert not _bound(70, 198, torch.bfloat16).takes_scaled_rows()
    assert not _bound(96, 70, torch.float32).takes_scaled_rows()  # a matrix the checkpoint stores in 32-bit
    assert not Linear(96, 70).takes_scaled_rows()  # nothing bound yet


class _ByteTokenizer:
    """Token id = one byte: a character of several bytes spans tokens."""

    def decode(self, ids, skip_special_tokens=True):
        return bytes(ids).decode("utf-8", errors="replace")


def test_text_is_released_only_with_whole_characters():
    from rapid_llm_amd.engine.tokenizer import Detokenizer

    text = "a é 漢字 ok"
    detok = Detokenizer(_ByteTokenizer())
    pieces = [detok.append(b) for b in text.encode("utf-8")]
    assert "".join(pieces) == text
    assert all("�" not in p for p in pieces)
    assert pieces[2] == "" and pieces[3] == "é"  # the first byte of a two-byte character releases nothing


def test_stop_ids_come_from_generation_config_and_config(tmp_path):
    from rapid_llm_amd.engine.tokenizer import load_stop_token_ids, load_tokenizer

    assert load_stop_token_ids(tmp_path, config_eos=[7]) == {7}
    (tmp_path / "generation_config.json").write_text('{"eos_token_id": [3, 9]}')
    assert load_stop_token_ids(tmp_path, config_eos=[7]) == {3, 7, 9}
    (tmp_path / "generation_config.json").write_text('{"eos_token_id": 4}')
    assert load_stop_token_ids(tmp_path) == {4}
    (tmp_path / "generation_config.json").write_text("{not json")
    assert load_stop_token_ids(tmp_path, config_eos=[1]) == {1}
    assert load_tokenizer(tmp_path) is None  # no tokenizer.json: prompts are token ids


def test_command_line_init_writes_a_model_folder_and_names_a_missing_one(tmp_path, capsys, monkeypatch):
    import json

    import pytest
    from safetensors.torch import load_file

    from rapid_llm_amd.cli import main
    from tiny_configs import TINY_B

    config = tmp_path / "config.json"
    config.write_text(json.dumps(TINY_B))
    for seed in (4, 4, 5):
        assert main(["init", "--config", str(config), "--out", str(tmp_path / f"m{seed}"), "--seed", str(seed),
                     "--dtype", "bfloat16"]) == 0
    a = load_file(str(tmp_path / "m4" / "model.safetensors"))
    assert json.loads((tmp_path / "m4" / "config.json").read_text())["torch_dtype"] == "bfloat16"
    assert a["model.layers.2.mlp.down_proj.weight"].shape == (96, 320)
    assert a["model.embed_tokens.weight"].dtype == __import__("torch").bfloat16
    b = load_file(str(tmp_path / "m5" / "model.safetensors"))
    assert not (a["lm_head.weight"] == b["lm_head.weight"]).all()
    # generation commands name the folder they lack, or take it from the environment
    monkeypatch.delenv("RAPID_LLM_MODEL_DIR", raising=False)
    with pytest.raises(SystemExit, match="Model directory not provided"):
        main(["batch"])
    monkeypatch.setenv("RAPID_LLM_MODEL_DIR", str(tmp_path / "nowhere"))
    with pytest.raises(SystemExit, match="does not exist"):
        main(["batch"])


def test_a_product_with_a_bias_folds_no_norm_into_itself():
    """The residual add and norm that follow a product are folded into its kernel only where
    nothing comes between: a bias is added by a kernel of its own after the product."""
    plain = _bound(128, 128, torch.bfloat16)
    x = torch.zeros(4, 128, dtype=torch.bfloat16)
    assert plain.folds(x) and plain.folds(torch.zeros(40, 128, dtype=torch.bfloat16))
    assert plain.folds(torch.zeros(192, 128, dtype=torch.bfloat16))  # runs of K, in blocks of 64 rows
    assert not plain.folds(torch.zeros(193, 128, dtype=torch.bfloat16))  # the library's product
    biased = Linear(128, 128)
    biased.bind(torch.zeros(128, 128, dtype=torch.bfloat16), torch.zeros(128))
    assert biased.folds(x) and biased.skinny(x)  # the epilogue adds the bias
    import pytest

    with pytest.raises(ValueError, match="bias"):
        Linear(128, 64).bind(torch.zeros(64, 128, dtype=torch.bfloat16), torch.zeros(128))
    with pytest.raises(ValueError, match="bias"):
        Linear(128, 64).bind(torch.zeros(64, 128, dtype=torch.bfloat16), torch.zeros(64, dtype=torch.bfloat16))


def test_a_mixer_may_ask_for_several_state_tensors():
    import pytest

    from rapid_llm_amd.cache.storage import state_bytes
    from rapid_llm_amd.parts import CacheNeed, StateSpec

    one = CacheNeed("state", state_shape=(48,), state_dtype="float32")
    assert [(s.name, s.shape, s.dtype) for s in one.state_specs()] == [("state", (48,), "float32")]
    two = CacheNeed.keys_and_values(2, 16,
                    states=(StateSpec("conv", (3, 48)), StateSpec("count", (1,), "int32")))
    assert [s.name for s in two.state_specs()] == ["conv", "count"]
    assert CacheNeed.keys_and_values(1, 16).state_specs() == ()
    # five slots: 48 float32 each; 3 x 48 in the engine's type (2 bytes) and one int32 each
    assert state_bytes([one, two], 5, 2) == 5 * 48 * 4 + 5 * (3 * 48 * 2 + 4)
    with pytest.raises(ValueError, match="alike"):
        CacheNeed("state", state_shape=(4,), states=(StateSpec("state", (2,)),)).state_specs()


def test_the_ends_of_a_model_are_parts_named_in_its_description():
    from rapid_llm_amd.models import linear_output, token_embedding
    from rapid_llm_amd.parts import EMBEDDINGS, OUTPUT_PROJECTIONS

    assert "token_embedding" in EMBEDDINGS.kinds() and "linear_output" in OUTPUT_PROJECTIONS.kinds()
    emb = token_embedding(100, 16, "model.embed_tokens.weight")
    part = EMBEDDINGS.create(emb.kind, **emb.params, name="embed")
    assert [(s.name, s.shape) for s in part.param_specs()] == [("embed.weight", (100, 16))]
    tied = linear_output(100, 16, "lm_head.weight", True)
    out = OUTPUT_PROJECTIONS.create(tied.kind, **tied.params, name="output")
    assert out.param_specs()[0].fallback == "embed.weight"
    assert OUTPUT_PROJECTIONS.create("linear_output", **linear_output(100, 16, "h", False).params, name="output").param_specs()[0].fallback is None


def test_prefill_launch_shapes_follow_an_estimate_of_the_launch():
    """Two wave groups on a tile where the longest tile would outlast everyone else's work (a
    prompt from its start), one where there is work for every slot, key runs for few, long tiles
    and only where they save more than their merge costs.  The choice is the host's alone."""
    from types import SimpleNamespace

    from rapid_llm_amd.kernels import ops

    def shape(seqs, nkv=8, group=4, window=0, rows=128):
        keys = []
        for start, n in seqs:
            for row0 in range(0, n * group, rows):
                keys.append(start + min(n, (row0 + rows) // group))
        return ops._prefill_shape(SimpleNamespace(tile_keys=keys, num_tiles=len(keys)), nkv, window, rows)

    assert shape([(0, 2048)]) == (2, 1) and shape([(0, 1024)]) == (2, 1) and shape([(0, 512)]) == (2, 1)
    assert shape([(0, 8192)]) == (1, 1) and shape([(0, 4096)]) == (1, 1) and shape([(2048, 2048)]) == (1, 1)
    assert shape([(3584, 512)]) == (1, 4) and shape([(7680, 512)]) == (1, 4) and shape([(16000, 150)]) == (1, 8)
    assert shape([(0, 2048)] * 4) == (1, 1) and shape([(0, 20)]) == (1, 1)
    # a window bounds what every tile reads: the long prefix no longer counts
    assert shape([(16000, 150)], window=256) == (2, 1)


@pytest.mark.parametrize("d,groups", [(64, 2), (128, 2), (160, 2), (192, 1), (224, 1), (256, 1)])
def test_prefill_launch_shapes_of_large_heads(d, groups):
    """Two wave groups of large heads keep their state in scratch: one prompt goes to one wave group a tile."""
    from types import SimpleNamespace

    from rapid_llm_amd.kernels import ops

    for n, nkv, group in ((2048, 8, 4), (1024, 8, 4), (300, 8, 4), (600, 16, 1)):
        keys = [min(n, (row0 + 128) // group) for row0 in range(0, n * group, 128)]
        assert ops._prefill_shape(SimpleNamespace(tile_keys=keys, num_tiles=len(keys)), nkv, 0, 128, 256, d=d) == (groups, 1)


def test_prefill_launch_shapes_of_short_tiles_and_of_last_rounds():
    """As many tiles of one step as there are units: one wave group each.  Tiles for one round and a part of the next are
    not cut into runs that leave most of a last round without work."""
    from types import SimpleNamespace

    from rapid_llm_amd.kernels import ops

    def shape(seqs, nkv, group, d):
        keys = [start + min(n, (row0 + 128) // group) for start, n in seqs for row0 in range(0, n * group, 128)]
        return ops._prefill_shape(SimpleNamespace(tile_keys=keys, num_tiles=len(keys)), nkv, 0, 128, 256, d=d)

    assert shape([(0, 8)] * 16, 16, 4, 160) == (1, 1) and shape([(0, 13)] * 16, 16, 1, 128) == (1, 1)
    lengths = (730, 604, 791, 988, 1082, 706, 766, 912)
    assert shape([(6019, n) for n in lengths], 8, 1, 80) == (1, 1)
    assert shape([(0, 10752)], 4, 1, 128) == (1, 2)  # (the longest tiles are many times the others)


def test_layers_of_unlike_heads_have_launch_shapes_of_their_own():
    """One step's plan serves every layer with its groups: heads of two sizes, whichever layer comes first."""
    from types import SimpleNamespace

    from rapid_llm_amd.kernels import ops

    lib = SimpleNamespace(rl_attn_prefill_rows=lambda: 128)
    for first, second in ((64, 256), (256, 64)):
        plan = ops.AttentionPlan.__new__(ops.AttentionPlan)
        plan.shapes, plan.tile_keys, plan.num_tiles = {}, [min(2048, row0 // 4 + 32) for row0 in range(0, 8192, 128)], 64
        for d in (first, second, first):
            assert plan.prefill_shape(8, 0, lib, d) == ops._prefill_shape(plan, 8, 0, 128, d=d) == ((2, 1) if d == 64 else (1, 1))


def test_which_products_run_in_one_launch_of_this_package():
    """The host's rule for the tile product (17 to 512 rows over a matrix of a few megabytes with
    enough result columns for every compute unit): the smallest model's QKV and gate/up products
    take it, its narrow products, larger models' matrices and steps of few or many rows do not."""
    from rapid_llm_amd.kernels import ops

    assert ops._tile_applies(64, 4096, 1024, 4096)        # Qwen3-0.6B QKV
    assert ops._tile_applies(256, 6144, 1024, 3072)       # its packed gate and up rows, 3,072 results
    assert ops._tile_applies(512, 4096, 1024, 4096)
    assert not ops._tile_applies(16, 4096, 1024, 4096)    # the few-row kernel's
    assert not ops._tile_applies(513, 4096, 1024, 4096)   # the library's
    assert not ops._tile_applies(64, 1024, 2048, 1024)    # output projection: 16 workgroups a row block
    assert not ops._tile_applies(64, 4096, 2048, 4096)    # 16 MB: the library is as fast
    assert not ops._tile_applies(64, 6144, 4096, 6144)    # Qwen3-8B QKV
    assert not ops._tile_applies(64, 4096, 1000, 4096)    # K in chunks of 128 only
    assert not ops._tile_applies(64, 4098, 1024, 4098)    # four result columns a lane


def test_where_the_many_row_product_applies():
    """The rule of the many-row product on the chip it was measured on: what it takes, the tiles at both ends
    of its range, runs of K that all hold a chunk, and what stays where it was."""
    from rapid_llm_amd.kernels import ops

    plan = lambda *a: ops.block_plan(*a, units=256)
    assert plan(512, 12288, 4096, "gated") == (3, 4, 1)    # 256 tiles of 192 x 256: one a compute unit
    assert plan(2048, 12288, 4096, "gated") == (4, 4, 1)
    assert plan(160, 3072, 1024, "gated") == (2, 2, 1)     # few rows: as many workgroups as there can be
    assert plan(64, 12288, 4096, "gated") is None          # the kernel for up to 64 rows
    # tiles for too few units, each of which would walk a long K alone
    assert plan(65, 2048, 5120, "gated") is None and plan(128, 5120, 2048, "gated") is None and plan(96, 6144, 4096, "gated") is None
    assert plan(128, 6144, 2048, "gated") and plan(129, 6144, 2048, "gated") and plan(65, 9728, 2560, "gated") and plan(65, 12288, 4096, "gated") and plan(65, 4096, 512, "gated")
    for units in (64, 128, 304):  # (as a share of the units that there are)
        for tiles in range(1, units + 1):
            assert (ops.block_plan(65, 64 * tiles, 2048, "gated", units=units) is None) == (8 * tiles < 3 * units)
            assert (ops.block_plan(65, 64 * tiles, 4096, "gated", units=units) is None) == (4 * tiles < 3 * units)
    assert plan(512, 12288, 4100, "gated") is None and plan(512, 12290, 4096, "gated") is None
    assert plan(90000, 12288, 12288, "gated") is None      # offsets beyond 31 bits
    assert plan(2048, 4096, 4096, "runs") is None          # short sums: the library's
    assert plan(2049, 4096, 12288, "runs") is None and plan(2048, 4096, 12288, "runs") == (4, 4, 2)
    assert plan(128, 2048, 6144, "runs") is None and plan(129, 2048, 6144, "runs") is not None
    assert plan(1025, 2048, 6144, "runs") is None
    few = lambda *a: ops.block_few_plan(*a, units=256)
    assert few(49, 12288, 4096) == few(64, 6144, 2048) == (2, 1, 1)
    assert few(48, 12288, 4096) is None and few(65, 12288, 4096) is None and few(64, 3072, 1024) is None
    assert few(64, 9728, 2560) is None and few(49, 8192, 4096) is None and few(64, 7168, 2048) is None and few(64, 12288, 5120) is None
    assert few(64, 11008, 4096) and few(49, 14336, 5120) and few(64, 16384, 8192) and few(64, 6152, 2048)
    assert few(64, 17408, 5120) is None and few(64, 6148, 2048) is None and few(64, 12288, 4100) is None
    for m in (65, 100, 300, 777, 1024):
        for n, k in ((4096, 12288), (2560, 9728), (2048, 6144), (8, 8192)):
            found = plan(m, n, k, "runs")
            if found is None:
                assert k < 8192
                continue
            per = -(-(k // 64) // found[2])
            assert per * (found[2] - 1) < k // 64


def test_products_over_long_sums_leave_the_others_for_a_filled_chip():
    """What a layer asks for, as against what the many-row product can do: it is to be the faster one."""
    from rapid_llm_amd.kernels import ops

    pays = lambda *a: ops.block_pays(*a, 256)
    # the mid-size product's range and the library's
    assert pays(65, 4096, 12288) and pays(128, 2560, 9728) and pays(160, 1536, 9728) and pays(384, 512, 12288)
    assert not pays(65, 512, 12288) and not pays(192, 1024, 12288) and not pays(128, 1536, 9728) and not pays(224, 512, 12288)
    assert pays(2048, 4096, 12288) and pays(1280, 2048, 8192) and not pays(1281, 2048, 8192) and not pays(300, 4096, 4096)
    for units in (64, 256, 304):
        for m in (65, 192, 193, 700, 2000):
            for n in (8, 512, 2056, 4096):
                for k in (6144, 8192, 12288):
                    if ops.block_pays(m, n, k, units):
                        plan = ops.block_plan(m, n, k, "runs", units=units)
                        assert 8 * plan[2] * ops._block_tiles(m, n, "runs", plan) >= 3 * units


def test_small_gate_and_up_matrices_leave_the_tile_product_for_a_filled_chip():
    from rapid_llm_amd.kernels import ops

    goes = lambda *a: ops._tile_gives_way(*a, 256)
    assert goes(129, 3072, 1024) and goes(512, 2048, 1024) and goes(400, 1536, 512)
    assert not goes(128, 3072, 1024) and not goes(256, 2048, 1024) and not goes(512, 1024, 1024) and not goes(129, 1536, 1024)
    for inter in range(512, 3585, 64):
        for m in (129, 200, 300, 512):
            plan = ops.block_plan(m, inter, 1024, "gated", units=256)
            assert goes(m, inter, 1024) == (8 * ops._block_tiles(m, inter, "gated", plan) >= 3 * 256)


def test_launch_rules_follow_the_number_of_compute_units():
    """Every launch rule takes the chip's geometry from one place on the host
    (``ops.chip()``; without a device the chip the rules were measured on), so that a part
    with another number of compute units gets shapes for itself: decode attention asks for the
    requests' order by length only beyond three workgroups a unit, and the few-row product's
    rows a workgroup and the runs of K of the mid-size product move with the unit count."""
    from types import SimpleNamespace

    from rapid_llm_amd.kernels import ops

    assert ops.chip().units == 256 and ops.chip().decode_resident == 3 * 256
    assert ops.Chip(304).first_round == 304 and ops.Chip(304).prefill_slots == 608
    # 384 tiles of 16 rows: one round of 24 rows on 256 units, nothing to gain on 384 units
    assert ops._skinny_tiles(8, 6144, plain=True, units=256) == 3
    assert ops._skinny_tiles(8, 6144, plain=True, units=384) == 1
    # 64 blocks of 64 rows: four runs of K fill 256 units, one run fills 64
    assert ops.mid_runs(4096, 4096, units=256) == 4 and ops.mid_runs(4096, 4096, units=64) == 1
    # a portion behind a long prefix is cut into key runs only while the launch leaves slots free
    tile = SimpleNamespace(tile_keys=[4096] * 4, num_tiles=4)
    assert ops._prefill_shape(tile, 8, 0, 128, units=256)[1] > 1
    assert ops._prefill_shape(tile, 8, 0, 128, units=8) == (1, 1)


def test_which_contexts_are_unlike_enough():
    """The rule asks for what a launch's workgroups make of the lengths: never where there are few of them, more than
    512 keys where they fill the chip evenly, and no launch that the chip takes in more than two rounds."""
    from rapid_llm_amd.kernels import ops

    def unlike(n, length, longer, count=1, each=8):
        return ops.ragged_contexts([length] * (n - count) + [longer] * count, each, 256)

    # few workgroups, whose keys are cut fine anyway: one and two kv heads
    assert not unlike(8, 4000, 8000, each=1) and not unlike(16, 4000, 8000, each=2) and not unlike(63, 100, 4000, each=1)
    assert unlike(200, 100, 4000, each=1) and unlike(100, 100, 4000, each=2) and not unlike(300, 100, 4000, each=2)
    assert not unlike(8, 1000, 2000) and unlike(8, 4000, 8000)
    # a chip filled by one round (24, 32) or two (64), and one that is not (17, 40, 48)
    assert unlike(24, 4000, 5000) and not unlike(24, 4000, 5000, 6) and not unlike(32, 4000, 5000, 8)
    assert unlike(32, 4000, 8000) and not unlike(64, 4000, 5000) and unlike(64, 4000, 8000)
    assert unlike(17, 4000, 5000, 4) and unlike(40, 4000, 5000, 10) and unlike(48, 4000, 5000, 12)
    for rows in range(1, 300):
        for each in (1, 2, 8, 16):
            pairs = rows * each
            assert ops.ragged_pairs(pairs, 256) == (64 <= pairs <= 512)
            if not ops.ragged_pairs(pairs, 256):
                assert not ops.ragged_contexts([1] * (rows - 1) + [100000], each, 256)


def test_spans_of_the_float32_attention():
    """When a float32 launch splits its keys, at the rule's edges, and that what is reserved for a recorded step of
    single tokens is what the launch takes."""
    from rapid_llm_amd.kernels import ops

    spans = lambda tiles, longest, window=0, held=16: ops.f32_spans(tiles, 8, 128, longest, window, held, 256)
    assert spans(1, 512) == 0 and spans(1, 513) == 3 and spans(31, 4096) == 16 and spans(32, 4096) == 0
    assert spans(1, 4096, 1023) == 0 and spans(1, 4096, 1024) == 16
    # the states of a decoding request's tile have its query heads alone: four, and two, where a full tile has 16
    assert spans(16, 8192) == 32 and spans(16, 16384) == 0
    assert spans(16, 16384, held=4) == 64 and spans(16, 24576, held=4) == 96 and spans(16, 65536, held=4) == 0
    assert spans(16, 32768, held=2) == 128
    for nq, nkv in ((32, 8), (16, 8), (8, 8), (40, 2)):
        group = nq // nkv
        for rows in (1, 8, 16):
            for longest in (512, 4096, 40000):
                tiles, held = rows * -(-group // 16), min(16, group)
                n = ops.f32_spans(tiles, nkv, 128, longest, 0, held)
                assert ops.f32_states_bytes(rows, nq, nkv, 128, longest, 0) == tiles * nkv * n * 4 * -(-held * 130 // 32) * 128


@pytest.mark.parametrize("units", [40, 64, 128, 256, 304])
def test_a_product_left_in_float32_is_one_run_of_k(units, monkeypatch):
    """What enters a recurrence in 32 bits is a whole sum, whatever the rule for products that a norm adds cuts K into."""
    from types import SimpleNamespace

    from rapid_llm_amd.kernels import ops

    asked = []

    class Library:
        def __getattr__(self, name):
            return lambda *args: asked.append((name, args)) or 0

    monkeypatch.setattr(ops, "chip", lambda: SimpleNamespace(units=units))
    monkeypatch.setattr(ops, "core", Library)
    monkeypatch.setattr(ops, "_stream", lambda: None)
    monkeypatch.setattr(ops, "_need", lambda *args: None)
    cut = 0
    for m, n, k in ((129, 4160, 6144), (129, 2112, 6144), (65, 1088, 8192), (192, 8192, 9728), (100, 512, 512)):
        x, w = (torch.empty((rows, k), dtype=torch.bfloat16, device="meta") for rows in (m, n))
        w.data_ptr = x.data_ptr = lambda: 0
        if ops.mid_runs(n, k) != 1:
            continue
        found = ops.block_plan(m, n, k, "runs")
        cut += found is not None and found[2] > 1
        monkeypatch.setattr(ops, "_p", lambda t: t)
        got = ops.gemm_bf16_wide(x, w)
        assert got.shape == (m, n) and got.dtype == torch.float32
        name, args = asked.pop()
        assert name == "rl_gemm_mid_parts" and args[8] == 1 and not asked
    assert cut > 0 or units >= 256  # (there the two rules meet nowhere)


def test_plans_of_the_float32_product():
    """Every plan is one that the kernel's entry takes, on chips of any number of compute units: streamed weights
    without sharing and within the grid, shared runs within the scratch that is reserved for them."""
    from rapid_llm_amd.kernels import ops

    for units in (1, 7, 40, 228, 256, 304):
        for m in (1, 4, 5, 16, 17, 32, 33, 64, 65, 225, 2048, 65535, 65536, 70000):
            for n in (1, 15, 16, 333, 1024, 4608, 6144, 8193, 24576, 151936):
                for k in (1, 31, 32, 256, 257, 512, 1000, 1024, 2048, 4096, 12288):
                    tile, groups = ops.f32_plan(m, n, k, units)
                    if tile in (1, 2, 3):
                        assert groups == 1 and (m <= 32 or k <= 256) and -(-m // 16) <= 65535
                    else:
                        assert m > 16 and tile in ((32,) if m <= 32 else (64,) if m <= 64 else (64, 128)) and groups in (1, 2, 4, 8)
                    if groups > 1:
                        assert 32 * m * n <= ops._F32_MOST_SCRATCH and m <= 65535
    assert ops.f32_scratch_bytes(40, 4096, 4096) == 32 * 40 * 4096 and ops.f32_scratch_bytes(2048, 24576, 4096) == 0
    # rows that are a multiple of 8 KB apart, on either side of what makes one round of two
    assert [ops.f32_plan(1, 6144, k, 256)[0] for k in (1024, 2048, 2560, 4064, 4096, 5120)] == [2, 1, 2, 2, 1, 2]
    assert ops.f32_plan(8, 8192, 4096, 256)[0] == 1 and ops.f32_plan(9, 8192, 4096, 256)[0] == 2


def test_plans_of_the_float32_product_for_many_rows():
    """Large tiles only for whole chunks and more than 64 rows, where they fill the chip; launches hold whole tiles and
    what they take is what is reserved."""
    from rapid_llm_amd.kernels import ops

    for units in (1, 40, 256, 304):
        for m in (1, 64, 65, 225, 2048, 8192, 70000):
            for n in (1, 333, 4096, 24576):
                for k in (32, 1000, 1024, 4096, 12288):
                    cols = ops.f32_wide(m, n, k, units)
                    assert cols in (0, 96, 128) and (not cols or (m > 64 and k % 32 == 0))
                    rows = ops._f32_piece_rows(m, k)
                    assert rows % 256 == 0 and 96 * k * (rows // 16 - 16) <= ops._F32_MOST_PIECES
    assert ops.f32_wide(2048, 24576, 4096, 256) == 128 and ops.f32_wide(2048, 6144, 4096, 256) == 96
    # short sums, and sizes at which the two are level
    assert ops.f32_wide(1982, 3120, 256, 256) == 0 and ops.f32_wide(269, 12032, 512, 256) == 0 and ops.f32_wide(247, 12784, 3296, 256) == 0
    assert ops.f32_wide(2048, 1024, 3072, 256) == 0 and ops.f32_wide(225, 4096, 1024, 256) == 0
    assert ops._f32_piece_rows(2048, 12288) == 2048 and ops._f32_piece_rows(8192, 12288) == 2816


def test_decode_splits_of_unlike_contexts():
    """Requests of unlike length get more splits of their keys, whatever that would be for fewer than eight
    and more than 64, and never splits that hold no whole step; the bytes reserved cover both."""
    from rapid_llm_amd.kernels import ops

    assert ops.ragged_contexts([64] * 7 + [4000]) and not ops.ragged_contexts([64] * 6 + [4000])
    assert not ops.ragged_contexts([2000, 2400] * 6) and not ops.ragged_contexts([64] * 64 + [4000])
    assert not ops.ragged_contexts([])
    for rows in (8, 12, 16, 17, 24, 32, 64):
        for span in (512, 1024, 4096, 40000):
            pairs, chunk, like = ops._decode_split(rows, 32, 8, span, 16, 0, units=256)
            _, fine, unlike = ops._decode_split(rows, 32, 8, span, 16, 0, units=256, ragged=True)
            assert unlike >= like and fine <= chunk and fine % 32 == 0 and fine * unlike >= span
            assert unlike == 1 or fine >= 128
            assert ops.decode_scratch_bytes(rows, 32, 8, 128, span, 16, 0) >= (0 if unlike == 1 else rows * 32 * unlike * 130 * 4)


def test_decode_splits_of_few_short_contexts():
    """Half-sized splits only where units would be idle and contexts are short; they cover the span, and the bytes
    reserved cover them."""
    from rapid_llm_amd.kernels import ops

    for rows in (1, 2, 4, 5, 8, 32):
        for span in (1, 64, 65, 128, 300, 512, 513, 4096):
            for window in (0, 100):
                pairs, chunk, nsplit = ops._decode_split(rows, 32, 8, span, 16, window, units=256)
                short = ops._decode_short(pairs, chunk, span, window, units=256)
                assert short is None or (short[0] == 64 and span <= 512 or window)
                if short is not None:
                    seen = min(span, window + 31) if window else span
                    assert short[0] * short[1] >= seen and short[0] % 64 == 0 and short[0] < chunk
                    assert pairs * short[1] <= 256 or pairs >= 256
                    assert ops.decode_scratch_bytes(rows, 32, 8, 128, span, 16, window) >= (short[1] > 1) * rows * 32 * short[1] * 130 * 4
    assert ops._decode_short(8, 128, 300, 0, units=256) == (64, 5) and ops._decode_short(256, 128, 100, 0, units=256) is None


def test_weight_rows_a_workgroup_of_the_few_row_product():
    """The host's rule: 24 rows (code 3) only for a product that just stores its result, on a
    matrix of 257 to 1,023 tiles, where that puts the fewest rows on a compute unit."""
    from rapid_llm_amd.kernels import ops

    assert ops._skinny_tiles(8, 6144, plain=True) == 3      # 384 tiles: 256 workgroups of 24 rows
    assert ops._skinny_tiles(1, 5120, plain=True) == 3      # 320 tiles: 214 workgroups
    assert ops._skinny_tiles(8, 7168, plain=True) == 2      # 448 tiles: 24 rows would need a second round
    assert ops._skinny_tiles(8, 6144) == 2                  # the residual epilogue keeps whole tiles
    assert ops._skinny_tiles(8, 4096, plain=True) == 1      # one tile a unit already
    assert ops._skinny_tiles(16, 151936, plain=True) == 2   # a thousand tiles and more: as measured
    assert ops._skinny_tiles(8, 151936, plain=True) == 1


def test_tiles_a_workgroup_of_the_product_for_tens_of_rows():
    """The host's rule for the product of 17 to 64 rows over wide matrices: a compute unit gets
    one workgroup with an even share of the tiles where a workgroup can hold such a share, and a
    matrix with more tiles is cut into workgroups of the most tiles one holds."""
    from rapid_llm_amd.kernels import ops

    plan = lambda m, n, k, sw: ops.rows_plan(m, n, k, sw, units=256)
    assert plan(64, 12288, 4096, True) == (3, 256)     # Qwen3-8B gate/up: 768 pairs, three a unit
    assert plan(32, 6144, 4096, False) == (2, 256)     # its QKV: 384 tiles, one or two a unit
    assert plan(64, 151936, 4096, False) == (6, 1583)  # the vocabulary: 9,496 tiles in groups of six
    assert plan(48, 25600, 5120, True) is None         # the 32B shape's gate/up, 1,600 pairs: the library's,
    assert plan(48, 51200, 5120, False) is None        # with the activation or without
    assert plan(33, 17408, 5120, True) == (5, 256) and plan(33, 10240, 5120, False) == (3, 256)
    assert plan(64, 17408, 5120, True) == (3, 363)     # at 64 rows a workgroup holds three pairs at most
    assert plan(33, 4096, 2048, False) == (1, 256) and plan(33, 2048, 2048, False) == (1, 128)
    assert plan(33, 12288, 4096, True) == (3, 256) and ops.rows_plan(33, 12288, 4096, True, units=304) == (3, 304)
    assert plan(16, 12288, 4096, True) is None and plan(65, 12288, 4096, True) is None
    assert plan(33, 12296, 4096, True) is None and plan(33, 12288, 4160, True) is None


@pytest.mark.parametrize("change", ["none", "derived", "replaced", "biased"])
def test_a_float32_feed_forward_asks_its_gate_and_up_product(change, monkeypatch):
    """Product and activation are one launch only where the product is nothing but its weight: a derived product, one with
    a call of its own and one with a bias are asked."""
    from rapid_llm_amd.kernels import ops
    from rapid_llm_amd.parts.mlp import SwiGLU

    ff = SwiGLU(4, 6, "mlp.")
    ff.down.deferred = lambda act, ctx: act
    gate_up, called = torch.randn(12, 4), []

    class Doubled(Linear):
        def product(self, x, out_dtype=None):
            called.append("derived")
            return 2 * (x @ self.weight.T)

    if change == "derived":
        ff.gate_up = Doubled(4, 12)
    ff.gate_up.bind(gate_up, torch.ones(12) if change == "biased" else None)
    if change == "replaced":
        ff.gate_up.product = lambda x, out_dtype=None: called.append("replaced") or 2 * (x @ gate_up.T)

    def swiglu(gu, act, *args, **kwargs):
        act.copy_(torch.nn.functional.silu(gu[:, :6]) * gu[:, 6:])

    monkeypatch.setattr(ops, "swiglu", swiglu)
    monkeypatch.setattr(ops, "gemm_f32", lambda x, w, out: out.copy_(x @ w.T))
    monkeypatch.setattr(ops, "add_bias", lambda y, bias: y.add_(bias))
    monkeypatch.setattr(ops, "gemm_f32_swiglu", lambda x, w: called.append("one launch") or torch.zeros(x.shape[0], 6))
    x = torch.randn(3, 4)
    got = ff.forward(x, None)
    if change == "none":
        assert called == ["one launch"]
        return
    gu = x @ gate_up.T + 1.0 if change == "biased" else 2 * (x @ gate_up.T)
    assert called == ([] if change == "biased" else [change])
    torch.testing.assert_close(got, torch.nn.functional.silu(gu[:, :6]) * gu[:, 6:])
