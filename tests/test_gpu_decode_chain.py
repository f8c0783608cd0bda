"""All layers of a recorded step of few tokens in one launch: as close to the plain implementation as any other way of
running the step, at the edges of its sizes, with any number of workgroups, and beside another launch of its kind."""

import threading

import pytest
import torch

import parity
from plain_model import plain_forward, plain_load
from tiny_configs import random_tokens

pytestmark = pytest.mark.gpu

BASE = dict(
    architectures=["Qwen3ForCausalLM"], model_type="qwen3", num_hidden_layers=3, hidden_size=256, num_attention_heads=4,
    num_key_value_heads=2, head_dim=128, intermediate_size=384, vocab_size=277, rope_theta=30000.0, rms_norm_eps=1e-5,
    tie_word_embeddings=False, max_position_embeddings=2048, hidden_act="silu", attention_bias=False,
)
# contractions of 1 chunk of 128 (waves without one), of 9 (more for one wave) and of 33 (more than the ring holds; gate and
# up in pairs), one to four query heads a kv head, one kv head, fewer items than workgroups
SHAPES = {
    "small": dict(hidden_size=128, intermediate_size=128, num_attention_heads=1, num_key_value_heads=1, num_hidden_layers=2),
    "base": {},
    "uneven": dict(hidden_size=1152, intermediate_size=1408, num_attention_heads=9, num_key_value_heads=3),
    "long": dict(hidden_size=4224, intermediate_size=640, num_attention_heads=4, num_key_value_heads=1, num_hidden_layers=2),
}
# tokens in the cache in front of the step: none, one; the ends of eights, pages, the waves' 32 and 256 keys, a share, two and more
CONTEXTS = [300, 1, 255, 256, 512, 513, 0, 31, 7, 16, 1100, 8, 64, 511, 767, 33]


def _runner(model, **engine):
    from rapid_llm_amd import EngineConfig, ModelRunner

    engine = EngineConfig(**{**dict(dtype="bfloat16", max_seq_len=2048, page_size=16, num_pages=420, max_num_seqs=16), **engine})
    return ModelRunner(model, engine, **({} if isinstance(model, str) else dict(load_format="random", weight_norm_std=0.1)))


def _fill(runner, contexts, vocab):
    """Requests with so many tokens in the cache, and the step that decodes one token of each."""
    from rapid_llm_amd import StepEntry

    tokens = {f"r{i}": random_tokens(n + 1, vocab, 31 + i) for i, n in enumerate(contexts)}
    for rid, ids in tokens.items():
        if len(ids) > 1:
            runner.step([StepEntry(rid, ids[:-1])])
    return tokens, [StepEntry(rid, ids[-1:], [0]) for rid, ids in tokens.items()]


def _again(runner, tokens, entries):
    logits = runner.step(entries).clone()
    for rid, ids in tokens.items():
        if len(ids) > 1:
            runner.computed[rid] = len(ids) - 1
        else:
            runner.finish(rid)
    return logits


def _chains(runner):
    return [e[3].static.get("decode_chain") for kinds in runner._graphs.values() for e in kinds.values()]


@pytest.mark.parametrize("page", [8, 24])
@pytest.mark.parametrize("which", list(SHAPES))
def test_step_is_the_plain_implementations(tmp_path, which, page):
    from rapid_llm_amd import write_random_model

    cfg = {**BASE, **SHAPES[which]}
    folder = str(write_random_model(cfg, 5, tmp_path / which, dtype="bfloat16"))
    config, weights = plain_load(folder)
    got, want = [], []
    for rows in (1, 2, 3, 5, 8, 16):
        runner = _runner(folder, page_size=page, num_pages=800)
        tokens, entries = _fill(runner, CONTEXTS[:rows], cfg["vocab_size"])
        got.append(_again(runner, tokens, entries).cpu())
        assert all(c is not None for c in _chains(runner)) and len(_chains(runner)) == 1
        # again, on the same and on other pages' contents: the same bits
        assert torch.equal(_again(runner, tokens, entries).cpu(), got[-1])
        want.append(torch.stack([plain_forward(config, weights, ids)[-1] for ids in tokens.values()]))
    parity.assert_bf16_close(torch.cat(got), torch.cat(want), f"decode chain/{which}/{page}")


@pytest.mark.parametrize("rows", [1, 2, 4, 16])
def test_any_number_of_workgroups_gives_the_same(rows, monkeypatch):
    from rapid_llm_amd.kernels import decode_chain, ops

    cfg = {**BASE, "hidden_size": 1024, "num_attention_heads": 8, "intermediate_size": 1536}
    results = []
    for units in (None, 1, 3, 50, 255):
        runner = _runner(cfg)
        tokens, entries = _fill(runner, CONTEXTS[:rows], cfg["vocab_size"])
        with monkeypatch.context() as m:
            if units is not None:
                # as many shares of the keys as ever, dealt to fewer workgroups: some have several of one request
                real = decode_chain.DecodeChain.run

                def run(self, *args, units=units, real=real):
                    with pytest.MonkeyPatch.context() as inner:
                        inner.setattr(decode_chain, "chip", lambda: ops.Chip(units))
                        return real(self, *args)

                m.setattr(decode_chain.DecodeChain, "run", run)
            results.append(_again(runner, tokens, entries))
        assert _chains(runner)[0] is not None
        torch.cuda.synchronize()
    for r in results[1:]:
        assert torch.equal(r, results[0])


def _launched_with(units):
    """A step's recorded launch has so many workgroups, and as many shares of the keys as ever."""
    from rapid_llm_amd.kernels import decode_chain, ops

    real, m = decode_chain.DecodeChain.run, pytest.MonkeyPatch()

    def run(self, *args):
        with pytest.MonkeyPatch.context() as inner:
            inner.setattr(decode_chain, "chip", lambda: ops.Chip(units))
            return real(self, *args)

    m.setattr(decode_chain.DecodeChain, "run", run)
    return m


@pytest.mark.parametrize("rows", [1, 2, 4, 8, 16])
def test_workgroups_that_start_too_late_leave(rows):
    """A workgroup's LDS leaves no room for another one on its unit: of twice as many as there are units, the list is closed
    without those that start when others have ended."""
    from rapid_llm_amd.kernels import ops

    cfg = {**BASE, "hidden_size": 1024, "num_attention_heads": 8, "intermediate_size": 1536}
    units, dealt = ops.chip().units, 32  # (the word that holds how many workgroups the items were dealt to)
    results = []
    for launched in (units, min(2 * units, 512)):
        runner = _runner(cfg)
        tokens, entries = _fill(runner, CONTEXTS[:rows], cfg["vocab_size"])
        m = _launched_with(launched)
        try:
            results.append(_again(runner, tokens, entries))
        finally:
            m.undo()
        for _ in range(5):
            assert torch.equal(_again(runner, tokens, entries), results[0])
            assert 1 <= int(runner.model._chain_space.control.view(torch.int32)[dealt]) <= units
        runner.check(runner.lost)
    assert torch.equal(results[1], results[0])


@pytest.mark.parametrize("kv_heads", [1, 2])
def test_contexts_of_nine_to_sixteen_shares(tmp_path, kv_heads):
    """Whoever folds a request's shares asks for eight at a time: contexts of 16, 9, 15 and 10 shares, each head folded by a workgroup
    of its own, and (fewer workgroups than items) all by the last share's."""
    from rapid_llm_amd import write_random_model

    cfg = {**BASE, "num_key_value_heads": kv_heads, "num_hidden_layers": 2, "max_position_embeddings": 4096}
    folder = str(write_random_model(cfg, 7, tmp_path / "long", dtype="bfloat16"))
    config, weights = plain_load(folder)
    contexts = [4089, 2303, 3839, 2304]
    plain = None
    for rows in (1, 2, 4):
        got = []
        for launched in (None, 5):
            runner = _runner(folder, max_seq_len=4096, num_pages=900)
            tokens, entries = _fill(runner, contexts[:rows], cfg["vocab_size"])
            m = _launched_with(launched) if launched else pytest.MonkeyPatch()
            try:
                got.append(_again(runner, tokens, entries).cpu())
            finally:
                m.undo()
            (chain,) = _chains(runner)
            assert chain is not None and chain.nsplit == 16
            assert torch.equal(_again(runner, tokens, entries).cpu(), got[-1])
        assert torch.equal(got[0], got[1])
        if plain is None:
            every = [random_tokens(n + 1, cfg["vocab_size"], 31 + i) for i, n in enumerate(contexts)]
            plain = torch.stack([plain_forward(config, weights, ids)[-1] for ids in every])
        parity.assert_bf16_close(got[0], plain[:rows], f"decode chain/long/{kv_heads}/{rows}")


def _count_from(runner, launch):
    """The number of the next launch, as if so many had gone before."""
    from rapid_llm_amd.kernels import decode_chain

    word = decode_chain._library().rl_decode_chain_launch_word() // 4
    torch.cuda.synchronize()
    runner.model._chain_space.control.view(torch.int32)[word] = launch - (1 << 32 if launch >= 1 << 31 else 0)
    torch.cuda.synchronize()


@pytest.mark.parametrize("rows", [1, 2, 4, 16])
def test_results_do_not_depend_on_how_many_launches_went_before(rows):
    layers = 4
    cfg = {**BASE, "hidden_size": 1024, "num_attention_heads": 8, "intermediate_size": 1536, "num_hidden_layers": layers}
    runner = _runner(cfg)
    tokens, entries = _fill(runner, CONTEXTS[:rows], cfg["vocab_size"])
    want = _again(runner, tokens, entries)
    # (a count of the phases of all launches would be beyond 2^31, beyond 2^32; the launch's number beyond 2^31)
    for launch in (2**31 // (5 * layers) + 1, 2**32 // (5 * layers) + 1, 2**31 + 5):
        _count_from(runner, launch)
        for _ in range(3):
            assert torch.equal(_again(runner, tokens, entries), want), launch


@pytest.mark.parametrize("rows", [(1, 2), (2, 4), (16, 1)])
def test_launch_numbers_begin_again(rows):
    """Behind the last number everything that carries one is cleared: no place that was written under a number, or never,
    is taken for written under the same number met again."""
    from rapid_llm_amd.kernels import decode_chain

    cfg = {**BASE, "hidden_size": 1024, "num_attention_heads": 8, "intermediate_size": 1536}
    steps = []
    runner = _runner(cfg)
    for n in rows:
        tokens, entries = _fill(runner, CONTEXTS[:n], cfg["vocab_size"])
        steps.append((_again(runner, tokens, entries), n))
        for rid in list(tokens):
            runner.finish(rid)
    space, last = runner.model._chain_space, decode_chain._library().rl_decode_chain_last_launch()
    word = decode_chain._library().rl_decode_chain_launch_word() // 4
    for before in (2, 0):  # launches in front of the last one
        _count_from(runner, last - before)
        for i in range(before + 3):
            want, n = steps[i % 2]
            tokens, entries = _fill(runner, CONTEXTS[:n], cfg["vocab_size"])
            assert torch.equal(_again(runner, tokens, entries), want), (before, i)
            for rid in list(tokens):
                runner.finish(rid)
            torch.cuda.synchronize()
            number = int(space.control.view(torch.int32)[word]) & 0xFFFFFFFF
            assert number == (last - before + i + 1 if i < before else i - before), (before, i)
            if number == 0:
                assert not space.tagged.any() and not space.shares.any()
                control = space.control.view(torch.int32).clone()
                assert not control.any()


def _give_up(model):
    """What a launch leaves that ran into the bound of a wait: every later one ends at once."""
    from rapid_llm_amd.kernels import decode_chain

    torch.cuda.synchronize()
    model._chain_space.control.view(torch.int32)[decode_chain._library().rl_decode_chain_abort_word() // 4] = 1
    torch.cuda.synchronize()


@pytest.mark.parametrize("rows", [1, 4, 16])
def test_a_launch_that_is_given_up_is_reported_and_not_made_again(rows):
    from rapid_llm_amd.engine.scheduler import LostStep

    cfg = {**BASE, "hidden_size": 512}
    runner = _runner(cfg)
    tokens, entries = _fill(runner, CONTEXTS[:rows], cfg["vocab_size"])
    want = _again(runner, tokens, entries)
    runner.check(runner.lost)
    _give_up(runner.model)
    before = runner.lost
    assert _again(runner, tokens, entries).isnan().all()
    torch.cuda.synchronize()
    with pytest.raises(LostStep):  # whoever reads that step asks, ...
        runner.check(before)
    with pytest.raises(LostStep):  # ... also behind somebody else
        runner.check(before)
    runner.check(runner.lost)
    got = _again(runner, tokens, entries)
    assert _chains(runner) == [None]
    parity.assert_bf16_close(got.cpu(), want.cpu(), f"kernels behind a lost launch/{rows}")
    for _ in range(3):
        assert torch.equal(_again(runner, tokens, entries), got)


def test_the_next_step_reports_a_launch_that_was_given_up():
    from rapid_llm_amd.engine.scheduler import LostStep

    cfg = {**BASE, "hidden_size": 512}
    runner = _runner(cfg)
    tokens, entries = _fill(runner, CONTEXTS[:2], cfg["vocab_size"])
    want = _again(runner, tokens, entries)
    _give_up(runner.model)
    _again(runner, tokens, entries)
    torch.cuda.synchronize()
    pages = runner.cache.num_free_pages()
    with pytest.raises(LostStep):
        runner.step(entries)
    assert runner.cache.num_free_pages() == pages and runner.computed[entries[0].request_id] == len(tokens["r0"]) - 1
    parity.assert_bf16_close(_again(runner, tokens, entries).cpu(), want.cpu(), "kernels behind a lost launch/next step")


@pytest.mark.parametrize("pipeline", [False, True])
def test_generation_goes_on_behind_a_launch_that_was_given_up(pipeline):
    from rapid_llm_amd import LLM, SamplingParams
    from rapid_llm_amd.engine.scheduler import LostStep

    cfg = {**BASE, "hidden_size": 512}
    llm = LLM(cfg, dtype="bfloat16", max_seq_len=256, max_num_seqs=8, num_pages=200, load_format="random", pipeline=pipeline)
    prompts = [random_tokens(n, cfg["vocab_size"], 3 + n) for n in (5, 17, 40)]
    params = SamplingParams(temperature=0.0, max_gen_len=24, ignore_eos=True)
    want = [o.outputs[0].token_ids for o in llm.generate(prompts, params)]
    requests = llm._submit(prompts, params)
    scheduler = llm.scheduler
    for _ in range(9):
        scheduler.step()
    known = [list(r.output_token_ids) for r in requests]
    _give_up(scheduler.runner.model)
    with pytest.raises(LostStep):
        while scheduler.has_unfinished_requests():
            scheduler.step()
    # what had been read by then is right, and everything else is computed again
    for r, k, w in zip(requests, known, want):
        assert r.output_token_ids[: len(k)] == k == w[: len(k)] and r.output_token_ids == w[: len(r.output_token_ids)]
    scheduler.run_to_completion()
    assert all(len(r.output_token_ids) == 24 and r.finish_reason == "length" for r in requests)
    assert all(c is None for c in _chains(scheduler.runner)) and scheduler.runner.lost == 1


def test_replays_between_other_steps():
    from rapid_llm_amd import StepEntry

    cfg = {**BASE, "hidden_size": 1024, "num_attention_heads": 8, "num_hidden_layers": 6, "intermediate_size": 1536}
    runner = _runner(cfg)
    steps = []
    for k, rows in enumerate((1, 2, 7, 16)):  # recorded steps that share one space
        tokens, entries = _fill(runner, CONTEXTS[:rows], cfg["vocab_size"])
        want = runner.step(entries, use_graph=False).clone()
        for rid in tokens:
            runner.computed[rid] = len(tokens[rid]) - 1
        first = _again(runner, tokens, entries)
        parity.assert_bf16_close(first.cpu(), want.cpu(), f"decode chain against kernels/{rows}")
        for _ in range(60):
            again = _again(runner, tokens, entries)
        assert torch.equal(again, first)
        for rid in list(tokens):
            runner.finish(rid)
        steps.append((tokens, first))
        runner.step([StepEntry("other", random_tokens(70, cfg["vocab_size"], k), [0])])
        runner.finish("other")
    for rows, (tokens, first) in zip((1, 2, 7, 16), steps):
        t2, entries = _fill(runner, CONTEXTS[:rows], cfg["vocab_size"])
        for _ in range(3):
            assert torch.equal(_again(runner, t2, entries), first)
        for rid in list(t2):
            runner.finish(rid)


def test_two_at_once():
    """Two runners on streams and threads of their own: the chip cannot hold both launches' workgroups at a time."""
    cfg = {**BASE, "hidden_size": 1024, "num_attention_heads": 8, "num_hidden_layers": 8, "intermediate_size": 3072}
    pairs = []
    for rows in (1, 6):
        runner = _runner(cfg)
        tokens, entries = _fill(runner, CONTEXTS[:rows], cfg["vocab_size"])
        pairs.append((runner, tokens, entries, _again(runner, tokens, entries)))
    torch.cuda.synchronize()
    wrong = []

    def work(runner, tokens, entries, want):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(80):
                if not torch.equal(_again(runner, tokens, entries), want):
                    wrong.append(len(tokens))

    threads = [threading.Thread(target=work, args=p) for p in pairs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not wrong


def test_pages_beyond_the_launchs_indices_keep_their_kernels():
    cfg = {**BASE, "max_position_embeddings": 131072}
    runner = _runner(cfg, max_seq_len=131072, page_size=65536, num_pages=6, max_num_seqs=2)
    tokens, entries = _fill(runner, [300, 20], cfg["vocab_size"])
    got = _again(runner, tokens, entries)
    assert _chains(runner) == [None]
    parity.assert_bf16_close(got.cpu(), runner.step(entries, use_graph=False).cpu(), "pages of 65,536 tokens")


def test_layers_that_do_something_else_keep_their_kernels(monkeypatch):
    cfg = {**BASE, "hidden_size": 512}
    for change in (dict(head_dim=64), dict(num_attention_heads=10), dict(intermediate_size=392)):
        runner = _runner({**cfg, **change})
        tokens, entries = _fill(runner, [20, 3], cfg["vocab_size"])
        _again(runner, tokens, entries)
        assert _chains(runner) == [None], change
    runner = _runner(cfg)
    real, calls = runner.model.blocks[1].mixer.forward, []
    runner.model.blocks[1].mixer.forward = lambda *a: calls.append(1) or real(*a)
    tokens, entries = _fill(runner, [20, 3], cfg["vocab_size"])
    before = len(calls)
    _again(runner, tokens, entries)
    assert _chains(runner) == [None] and len(calls) > before
