"""The engine's work by size: steps of the Qwen3 dense decoder through ``ModelRunner.step``.

A case is one step as a scheduler makes it: some requests decode one token behind their
context, others bring prompt tokens (a whole prompt, or a portion behind what the cache already
holds), in one flat batch.  Layer sizes are those of the family's members that ``bench.py``
knows; weights and token ids are random, drawn from the seed.  After the step every request is put
back to where it was, so that the same step can be run again.
"""

import json
import math
import random

import torch

from rapid_llm_amd import EngineConfig, ModelRunner, StepEntry

_VOCAB, _HEAD_DIM, _KV_HEADS, _THETA, _EPS = 151936, 128, 8, 1e6, 1e-6
_PAGE = 16  # tokens a cache page
_FILL = 8192  # tokens of context that one step of prepare() computes
_NORM_STD = 0.1  # norm weights are 1 + N(0, this)
# what the matrices that write to the residual stream are multiplied by: as in a trained model, a
# layer then adds a few per cent to a stream that begins with the embedding (with N(0, 0.02) as
# drawn, the first layer's output is fifty times the embedding, and rounding grows with depth)
_BRANCH = 1 / 512

# layers, hidden size, query heads, intermediate size, whether the output shares the embedding
_SHAPES = {
    "0.6b": (28, 1024, 16, 3072, True),
    "1.7b": (28, 2048, 16, 6144, True),
    "4b": (36, 2560, 32, 9728, True),
    "8b": (36, 4096, 32, 12288, False),
}


def _case(shape, dtype, decoding=0, contexts=(0, 0), prompts=0, tokens=(0, 0), behind=0):
    """``decoding`` requests with contexts of ``contexts`` (least, most) tokens, and ``prompts`` more that
    bring ``tokens`` (least, most) tokens each behind ``behind`` tokens in the cache."""
    return {
        "shape": shape, "dtype": dtype, "decoding": decoding, "context_low": contexts[0], "context_high": contexts[1],
        "prompts": prompts, "prompt_low": tokens[0], "prompt_high": tokens[1], "behind": behind,
    }


def listed():
    return [
        # interactive use of the smallest model: the next token of one short chat
        dict(_case("0.6b", "bfloat16", 1, (300, 300)), name="0.6b decode 1"),
        # its time to first token: one short question
        dict(_case("0.6b", "bfloat16", prompts=1, tokens=(37, 37)), name="0.6b prompt 37"),
        # offline generation: 256 requests at once with prompts of 64 to 1,024 tokens, a decode step ...
        dict(_case("0.6b", "bfloat16", 256, (64, 1151)), name="0.6b decode 256"),
        # ... and one of the steps that bring the prompts in
        dict(_case("0.6b", "bfloat16", prompts=14, tokens=(64, 1024)), name="0.6b prompts 14"),
        # the headline model behind prompts of about 2,048 tokens: one user, ...
        dict(_case("8b", "bfloat16", 1, (2048, 2048)), name="8b decode 1"),
        # ... the benchmark's batch, ...
        dict(_case("8b", "bfloat16", 8, (2048, 2304)), name="8b decode 8"),
        # ... a busy server, whose requests have contexts of every length
        dict(_case("8b", "bfloat16", 64, (64, 2048)), name="8b decode 64"),
        # the headline prompt
        dict(_case("8b", "bfloat16", prompts=1, tokens=(2048, 2048)), name="8b prompt 2048"),
        # chunked prefill: a portion of a long prompt beside decoding requests, 512 tokens in all
        dict(_case("8b", "bfloat16", 15, (64, 2048), 1, (497, 497), 7680), name="8b chunk and decode 15"),
        # the true 32-bit engine: a few short prompts of the smallest model, ...
        dict(_case("0.6b", "float32", prompts=3, tokens=(17, 300)), name="0.6b f32 prompts 3"),
        # ... and the headline model's decode step and prompt
        dict(_case("8b", "float32", 8, (512, 1536)), name="8b f32 decode 8"),
        dict(_case("8b", "float32", prompts=1, tokens=(2048, 2048)), name="8b f32 prompt 2048"),
    ]


def draw(rng):
    """A step of one of the three kinds (decoding, prompts, both) at any member and type; sizes are
    spread over their logarithm, within what the largest listed cases cost."""

    def size(low, high):
        return round(math.exp(rng.uniform(math.log(low), math.log(high))))

    while True:
        shape, dtype = rng.choice(list(_SHAPES)), rng.choice(["bfloat16", "bfloat16", "float32"])
        kind = rng.choice(["decode", "prompt", "mixed"])
        decoding = prompts = behind = 0
        contexts = tokens = (0, 0)
        if kind != "prompt":
            decoding = size(1, 256) if kind == "decode" else size(1, 48)
            low = size(16, 2048)
            contexts = (low, size(low, 4096))
        if kind != "decode":
            prompts = size(1, 16)
            low = size(8, 2048)
            tokens = (low, size(low, 4096))
            behind = rng.choice([0, size(16, 8192)])
        case = _case(shape, dtype, decoding, contexts, prompts, tokens, behind)
        old, new = (sum(n) for n in zip(*_requests(case)))
        if new <= 8192 and _seconds(case, new) <= 0.25 and _seconds(case, old) <= 1.5 and _bytes(case) <= 20e9:
            return case


def _requests(case):
    """(tokens in the cache, tokens of the step) of every request, the decoding ones first."""
    rng = random.Random(json.dumps([v for k, v in sorted(case.items()) if k != "name"]))
    decoding = [(rng.randint(case["context_low"], case["context_high"]), 1) for _ in range(case["decoding"])]
    prompts = [(case["behind"], rng.randint(case["prompt_low"], case["prompt_high"])) for _ in range(case["prompts"])]
    return decoding + prompts


def _layer_weights(case):
    _, h, heads, inter, _ = _SHAPES[case["shape"]]
    q, kv = heads * _HEAD_DIM, _KV_HEADS * _HEAD_DIM
    return (q + 2 * kv) * h + h * q + 3 * inter * h


def _seconds(case, tokens):
    """About what so many prompt tokens cost (only to keep drawn cases within the listed ones)."""
    return 2.0 * tokens * _layer_weights(case) * _SHAPES[case["shape"]][0] / (6e14 if case["dtype"] == "bfloat16" else 9e13)


def _bytes(case):
    layers = _SHAPES[case["shape"]][0]
    return sum(a + b for a, b in _requests(case)) * layers * 2 * _KV_HEADS * _HEAD_DIM * (2 if case["dtype"] == "bfloat16" else 4)


def work(case):
    layers, h, heads, _, _ = _SHAPES[case["shape"]]
    elem = 2 if case["dtype"] == "bfloat16" else 4
    requests = _requests(case)
    tokens = sum(n for _, n in requests)
    weights = layers * _layer_weights(case) + _VOCAB * h
    # cached keys and values are read once a request, the step's own are written
    moved = elem * (weights + tokens * h) + _bytes(case) + 4 * len(requests) * _VOCAB
    pairs = sum(n * old + n * (n + 1) // 2 for old, n in requests)  # (query, visible key)
    flops = 2.0 * layers * (tokens * _layer_weights(case) + 2 * pairs * heads * _HEAD_DIM)
    return {"bytes": moved, "flops": flops + 2.0 * len(requests) * _VOCAB * h}


def tolerance(case):
    # four times what the same step gives when it is cut into other batches: other kernels, other
    # orders of summation (bfloat16), the error against 64 bits (float32)
    return {"rel": 0.03, "max": 0.2} if case["dtype"] == "bfloat16" else {"rel": 1e-5}


def _config(case):
    layers, h, heads, inter, tied = _SHAPES[case["shape"]]
    return dict(
        architectures=["Qwen3ForCausalLM"], model_type="qwen3", num_hidden_layers=layers, hidden_size=h,
        num_attention_heads=heads, num_key_value_heads=_KV_HEADS, head_dim=_HEAD_DIM, intermediate_size=inter,
        vocab_size=_VOCAB, rope_theta=_THETA, rms_norm_eps=_EPS, tie_word_embeddings=tied, max_position_embeddings=40960,
    )


def _token_ids(case, seed):
    """Every request's tokens, those in the cache first."""
    gen = torch.Generator().manual_seed(seed)
    return [torch.randint(0, _VOCAB, (old + new,), generator=gen).tolist() for old, new in _requests(case)]


def prepare(case, seed):
    requests, ids = _requests(case), _token_ids(case, seed)
    longest = max(old + new for old, new in requests)
    engine = EngineConfig(
        dtype=case["dtype"], max_seq_len=max(4096, 1 << (longest - 1).bit_length()), page_size=_PAGE, seed=seed,
        num_pages=sum(-(-(old + new) // _PAGE) for old, new in requests) + 2, max_num_seqs=max(32, len(requests)),
    )
    runner = ModelRunner(_config(case), engine, load_format="random", weight_norm_std=_NORM_STD)
    for name, weight in runner.params.items():
        if name.endswith((".mixer.o", ".ff.down")):
            weight.mul_(_BRANCH)
    names = [f"r{i}" for i in range(len(requests))]
    # the contexts, several requests a step
    batch, room = [], _FILL
    for name, (old, _), toks in zip(names, requests, ids):
        at = 0
        while at < old:
            n = min(room, old - at)
            batch.append(StepEntry(name, toks[at : at + n]))
            at, room = at + n, room - n
            if room == 0:
                runner.step(batch)
                batch, room = [], _FILL
    if batch:
        runner.step(batch)
    entries = [StepEntry(name, toks[old:], [new - 1]) for name, (old, new), toks in zip(names, requests, ids)]
    return {"runner": runner, "entries": entries, "cached": {name: old for name, (old, _) in zip(names, requests)}}


def run(state):
    runner, cached = state["runner"], state["cached"]
    logits = runner.step(state["entries"])
    for name, old in cached.items():
        if old:
            runner.computed[name] = old
        else:
            runner.finish(name)
    return logits


# ---- the same in 64 bits ----------------------------------------------------------------------


def _weights(case, seed):
    """The random weights in the order in which they are drawn, as functions that draw the next."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = torch.bfloat16 if case["dtype"] == "bfloat16" else torch.float32

    def matrix(rows, cols):
        return torch.empty((rows, cols), dtype=dtype, device="cuda").normal_(0.0, 0.02, generator=gen)

    def norm(size):
        return (torch.ones(size, device="cuda") + torch.randn(size, generator=gen, device="cuda") * _NORM_STD).double()

    return matrix, norm


def _rms(x, weight):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + _EPS) * weight


def _times(x, w):
    """``x w^T`` in 64 bits, a piece of the weight's rows at a time."""
    return torch.cat([x @ piece.double().t() for piece in w.split(16384)], dim=1)


def _rotate(x, cos, sin):
    a, b = x.chunk(2, dim=-1)
    return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1)


def _attention(q, k, v):
    """Causal, one request: q [T, heads, d], k and v [T, kv heads, d]."""
    t, heads, d = q.shape
    k, v = (x.repeat_interleave(heads // x.shape[1], dim=1).transpose(0, 1).contiguous() for x in (k, v))
    k = k.transpose(1, 2).contiguous()
    out = []
    for piece in q.split(max(16, (1 << 28) // (heads * t))):
        lo = sum(o.shape[0] for o in out)
        hi = lo + piece.shape[0]
        scores = piece.transpose(0, 1).contiguous() @ k[:, :, :hi].contiguous() / math.sqrt(d)
        hidden = torch.arange(hi, device=q.device) > torch.arange(lo, hi, device=q.device)[:, None]
        probs = torch.softmax(scores.masked_fill_(hidden, -math.inf), dim=-1)
        out.append((probs @ v[:, :hi].contiguous()).transpose(0, 1))
    return torch.cat(out)


@torch.no_grad()
def exact(case, seed):
    layers, h, heads, inter, tied = _SHAPES[case["shape"]]
    ids = _token_ids(case, seed)
    lengths = [len(i) for i in ids]
    flops = 2.0 * layers * (sum(lengths) * _layer_weights(case) + sum(n * n for n in lengths) * heads * _HEAD_DIM * 2)
    if flops > 4e14:
        return None  # over about 20 seconds
    matrix, norm = _weights(case, seed)
    table = matrix(_VOCAB, h)
    x = table[torch.tensor(sum(ids, []), device="cuda")].double()
    # angles are products in 32 bits by definition of the model
    freq = 1.0 / (_THETA ** (torch.arange(0, _HEAD_DIM, 2, dtype=torch.float32) / _HEAD_DIM))
    angles = torch.cat([torch.outer(torch.arange(n, dtype=torch.float32), freq) for n in lengths]).double().cuda()[:, None]
    cos, sin = angles.cos(), angles.sin()
    for _ in range(layers):
        before, qkv, o = norm(h), matrix((heads + 2 * _KV_HEADS) * _HEAD_DIM, h), matrix(h, heads * _HEAD_DIM).mul_(_BRANCH)
        q_norm, k_norm, between = norm(_HEAD_DIM), norm(_HEAD_DIM), norm(h)
        gate_up, down = matrix(2 * inter, h), matrix(h, inter).mul_(_BRANCH)
        packed = _times(_rms(x, before), qkv).view(x.shape[0], -1, _HEAD_DIM)
        q, k, v = packed.split([heads, _KV_HEADS, _KV_HEADS], dim=1)
        q, k = _rotate(_rms(q, q_norm), cos, sin), _rotate(_rms(k, k_norm), cos, sin)
        mixed = [_attention(*part) for part in zip(q.split(lengths), k.split(lengths), v.split(lengths))]
        x = x + _times(torch.cat(mixed).flatten(1), o)
        normed = _rms(x, between)
        x = torch.cat([
            piece + _times(torch.nn.functional.silu(_times(n, gate_up[:inter])) * _times(n, gate_up[inter:]), down)
            for piece, n in zip(x.split(4096), normed.split(4096))
        ])
    final = norm(h)
    out = table if tied else matrix(_VOCAB, h)
    last = torch.tensor(lengths, device="cuda").cumsum(0) - 1
    return _times(_rms(x[last], final), out)
