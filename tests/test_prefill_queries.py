"""Queries that the prefill attention finishes itself, as it reads them from the packed rows."""

import random
from types import SimpleNamespace

import pytest
import torch

from rapid_llm_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
SHAPES = [(1, 1), (2, 1), (1, 3), (2, 3)]  # wave groups, runs of keys
EPS = 3e-6


def _problem(seqs, nq, nkv, d, page, seed, change=None):
    """Packed rows whose keys and values are in the caches already; ``change(i, keys)`` may change those of request i."""
    gen, rng = torch.Generator().manual_seed(seed), random.Random(seed)
    pages = [-(-(a + n) // page) for a, n in seqs]
    ids, slots = list(range(1, sum(pages) + 1)), list(range(len(seqs) + 3))
    rng.shuffle(ids)
    rng.shuffle(slots)
    table = torch.zeros(len(slots), max(pages) + 1, dtype=torch.int32)
    kc, vc = torch.full((len(ids) + 1, nkv, page, d), float("nan")), torch.full((len(ids) + 1, nkv, d, page), float("nan"))
    rows, requests, positions, token_slot = [], [], [], []
    for i, (a, n) in enumerate(seqs):
        k, v = (torch.randn(a + n, nkv, d, generator=gen) for _ in range(2))
        if change is not None:
            change(i, k)
        k, v = k.bfloat16().float(), v.bfloat16().float()
        for p in range(pages[i]):
            pid = ids.pop()
            table[slots[i], p] = pid
            lo, hi = p * page, min(a + n, (p + 1) * page)
            kc[pid, :, : hi - lo], vc[pid, :, :, : hi - lo] = k[lo:hi].transpose(0, 1), v[lo:hi].permute(1, 2, 0)
        rows.append(torch.randn(n, (nq + 2 * nkv) * d, generator=gen).bfloat16())
        requests.append((k, v, torch.arange(a, a + n)))
        positions += range(a, a + n)
        token_slot += [slots[i]] * n
    ctx = SimpleNamespace(
        positions=torch.tensor(positions, dtype=torch.int32, device=DEV), token_slot=torch.tensor(token_slot, dtype=torch.int32, device=DEV),
        token_ids=torch.zeros(len(positions), dtype=torch.int32, device=DEV), h_seq_starts=[a for a, _ in seqs], h_seq_lens=[n for _, n in seqs],
        max_position=max(positions), extra={},
    )
    return torch.cat(rows), requests, slots[: len(seqs)], kc.bfloat16().to(DEV), vc.bfloat16().to(DEV), table.to(DEV), ctx


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"g{s[0]}n{s[1]}")
@pytest.mark.parametrize("nq,nkv,d,page", [(8, 2, 64, 16), (8, 2, 128, 16), (6, 3, 128, 12), (4, 2, 192, 8), (4, 4, 256, 16)])
def test_queries_that_nothing_changes_are_not_rounded(nq, nkv, d, page, shape, monkeypatch):
    """Without a norm, and without a rotation or with one by no angle, a query is the bfloat16 numbers of its row: bit for bit what
    the kernel gives for queries that were written out."""
    monkeypatch.setattr(ops, "_prefill_shape", lambda *a, **k: shape)
    seqs = [(0, 70), (300, 37), (5, 1), (0, 2)]
    rows, _, _, kc, vc, table, ctx = _problem(seqs, nq, nkv, d, page, d + page)
    cos, sin = torch.ones(400, d // 2, device=DEV), torch.zeros(400, d // 2, device=DEV)
    outs = []
    for q, prepare in ((rows[:, : nq * d].contiguous(), None), (rows, (None, None, None, EPS)), (rows, (None, cos, sin, EPS))):
        out = torch.full((len(rows), nq * d), float("nan"), dtype=torch.bfloat16, device=DEV)
        ops.paged_attention(q.to(DEV), kc, vc, out, ctx, table, page, nq, nkv, d, 0, d**-0.5, prepare=prepare)
        outs.append(out)
    assert bool(outs[0].isfinite().all()) and torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.parametrize("group", [32769, 46347])
def test_as_many_query_heads_as_there_may_be_on_a_kv_head(group):
    """Rows of a portion are divided by the group's heads: more heads than the square root of what a 32-bit product reaches."""
    d, page, seqs = 16, 16, [(0, 2), (5, 3)]
    _, requests, _, kc, vc, table, ctx = _problem(seqs, 1, 1, d, page, 3)
    gen = torch.Generator().manual_seed(group)
    q = torch.randn(5, group, d, generator=gen).bfloat16().to(DEV)
    out = torch.full((5, group * d), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.paged_attention(q.view(5, -1), kc, vc, out, ctx, table, page, group, 1, d, 0, d**-0.5)
    at = 0
    for k, v, positions in requests:
        for pos in positions.tolist():
            k1, v1 = k[: pos + 1, 0].to(DEV).double(), v[: pos + 1, 0].to(DEV).double()
            want = torch.softmax(q[at].double() @ k1.T.contiguous() * d**-0.5, dim=1) @ v1
            # weights and results are rounded to bfloat16, 2^-9 each, and the weights' sum is not of the rounded ones
            assert bool(((out[at].view(group, d).double() - want).abs() <= 2.0**-7 * v1.abs().amax()).all())
            at += 1


# Levels of the keys of each step of 64, as powers of two of their weights: one key of every step at the first number, the others at the
# second.  The maximum moves by less than the rescaling's 8 and by more, at once and step by step, up from far below and never again.
LEVELS = {
    "below eight": [(0, 0), (7.5, 0), (0, 0), (7.9, 1)],
    "nine, then less": [(0, 0), (0, 0), (9, 0), (8, 2), (8.9, 0)],
    "steps of five": [(0, 0), (5, 0), (10, 5), (15, 10), (20, 14)],
    "up from far below": [(-60, -60), (-20, -60), (0, -7), (9, 0)],
    "first": [(20, 14), (0, 0), (13, 0)],
    "far up and on": [(0, 0), (60, 0), (61, 55), (69.5, 62)],
}


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"g{s[0]}n{s[1]}")
@pytest.mark.parametrize("nq,nkv,d,page", [(8, 2, 64, 16), (8, 2, 128, 16), (6, 3, 128, 12), (4, 2, 192, 8), (4, 4, 256, 16), (6, 2, 80, 8)])
@pytest.mark.parametrize("window", [0, 150])
def test_maxima_that_move(nq, nkv, d, page, window, shape, monkeypatch):
    """Rows whose largest score moves from step to step, a request for each course of it, finished in the kernel (with a norm, whose
    scores begin with the negative maximum, with a rotation, by no angle, and both) and finished before; the tiles bring the
    requests' rows of the block table with them, the tokens' own say another."""
    monkeypatch.setattr(ops, "_prefill_shape", lambda *a, **k: shape)
    seqs = [(64 * len(LEVELS[name]) - 40, 50 + 3 * i) for i, name in enumerate(LEVELS)]
    gen = torch.Generator().manual_seed(d)
    u = torch.randn(d, generator=gen)
    u /= u.norm()

    def levels(i, keys):
        for t in range(keys.shape[0]):
            course = list(LEVELS.values())[i]
            top, rest = course[min(t // 64, len(course) - 1)]
            keys[t] *= 0.3
            keys[t] += (top if t % 64 == 37 else rest) / 1.4426950408889634 * u

    rows, requests, slots, kc, vc, table, ctx = _problem(seqs, nq, nkv, d, page, d + page, levels)
    # every query points the keys' way: u times the square root of d behind a norm
    q = (u + 0.02 * torch.randn(len(rows), nq, d, generator=gen)).view(len(rows), nq * d)
    weight = 1 + 0.1 * torch.randn(d, generator=gen)
    rows[:, : nq * d] = (q.view(-1, nq, d) / weight).view(len(rows), -1).bfloat16()
    lie = next(s for s in range(table.shape[0]) if s not in slots)  # (its pages hold NaN)
    ctx.h_seq_slots = slots
    ctx.token_slot.fill_(lie)
    raw = rows[:, : nq * d].double().view(-1, nq, d)
    finished = raw * torch.rsqrt(raw.square().mean(-1, keepdim=True) + EPS) * weight.double()
    cos, sin = torch.ones(600, d // 2, device=DEV), torch.zeros(600, d // 2, device=DEV)
    ways = [(finished.bfloat16().view(len(rows), -1), None)]
    if d % 64 == 0:
        packed = rows.clone()
        packed[:, : nq * d] = ways[0][0]
        ways += [(rows, (weight.to(DEV), None, None, EPS)), (rows, (weight.to(DEV), cos, sin, EPS)), (packed, (None, cos, sin, EPS))]
    for way, prepare in ways:
        out = torch.full((len(rows), nq * d), float("nan"), dtype=torch.bfloat16, device=DEV)
        ops.paged_attention(way.to(DEV), kc, vc, out, ctx, table, page, nq, nkv, d, window, d**-0.5, prepare=prepare)
        at = 0
        for name, (k, v, positions) in zip(LEVELS, requests):
            n = len(positions)
            k, v = (x.repeat_interleave(nq // nkv, 1).transpose(0, 1).double() for x in (k, v))
            scores = finished[at : at + n].transpose(0, 1) @ k.transpose(1, 2).contiguous() * d**-0.5
            keys = torch.arange(k.shape[1])
            seen = (keys <= positions[:, None]) & ((keys > positions[:, None] - window) if window else True)
            want = (torch.softmax(scores.masked_fill(~seen, float("-inf")), dim=-1) @ v).transpose(0, 1).reshape(n, -1)
            got = out[at : at + n].cpu().double()
            at += n
            # the bounds of attention over normal keys, of the outputs' spread (2.5% and 0.4% seen); any step's keys weighed twice would
            # move the rows of "nine, then less" by 4% to 39%, of "below eight" by 9% to 35%
            off = (got - want) / want.std()
            assert float(off.abs().max()) <= 0.06 and float(off.square().mean(1).sqrt().max()) <= 0.012, name
