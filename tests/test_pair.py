"""The product whose waves share a tile over halves of K: what its plans ask of the kernel, and the kernel against 64 bits."""

import random

import pytest
import torch

from rapid_llm_amd.kernels import ops


@pytest.mark.parametrize("kind", ["plain", "runs", "gated"])
def test_plans_are_what_the_kernel_takes(kind):
    rng = random.Random(1)
    found = 0
    for _ in range(4000):
        m, n, k = rng.choice((rng.randint(1, 1400), rng.randint(1, 80))), 8 * rng.randint(1, 1600), 64 * rng.randint(1, 200)
        plan = ops.pair_plan(m, n, k, kind, 256)
        if plan is None:
            continue
        found += 1
        tw, tx, ks = plan
        assert ops.SKINNY_MAX_ROWS < m <= 1024 and tw in (2, 3, 4) and tx in (2, 4) and (kind != "gated" or tw % 2 == 0) and (kind == "runs" or ks == 1)
        chunks = k // 64
        assert -(-chunks // ks) * (ks - 1) < chunks  # every run holds a chunk
        tiles = -(-n // ((16 if kind == "gated" else 32) * tw)) * -(-m // (32 * tx))
        assert tiles * ks <= 256 and (m + 128) * k * 2 <= 0x7FFFFFFF
    assert found > 100
    assert ops.pair_plan(200, 4092, 2048, kind, 256) is None and ops.pair_plan(200, 4096, 2080, kind, 256) is None


@pytest.mark.parametrize("kind,m,n,k,there", [
    ("gated", 87, 512, 2560, False), ("gated", 113, 1024, 2560, True), ("gated", 120, 768, 4352, False), ("gated", 708, 1224, 4608, True),
    ("gated", 618, 664, 16128, False), ("gated", 74, 1024, 4608, False), ("runs", 359, 10328, 320, False), ("runs", 332, 2560, 512, False), ("runs", 265, 1624, 512, True),
    ("runs", 459, 3800, 768, False), ("runs", 128, 9728, 768, True), ("runs", 225, 14336, 768, False), ("runs", 87, 11624, 1920, True)])
def test_sizes_that_other_products_are_faster_at(kind, m, n, k, there):
    """Widths of no one model: few tiles over long sums, and results of short sums that are most of the bytes."""
    assert (ops.pair_plan(m, n, k, kind, 256) is not None) == there


def test_only_steps_of_a_model_go_there():
    assert ops.pair(200, 6144, 4096, "plain") is None and ops.library_takes(200, 6144, 4096)
    with ops.shared_tiles():
        assert ops.pair(200, 6144, 4096, "plain") == ops.pair_plan(200, 6144, 4096, "plain", ops.chip().units) is not None
        assert not ops.library_takes(200, 6144, 4096) and ops.pair(64, 6144, 4096, "plain") is None
        assert ops.pair(64, 4096, 12288, "runs") == (2, 2, 4) and ops.pair(17, 3072, 1024, "gated") == (2, 2, 1) and ops.pair(16, 3072, 1024, "gated") is None
        assert ops.pair(100, 4096, 1024, "plain") is None  # the tile product is level there
    assert ops.pair(200, 6144, 4096, "plain") is None


# One chunk and an odd number of them (the second group multiplies zeros), fewer chunks than buffers and more; rows and columns that end
# inside a tile of 16, a wave's tiles and a workgroup's; several tiles on both sides.
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(1, 8, 64), (70, 72, 128), (129, 200, 192), (257, 1000, 320), (65, 520, 704), (300, 264, 4096)])
@pytest.mark.parametrize("tile", [(4, 4), (3, 4), (2, 4), (4, 2), (3, 2), (2, 2)])
def test_kernel(m, n, k, tile):
    gen = torch.Generator().manual_seed(m + k)
    dev = "cuda"
    x, w, w2 = ((torch.randn(r, k, generator=gen) * s).to(torch.bfloat16).to(dev) for r, s in ((m, 1.0), (n, 0.1), (2 * n, 0.1)))
    lib, p = ops.core(), ops._p
    want = x.double() @ w.double().t()

    def launch(weight, out, kind, ks=1):
        assert lib.rl_gemm_pair(p(x), p(weight), p(out), m, n, k, k, k, n, kind, *tile, ks, ops._stream()) == 0

    # bfloat16 results: half a unit in the last place of each, 2^-9, and the float32 sums before it
    out = torch.full((m + 1, n), 7.0, dtype=torch.bfloat16, device=dev)
    launch(w, out, 3)
    assert bool((out[m] == 7.0).all())
    assert float(((out[:m].double() - want).abs() - want.abs() / 256).max()) <= 1e-5 * float(want.abs().max())
    # float32 runs: sums of k terms in float32, in an order of their own: sqrt(k) roundings of 2^-24 of the largest, eight times over
    for ks in (1, 2, 3):
        if -(-(k // 64) // ks) * (ks - 1) >= k // 64:
            continue
        runs = torch.full((ks * m + 1, n), 7.0, device=dev)
        launch(w, runs, 1, ks)
        assert bool((runs[ks * m] == 7.0).all())
        got = runs[: ks * m].view(ks, m, n).double().sum(0)
        assert float((got - want).abs().max()) <= 8 * k**0.5 * 2.0**-24 * float(want.abs().max())
    if tile in ops._PAIR_COSTS["gated"]:
        # gate and up are rounded to bfloat16 first: off by 2^-8 of themselves where a sum on the edge goes the other way, and by
        # what the sums may be off, as above; silu's slope is 1.1 at most; then the result is rounded
        both = (x.double() @ w2.double().t()).to(torch.bfloat16).double()
        gate, up, off = both[:, :n], both[:, n:], 8 * k**0.5 * 2.0**-24 * float(both.abs().max())
        act = torch.nn.functional.silu(gate) * up
        out = torch.full((m + 1, n), 7.0, dtype=torch.bfloat16, device=dev)
        launch(w2, out, 2)
        assert bool((out[m] == 7.0).all())
        slack = 1.1 * up.abs() * (gate.abs() / 256 + off) + torch.nn.functional.silu(gate).abs() * (up.abs() / 256 + off) + act.abs() / 256
        assert bool(((out[:m].double() - act).abs() <= slack).all())


# A kind's smallest and largest rows of a plan, and sizes in between.
@pytest.mark.gpu
@pytest.mark.parametrize("kind,m,n,k", [("plain", 65, 6144, 2560), ("plain", 200, 4096, 2048), ("plain", 1023, 1024, 1024), ("gated", 17, 3072, 1024),
                                        ("gated", 129, 3072, 1024), ("runs", 18, 2560, 9728), ("runs", 100, 2560, 4096), ("runs", 500, 1024, 3072)])
def test_a_layers_products_go_there_with_operands_of_any_place(kind, m, n, k, monkeypatch):
    """Through the entry points that the layers call: rows side by side in whole units of 16 bytes go there, rows that are columns
    of wider ones as a copy (runs: elsewhere), operands that begin inside a unit elsewhere.  All of them give the product."""
    from rapid_llm_amd.parts.linear import Linear

    went, launch = [], ops._pair
    monkeypatch.setattr(ops, "_pair", lambda *args: went.append(args[3]) or launch(*args))
    gen = torch.Generator().manual_seed(m + n)
    rows = 2 * n if kind == "gated" else n
    room_x, room_w = torch.randn(m * k + 8, generator=gen).to(torch.bfloat16).cuda(), (torch.randn(rows * k + 8, generator=gen) * k**-0.5).to(torch.bfloat16).cuda()

    def operands(x_at, w_at, apart):
        x, w = room_x[x_at : x_at + m * k].view(m, k), room_w[w_at : w_at + rows * k].view(rows, k)
        if apart:
            wider = torch.full((m, k + 8), float("nan"), dtype=torch.bfloat16, device="cuda")
            wider[:, :k] = x
            x = wider[:, :k]
        return x, w

    for x_at, w_at, apart in ((0, 0, False), (8, 8, False), (1, 0, False), (0, 3, False), (0, 0, True)):
        if apart and (kind == "gated" or kind == "runs" and m <= ops.mid_max_rows(n, k)):
            continue  # (refused, as they were: a layer's rows are side by side)
        x, w = operands(x_at, w_at, apart)
        linear = Linear(k, rows)
        linear.bind(w)
        went.clear()
        with ops.shared_tiles():
            there = x_at % 8 == 0 and w_at % 8 == 0 and not (apart and kind == "runs")
            if kind == "gated":
                got = ops.gemm_bf16_swiglu(x, w)
                if got is None:
                    got = ops.gemm_bf16(x, w, torch.bfloat16)
                    gate, up = got[:, :n].double(), got[:, n:].double()
                    got = torch.nn.functional.silu(gate) * up
            elif kind == "runs":
                assert ops.pair_reads(x, w) == there
                got = linear.partial_sums(x).double().sum(0) if linear.midsize(x) else linear(x)
            else:
                got = linear(x)
        assert went == ([kind] if there else [])
        want = x.double() @ w.double().t().contiguous()
        # float32 sums in an order of their own, as above; rounded to bfloat16 where they are stored as that
        off = 8 * k**0.5 * 2.0**-24 * float(want.abs().max())
        if kind == "gated":
            both = want.to(torch.bfloat16).double()
            gate, up = both[:, :n], both[:, n:]
            want = torch.nn.functional.silu(gate) * up
            bound = 1.1 * up.abs() * (gate.abs() / 256 + off) + torch.nn.functional.silu(gate).abs() * (up.abs() / 256 + off) + want.abs() / 256
        else:
            bound = want.abs() / 256 + off
        assert bool(((got.double() - want).abs() <= bound).all()), (x_at, w_at, apart)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [(2, 2), (2, 4), (4, 2)])
def test_every_gate_has_the_activation_of_the_many_row_product(tile):
    """All bfloat16 gates against sixty factors, infinities and NaN among both: bit for bit what the other product with an activation
    stores, whose form is the more exact one (a wave's numbers below 87, some beyond and all of them)."""
    lib, p = ops.core(), ops._p
    gates = torch.arange(1 << 16, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    gen = torch.Generator().manual_seed(3)
    ups = torch.cat((torch.randn(40, generator=gen), torch.randn(20, generator=gen) * 100, torch.tensor([0.0, -0.0, float("inf"), float("nan")]))).to(torch.bfloat16)
    m, n, k = gates.numel(), ups.numel(), 64
    x, w = torch.zeros(m, k, dtype=torch.bfloat16), torch.zeros(2 * n, k, dtype=torch.bfloat16)
    # gate * 1 and 1 * up, beside products with 0: NaN for a number that is not finite
    x[:, 0], x[:, 1], w[:n, 0], w[n:, 1] = gates, 1.0, 1.0, ups
    x, w = x.cuda(), w.cuda()
    want, out = (torch.full((m, n), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    assert lib.rl_gemm_block(p(x), p(w), p(want), m, n, k, k, k, n, 2, 2, 2, 1, ops._stream()) == 0
    assert lib.rl_gemm_pair(p(x), p(w), p(out), m, n, k, k, k, n, 2, *tile, 1, ops._stream()) == 0
    assert torch.equal(out.isnan(), want.isnan())
    same = (out.view(torch.int16) == want.view(torch.int16)) | want.isnan()
    assert bool(same.all()), int((~same).sum())


@pytest.mark.gpu
def test_sizes_the_kernel_refuses():
    lib, p = ops.core(), ops._p
    x, w, out = (torch.zeros(256, 256, dtype=torch.bfloat16, device="cuda") for _ in range(3))
    ok = dict(M=64, N=64, K=64, ldx=256, ldw=256, ldo=256, kind=3, tw=2, tx=2, splits=1)

    def code(**change):
        a = {**ok, **change}
        return lib.rl_gemm_pair(p(x), p(w), p(out), a["M"], a["N"], a["K"], a["ldx"], a["ldw"], a["ldo"], a["kind"], a["tw"], a["tx"], a["splits"], ops._stream())

    assert code() == 0 and code(M=0) == 0
    for change in (dict(K=96), dict(N=60), dict(ldx=60), dict(ldo=63), dict(kind=0), dict(kind=2, tw=3), dict(kind=2, tw=4, tx=4), dict(tw=5), dict(tx=3), dict(splits=2),
                   dict(kind=1, splits=2), dict(ldx=100)):
        assert code(**change) != 0, change
