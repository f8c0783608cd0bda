"""The float32 product whose waves have a run of K each: what its plans ask of the kernel, and the kernel's bits against the
shared tiles'."""

import ctypes
import random

import pytest
import torch

from rapid_llm_amd.kernels import ops

TILES = [(1, 1), (2, 1), (3, 1), (6, 1), (1, 2), (2, 2), (3, 2), (4, 2), (6, 2), (2, 3), (3, 3), (4, 3), (3, 4), (4, 4), (6, 4), (4, 5)]


def test_plans_are_what_the_kernel_takes():
    rng = random.Random(1)
    found = set()
    for _ in range(4000):
        m, n, k, units = rng.choice((rng.randint(1, 1400), rng.randint(1, 80))), rng.randint(1, 30000), 32 * rng.randint(1, 400), rng.choice((40, 256, 304))
        plan = ops.f32_waves(m, n, k, units)
        if plan is None:
            assert ops.f32_waves(m, n, k, units, True) is None
            continue
        found.add(plan)
        assert plan in TILES and m <= 1024 and k >= 512 and 16 * (plan[1] - 1) < m and ops.f32_wide(m, n, k, units) == 0
        assert (n + 256) * k < 1 << 30 and (m + 256) * k < 1 << 30  # (the entry point's limit: offsets of 32 bits)
        # the norm that would add the others' runs only makes those better
        assert ops.f32_waves(m, n, k, units, True) in (plan, None)
    assert len(found) > 10
    assert ops.f32_waves(225, 4096, 1000, 256) is None and ops.f32_waves(225, 4096, 480, 256) is None and ops.f32_waves(40, 1 << 20, 4096, 256) is None


@pytest.mark.parametrize("m,n,k", [(8, 261888, 4096), (8, 130816, 8192), (300, 261888, 4096)])
def test_matrices_whose_last_offset_is_one_too_many(m, n, k):
    assert (n + 256) * k == 1 << 30 and ops.f32_waves(m, n, k, 256) is None
    assert ops.f32_waves(m, n - 16, k, 256) is not None or m > 16


@pytest.mark.parametrize("rows_a,rows_w,ld_a,ld_w", [(256, 1024, 1 << 21, 1024), (256, 768, 1024, 1 << 20), (256, 1024, (1 << 21) - 4, 1024)])
def test_rows_whose_last_offset_is_one_too_many(rows_a, rows_w, ld_a, ld_w, monkeypatch):
    """Strided rows that reach the limit go to the kernels behind, one stride less does not."""
    called = []

    class Library:
        def __getattr__(self, name):
            return lambda *args: called.append(name) or 0

    monkeypatch.setattr(ops, "core", Library)
    monkeypatch.setattr(ops, "_stream", lambda: None)
    a, w = (torch.empty_strided((rows, 1024), (ld, 1), device="meta") for rows, ld in ((rows_a, ld_a), (rows_w, ld_w)))
    assert ops.f32_waves(rows_a, rows_w, 1024, 256) is not None
    ops._f32_product(a, w, torch.empty((rows_a, rows_w), device="meta"), rows_w, False)
    over = max((rows_a + 256) * ld_a, (rows_w + 256) * ld_w) > 0xFFFFFFFF // 4
    assert called == (["rl_gemm_f32"] if over else ["rl_gemm_f32_runs"]) and over == (ld_a != (1 << 21) - 4)


def test_what_the_entry_points_refuse():
    """Rows that begin inside a unit of 16 bytes, sums that are no whole chunks, offsets beyond 32 bits, tiles that there are not: an
    error before anything is launched."""
    lib, at = ops.core(), 1 << 20  # (addresses that nothing reads)
    good = dict(A=at, W=at, C=at, M=8, N=64, K=512, lda=512, ldw=512, ldc=64, nt=1, mt=1)
    changes = [dict(A=at + 4), dict(W=at + 8), dict(lda=513), dict(ldw=514), dict(K=500), dict(lda=508), dict(N=(1 << 21) - 256),
               dict(ldw=1 << 22), dict(lda=1 << 23, M=24), dict(nt=5), dict(mt=0), dict(A=0), dict(ldc=63)]
    for entry in (lib.rl_gemm_f32_runs, lib.rl_gemm_f32_runs_gated):
        for change in changes:
            assert entry(*(v if name in ("M", "N", "K", "lda", "ldw", "ldc", "nt", "mt") else ctypes.c_void_p(v) for name, v in {**good, **change}.items()), None) == 1, change


# One chunk (seven waves without), runs of unlike length, fewer chunks than are asked for ahead and more; rows and columns that
# end inside a tile of 16 and a workgroup's; several tiles on both sides; strided rows.  Elements that the pieces cannot hold.
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(1, 1, 32), (17, 97, 64), (81, 200, 288), (65, 193, 1056), (130, 259, 4128)])
@pytest.mark.parametrize("tile", TILES)
def test_kernel(m, n, k, tile):
    gen = torch.Generator().manual_seed(m + k)
    lib, p, gap = ops.core(), ops._p, 4
    a, w, w2 = (torch.randn(r, k + gap, generator=gen) * torch.exp2(torch.randint(-5, 6, (r, k + gap), generator=gen)) for r in (m, n, 2 * n))
    a[m // 2, k // 2], w[n - 1, k - 1], w2[n + n // 2, 0] = float("inf"), 2.0**104, -(2.0**110)
    a[:, k:] = w[:, k:] = w2[:, k:] = float("nan")  # what lies between the rows
    a, w, w2 = (t.cuda()[:, :k] for t in (a, w, w2))
    want, out = torch.empty((m, n), device="cuda"), torch.full((m + 1, n + 1), 7.0, device="cuda")
    assert lib.rl_gemm_f32(p(a), p(w), p(want), None, m, n, k, k + gap, k + gap, n, 64, 1, ops._stream()) == 0
    assert lib.rl_gemm_f32_runs(p(a), p(w), p(out), m, n, k, k + gap, k + gap, n + 1, *tile, ops._stream()) == 0
    assert bool((out[m] == 7.0).all()) and bool((out[:, n] == 7.0).all())
    torch.testing.assert_close(out[:m, :n], want, rtol=0, atol=0, equal_nan=True)
    out.fill_(7.0)
    assert lib.rl_gemm_f32_gated(p(a), p(w2), p(want), None, m, n, k, k + gap, k + gap, n, 64, 1, ops._stream()) == 0
    assert lib.rl_gemm_f32_runs_gated(p(a), p(w2), p(out), m, n, k, k + gap, k + gap, n + 1, *tile, ops._stream()) == 0
    assert bool((out[m] == 7.0).all()) and bool((out[:, n] == 7.0).all())
    torch.testing.assert_close(out[:m, :n], want, rtol=0, atol=0, equal_nan=True)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(8, 1024, 2048), (40, 1536, 512), (225, 1024, 2048)])
def test_operands_that_it_does_not_take(m, n, k):
    """Rows that begin inside a unit of 16 bytes go where they went, with the same bits; so do contiguous ones in each form."""
    assert ops.f32_waves(m, n, k, ops.chip().units) is not None
    gen = torch.Generator().manual_seed(m)
    a, w = torch.randn(m, k, generator=gen).cuda(), torch.randn(n, k, generator=gen).cuda()
    first = torch.empty((m, n), device="cuda")
    ops.gemm_f32(a, w, first)
    bound = (a.double().abs() @ w.double().abs().T) * (2 * (6 * -(-k // 256) + 8) + 2) * 2.0**-24  # additions a sum, as the tiles'
    assert bool(((first.double() - a.double() @ w.double().T).abs() <= bound).all())
    for shift, gap in ((1, 0), (0, 1), (2, 2)):
        moved = []
        for t in (a, w):
            flat = torch.full((t.shape[0] * (k + gap) + shift,), float("nan"), device="cuda")
            moved.append(flat[shift:].view(-1, k + gap)[:, :k])
            moved[-1].copy_(t)
        out = torch.empty_like(first)
        ops.gemm_f32(*moved, out)
        assert torch.equal(out, first)


# What is asked for ahead of a wave's last chunk is not there: operands that end with their memory, where the last wave's run ends
# with the rows (64 chunks), where it is shorter than the others' (61) and where waves have none (3).
@pytest.mark.gpu
@pytest.mark.parametrize("k", [2048, 1952, 96])
@pytest.mark.parametrize("tile", [(1, 1), (1, 2), (6, 1), (4, 5)])
def test_operands_that_end_with_their_memory(tile, k):
    m, n = 37, 150
    lib, p = ops.core(), ops._p
    gen = torch.Generator().manual_seed(k)

    def at_the_end(rows):
        held = torch.empty(24 << 20, dtype=torch.uint8, device="cuda")  # (an allocation of its own, whole pages of 2 MB)
        t = held[held.numel() - rows * k * 4 :].view(torch.float32).view(rows, k)
        return t.copy_(torch.randn(rows, k, generator=gen))

    for gated in (False, True):
        a, w = at_the_end(m), at_the_end(2 * n if gated else n)
        want, out = torch.empty((m, n), device="cuda"), torch.empty((m, n), device="cuda")
        entry, runs = (lib.rl_gemm_f32_gated, lib.rl_gemm_f32_runs_gated) if gated else (lib.rl_gemm_f32, lib.rl_gemm_f32_runs)
        assert entry(p(a), p(w), p(want), None, m, n, k, k, k, n, 64, 1, ops._stream()) == 0
        assert runs(p(a), p(w), p(out), m, n, k, k, k, n, *tile, ops._stream()) == 0
        assert torch.equal(out, want)
