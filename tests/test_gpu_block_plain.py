"""The many-row product stored as bfloat16: every tile at its edges against 64 bits, and the products that a layer of a small
model runs instead of the library's."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _bound(x, w):
    """Of a product summed in float32 in any order and rounded to bfloat16."""
    a, b = x.double().abs(), w.double().abs()
    size = a @ b.t().contiguous()
    return (x.shape[1] * 2.0**-24) * size * (1 + 2.0**-8), 2.0**-8


@pytest.mark.parametrize("tile", [(4, 4), (3, 4), (2, 4), (4, 2), (3, 2), (2, 2), (2, 1)])
@pytest.mark.parametrize("m,n,k", [(65, 8, 64), (64, 128, 128), (129, 200, 192), (256, 256, 640), (257, 264, 1024), (511, 1032, 320), (1000, 776, 2048)])
def test_every_tile(tile, m, n, k):
    from rapid_llm_amd.kernels import ops

    gen = torch.Generator(device="cuda").manual_seed(m * n + k)
    x = torch.randn(m, k, generator=gen, device="cuda").to(torch.bfloat16)
    w = torch.randn(n, k, generator=gen, device="cuda").to(torch.bfloat16)
    whole = torch.full((m + 8, n), 7.0, dtype=torch.bfloat16, device="cuda")
    out = whole[:m]
    ops._block(x, w, out, "plain", (*tile, 1))
    want = x.double() @ w.double().t().contiguous()
    absolute, relative = _bound(x, w)
    assert bool(((out.double() - want).abs() <= absolute + relative * want.abs()).all())
    assert bool((whole[m:] == 7.0).all())  # nothing behind the last row


def test_special_values_stay_in_their_rows_and_columns():
    from rapid_llm_amd.kernels import ops

    x = torch.ones(300, 256, dtype=torch.bfloat16, device="cuda")
    w = torch.ones(264, 256, dtype=torch.bfloat16, device="cuda")
    x[17, 3] = float("nan")
    w[260, 100] = float("inf")
    out = ops._block(x, w, torch.empty(300, 264, dtype=torch.bfloat16, device="cuda"), "plain", (3, 4, 1))
    rows = torch.ones(300, dtype=torch.bool, device="cuda")
    rows[17] = False
    assert bool(out[17].isnan().all()) and bool((out[rows][:, 260] == float("inf")).all())
    cols = torch.ones(264, dtype=torch.bool, device="cuda")
    cols[260] = False
    assert bool((out[rows][:, cols] == 256).all())


@pytest.mark.parametrize("m", [193, 256, 320, 321, 512, 513, 700, 1024, 1536])
def test_layers_of_a_small_model_call_no_library(m):
    from rapid_llm_amd.kernels import ops

    gen = torch.Generator(device="cuda").manual_seed(m)
    with ops.own_products():
        _small_layers(m, gen)


def _small_layers(m, gen):
    from rapid_llm_amd.kernels import ops
    from rapid_llm_amd.parts.lazy import DeferredProduct
    from rapid_llm_amd.parts.linear import Linear

    for n, k, folded in ((4096, 1024, False), (1024, 2048, True), (1024, 3072, True)):
        linear = Linear(k, n)
        linear.bind(torch.randn(n, k, generator=gen, device="cuda").to(torch.bfloat16))
        x = torch.randn(m, k, generator=gen, device="cuda").to(torch.bfloat16)
        assert not linear.calls_library(m, folded)
        before = ops.library_products
        if folded:
            y = linear.deferred(x)
            assert isinstance(y, DeferredProduct) and linear.midsize(x)
            got = linear.partial_sums(x).double().sum(0)
        else:
            got = linear(x).double()
        assert ops.library_products == before
        want = x.double() @ linear.weight.double().t().contiguous()
        absolute, relative = _bound(x, linear.weight)
        assert bool(((got - want).abs() <= absolute + relative * want.abs()).all())
