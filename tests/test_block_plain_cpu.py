"""Where the many-row product stored as bfloat16 runs, and that a layer's answer to "is this the library's?" is what it does."""

import random
import threading

import pytest

from rapid_llm_amd.kernels import ops


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
