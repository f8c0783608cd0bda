"""The rules of the launch that runs all layers of a step of few tokens."""

import ctypes

import pytest

from rapid_llm_amd.kernels import decode_chain as chain


def test_sizes():
    family = {"0.6b": (1024, 16, 8, 3072), "1.7b": (2048, 16, 8, 6144), "4b": (2560, 32, 8, 9728), "8b": (4096, 32, 8, 12288)}
    for name, (h, nq, nkv, inter) in family.items():
        for rows in (1, 16):
            assert chain.fits(rows, h, nq, nkv, 128, inter, 16) == (name in ("0.6b", "1.7b"))
        assert chain.fits(2, h, nq, nkv, 128, inter, 16) == (name == "0.6b")
    assert not chain.fits(0, 1024, 16, 8, 128, 3072, 16) and not chain.fits(17, 1024, 16, 8, 128, 3072, 16)
    for sizes in ((1024, 16, 8, 64, 3072, 16), (1024, 16, 8, 128, 3008, 16), (1000, 16, 8, 128, 3072, 16), (1024, 16, 8, 128, 3072, 4),
                  (1024, 15, 8, 128, 3072, 16), (1024, 40, 8, 128, 3072, 16)):
        assert not chain.fits(1, *sizes), sizes


@pytest.mark.parametrize("units", [1, 64, 256, 304])
def test_shares(units):
    for rows in range(1, 17):
        for nkv in (1, 2, 8, 32):
            for span in (1, 255, 256, 257, 4096, 40960, 1 << 20):
                n = chain.shares(rows, nkv, span, units)
                assert 1 <= n <= chain.MAX_SHARES and (n - 1) * chain.MIN_KEYS < span
                assert n == 1 or n * rows * nkv <= units


@pytest.mark.parametrize("layers", [2, 28, 64])
def test_a_flag_speaks_of_its_own_launch_only(layers):
    """Launches of one or two rows write no flags, any number of them: what the flags of the last launch that did say must
    not be taken for this one's, also where a count of phases over all launches would have wrapped."""
    phases = 5 * layers

    def done(flag, launch, ph):
        return chain._library().rl_decode_chain_done(ctypes.c_ulonglong(flag), ctypes.c_uint(launch), ctypes.c_uint(ph))

    wraps = [2**31 // phases, 2**32 // phases, 2**31, 2**32 - 1]
    launches = sorted({max(0, w + d) for w in wraps for d in (-2, -1, 0, 1) if w + d < 2**32 - 1} | {0, 1, 2})
    for launch in launches:
        for ph in (1, phases - 1):
            assert not done(0, launch, ph)  # never written
            for earlier in launches:
                if earlier < launch:
                    assert not done((earlier + 1) << 32 | phases, launch, ph), (earlier, launch)
            for at in range(phases + 1):
                assert done((launch + 1) << 32 | at, launch, ph) == (at >= ph)


def test_indices_that_the_launch_does_not_reach():
    """Divisions by a multiplication are exact below 2^32 / divisor: steps beyond keep their own kernels."""
    sizes = (1024, 16, 8, 3072)
    assert chain.takes(28, 1, *sizes, 256, 16, 4096)
    assert chain.takes(28, 1, *sizes, 8, 16384, 4096) and not chain.takes(28, 1, *sizes, 3, 65536, 4096)  # keys times tokens a page
    wide = (128, 1, 1, 131072)  # 8 k items a layer
    assert chain.takes(8, 1, *wide, 256, 16, 4096) and not chain.takes(80, 1, *wide, 256, 16, 4096)


def test_where_the_launch_is_the_faster_one():
    """Microseconds of both ways, measured: (rows, millions of elements a layer, keys), and whether the launch was the faster."""
    for rows, millions, keys, launch in (
        (1, 15.7, 4096, True), (1, 50.3, 8192, True), (1, 56.8, 512, False), (1, 63.7, 2048, False), (1, 15.7, 16384, True), (1, 15.7, 32768, False),
        (2, 23.2, 1024, True), (2, 28.3, 1024, False), (2, 28.3, 4096, False), (2, 50.3, 1024, False), (4, 19.7, 4096, True), (4, 23.2, 1024, False),
        (4, 63.7, 1024, False), (8, 19.7, 2048, True), (8, 28.3, 1024, False), (8, 15.7, 4096, False), (12, 28.3, 1024, True), (12, 38.5, 1024, False),
        (12, 15.7, 2048, True), (12, 19.7, 2048, False), (12, 15.7, 4096, False), (16, 63.7, 1024, True), (16, 76.0, 1024, False), (16, 28.3, 4096, False),
    ):
        assert chain.faster(rows, int(millions * 1e6), keys) == launch, (rows, millions, keys)
    # more keys or larger layers never bring the launch back
    for rows in range(1, 17):
        for millions in (1, 15, 20, 30, 50, 66):
            answers = [chain.faster(rows, millions * 1000000, 512 << i) for i in range(9)]
            assert answers == sorted(answers, reverse=True) and not answers[-1]
            assert answers[0] or not chain.faster(rows, millions * 1000000 + (8 << 20), 512)
