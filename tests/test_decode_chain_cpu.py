"""The rules of the launch that runs all layers of a step of few tokens."""

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
