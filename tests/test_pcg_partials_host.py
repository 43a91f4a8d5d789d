"""Partial rows of the generic PCG's vector passes, from their workspace size (CPU).

Every block of an update reads all partials of its batch, so launches of many blocks hold them below the values a block
reads: past 2048 blocks a thread takes four values or more, and a launch has no more blocks than values / 1024.
"""
import pytest

from pgj import _lib


@pytest.mark.parametrize('B, n', [(1, 3000), (1, 262144), (1, 3000000), (2, 262144), (3, 331776), (6, 98304),
                                  (6, 262144), (16, 262144), (64, 98304), (1024, 3000), (4096, 300), (65535, 1)])
def test_partials_per_launch(B, n):
    doubles = _lib.lib().pgj_pcg_ws_bytes(B, n) // 8
    rows = (doubles - 2 * B - 1) // (3 * B)      # rounded down over the padding to 256 bytes
    least = min((n + 1023) // 1024, 1024)
    assert rows >= least
    if B * min((n + 255) // 256, 1024) > 2048:
        assert rows <= least + 32 // (3 * B)
