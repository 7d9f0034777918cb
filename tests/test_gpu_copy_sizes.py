"""Device copies on both sides of the size from which they move whole tiles,
with every remainder of a 16-byte vector, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TILES_FROM = 48 << 20


@pytest.mark.parametrize("words", [1, 3, 4, 5, 1023, 65536, 65537, (1 << 20) + 2, TILES_FROM // 4 - 1, TILES_FROM // 4,
                                   TILES_FROM // 4 + 1, TILES_FROM // 4 + 65536 + 7])
def test_copies(device, oracle, words):
    host = oracle.uniform_int(words, seed=words, lo=0, hi=2**32 - 1)
    src, dst = device.upload(host), device.alloc_zeroed(np.uint32, words)
    device.copy_buffer(src, dst)
    assert np.array_equal(device.download_owned(dst), host)
    assert np.array_equal(device.download_owned(src), host)
