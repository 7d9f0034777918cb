"""Scans of few lines of more than 2048 elements, which run in tiles of 2048,
4096 or 8192 elements up to 10 * 2^20 elements: the edges of tiles, of
superblocks (64 tiles) and of each tile size's range, one line and several,
and outputs off the 128-byte grid.  Integers bit for bit against the oracle,
f32 within 2*ceil(log2 n)*eps*prefix(|x|); lines of at most 64 tiles also
reproduce their f32 bits."""
from __future__ import annotations

import numpy as np
import pytest

import hephaestus_amd as hx
from hephaestus_amd import Layout, StridedView

from test_gpu_fallbacks import wait_limits

pytestmark = pytest.mark.gpu

SCAN = hx.RocmScanOps()


def run(device, x, lines, exclusive, reverse, out_off=0, op=hx.CumSumOp):
    n = x.size // lines
    buf, out = device.upload(x), device.upload(np.full(x.size + out_off, 7, x.dtype))
    lay = Layout.try_new([lines, n], [n, 1], 0)
    SCAN.scan_axis_into(device, op, StridedView(buf, lay), 1,
                        hx.ScanDirection.Reverse if reverse else hx.ScanDirection.Forward,
                        StridedView(out, Layout.try_new([lines, n], [n, 1], out_off)),
                        hx.ScanKind.Exclusive if exclusive else hx.ScanKind.Inclusive)
    got = device.download_owned(out)
    assert np.all(got[:out_off] == 7)
    return got[out_off:].reshape(lines, n)


MID = [(1, 2049), (1, 4096), (1, 32769), (1, (1 << 17) - 1), (1, (1 << 17) + 1), (1, 64 * 4096), (1, 64 * 4096 + 1),
       (1, 1 << 22), (1, (1 << 22) + 5), (1, 1 << 23), (1, (1 << 23) + 3), (1, (10 << 20) + 1), (3, 5001),
       (60, 2051), (255, 4099), (256, 4099), (7, 40000), (40, 262145)]


@pytest.mark.parametrize("exclusive,reverse,out_off", [(False, False, 0), (True, True, 0), (True, False, 3)])
@pytest.mark.parametrize("lines,n", MID)
def test_mid_scan(device, oracle, lines, n, exclusive, reverse, out_off):
    x = oracle.uniform_int(lines * n, seed=n, lo=0, hi=2**32 - 1)
    want = np.stack([oracle.scan_sum(l, exclusive=exclusive, reverse=reverse) for l in x.reshape(lines, n)])
    assert np.array_equal(run(device, x, lines, exclusive, reverse, out_off), want)
    f = oracle.uniform_real(lines * n, seed=n + 1, lo=-1.0, hi=1.0)
    got = run(device, f, lines, exclusive, reverse, out_off)
    for g, l in zip(got, f.reshape(lines, n)):
        ref, ab = oracle.scan_sum(l, exclusive=exclusive, reverse=reverse)
        assert oracle.check_f32_bound(g, ref, ab, n)[0] == 0
    if n <= 64 * 2048:  # at most 64 tiles a line, whatever the tile
        again = run(device, f, lines, exclusive, reverse, out_off)
        assert np.array_equal(again.view(np.uint32), got.view(np.uint32))


@pytest.mark.parametrize("limits", [(0, 0), (1, 1)])
@pytest.mark.parametrize("lines,n", [(1, 100003), (1, 300001), (9, 20001), (1, (1 << 22) + 7)])
def test_mid_scan_under_forced_fallbacks(device, oracle, limits, lines, n):
    x = oracle.uniform_int(lines * n, seed=n, lo=0, hi=2**32 - 1)
    f = oracle.uniform_real(lines * n, seed=n + 1, lo=0.0, hi=1.0)
    with wait_limits(*limits):
        got, got_f = run(device, x, lines, True, False), run(device, f, lines, False, True)
        prod = run(device, x, lines, False, False, op=hx.CumProdOp)
    x, f = x.reshape(lines, n), f.reshape(lines, n)
    assert np.array_equal(got, np.stack([oracle.scan_sum(l, exclusive=True) for l in x]))
    assert np.array_equal(prod, np.multiply.accumulate(x, axis=1, dtype=np.uint32))
    for g, l in zip(got_f, f):
        ref, ab = oracle.scan_sum(l, exclusive=False, reverse=True)
        assert oracle.check_f32_bound(g, ref, ab, n)[0] == 0


# Short dense lines (fewer than 256 elements) run as one flat range in tiles
# of 2048 elements up to 2^22 (2^25 for lines of at most 48), 4096 beyond:
# lines that end at, straddle and exceed tile edges, and a partial last tile.
@pytest.mark.parametrize("exclusive,reverse", [(False, False), (True, True)])
@pytest.mark.parametrize("dtype", [np.uint32, np.float32])
@pytest.mark.parametrize("lines,n", [(8, 255), (9, 255), (32, 64), (33, 64), (2048, 1), (683, 3), (41, 100), (16451, 255),
                                     (87383, 48), (85600, 49), (41944, 100), (699052, 48), (684786, 49)])
def test_short_line_tiles(device, oracle, lines, n, dtype, exclusive, reverse):
    x = (oracle.uniform_int(lines * n, seed=n, lo=0, hi=2**32 - 1) if dtype == np.uint32
         else oracle.uniform_real(lines * n, seed=n, lo=-1.0, hi=1.0))
    got = run(device, x, lines, exclusive, reverse)
    x = x.reshape(lines, n)[:, ::-1 if reverse else 1]
    want = np.add.accumulate(x, axis=1, dtype=np.uint32 if dtype == np.uint32 else np.float64)
    bound = 2 * max(1, (n - 1).bit_length()) * 2.0**-23 * np.add.accumulate(np.abs(x), axis=1, dtype=np.float64)
    if exclusive:
        want, bound = (np.concatenate([np.zeros((lines, 1), a.dtype), a[:, :-1]], axis=1) for a in (want, bound))
    want, bound = (a[:, ::-1 if reverse else 1] for a in (want, bound))
    assert np.array_equal(got, want) if dtype == np.uint32 else np.all(np.abs(got - want) <= bound)
