"""Strip column scans: many lines adjacent in memory, scanned in strips of 32
or 64 lines cut into chunks of 224 to 896 rows, with a look-back over each
strip's chunks.  Shapes stand at the edges of chunks (448 and 896 rows at up
to 32 lines, 224 and 448 above), of strips (a last strip of one line, lane
vectors that overlap) and of each way blocks are dealt to XCDs.  Integers are
compared bit for bit with numpy's wrapped scans, f32 with an f64 scan within
2*ceil(log2 n)*eps*prefix(|x|)."""
from __future__ import annotations

import numpy as np
import pytest

import hephaestus_amd as hx
from hephaestus_amd import Layout, StridedView, _ffi

from test_gpu_fallbacks import wait_limits

pytestmark = pytest.mark.gpu

SCAN = hx.RocmScanOps()


def _numpy_scan(x, prod, exclusive, reverse):
    x = x[::-1] if reverse else x
    y = (np.multiply if prod else np.add).accumulate(x, axis=0, dtype=x.dtype)
    if exclusive:
        y = np.concatenate([np.full((1, x.shape[1]), 1 if prod else 0, y.dtype), y[:-1]])
    return y[::-1] if reverse else y


def check(device, oracle, rows, cols, dtype, seed, pitch=None, offset=0, prod=False, exclusive=False, reverse=False,
          noalloc=False):
    pitch = pitch or cols
    n = offset + rows * pitch
    if dtype == np.float32:
        host = oracle.uniform_real(n, seed, *((0.999, 1.001) if prod else (-1.0, 1.0)))
    else:
        host = oracle.uniform_int(n, seed, 0, 2**32 - 1).view(dtype)
    lay = Layout.try_new([rows, cols], [pitch, 1], offset)
    x, out = device.upload(host), device.upload(np.full(n, 7, dtype))
    scan = SCAN.scan_axis_into_noalloc if noalloc else SCAN.scan_axis_into
    scan(device, hx.CumProdOp if prod else hx.CumSumOp, StridedView(x, lay), 0,
         hx.ScanDirection.Reverse if reverse else hx.ScanDirection.Forward, StridedView(out, lay),
         hx.ScanKind.Exclusive if exclusive else hx.ScanKind.Inclusive)
    got = device.download_owned(out)
    assert np.all(got[:offset] == 7)
    got = got[offset:].reshape(rows, pitch)
    assert np.all(got[:, cols:] == 7)
    got, values = got[:, :cols], host[offset:].reshape(rows, pitch)[:, :cols]
    if dtype != np.float32:
        assert np.array_equal(got, _numpy_scan(values.view(np.uint32), prod, exclusive, reverse).view(dtype))
        return
    want = _numpy_scan(values.astype(np.float64), prod, exclusive, reverse)
    eps = 2.0**-23
    if prod:  # gamma_n of n rounded factors, relative
        bound = rows * eps / (1 - rows * eps) * np.abs(want)
    else:
        bound = 2 * max(1, (rows - 1).bit_length()) * eps * _numpy_scan(np.abs(values).astype(np.float64), False,
                                                                       exclusive, reverse) + eps * np.abs(want)
    assert np.all(np.abs(got - want) <= bound)


# (rows, cols): chunk edges of both widths, strips whose lines are no multiple
# of 4 or that end in one line, chunks dealt to XCDs (32 chunks and more,
# shared lines), strips dealt to XCDs (16 strips and more), whole lines stored
# through the L2 (2^24 elements and more), 16 rows a lane (past 65536 rows).
SHAPES = [(447, 32), (448, 32), (449, 31), (223, 64), (224, 64), (225, 65), (1, 40), (2, 25), (700, 33), (900, 47),
          (500, 66), (300, 127), (300, 129), (460, 257), (230, 4097), (7200, 70), (7300, 130), (1000, 1030),
          (7300, 515), (1 << 17, 132), (1 << 17, 160), (65537, 64), (70001, 30), (66000, 100), (66000, 520)]


@pytest.mark.parametrize("dtype", [np.uint32, np.float32])
@pytest.mark.parametrize("rows,cols", SHAPES)
def test_strip_scan(device, oracle, rows, cols, dtype):
    check(device, oracle, rows, cols, dtype, seed=rows + cols)


@pytest.mark.parametrize("prod", [False, True])
@pytest.mark.parametrize("exclusive,reverse", [(True, False), (False, True), (True, True)])
@pytest.mark.parametrize("dtype", [np.int32, np.float32])
@pytest.mark.parametrize("rows,cols,pitch,offset", [(449, 32, 32, 0), (451, 33, 40, 3), (7300, 66, 67, 1),
                                                    (1000, 1030, 1030, 0), (230, 4097, 4100, 5)])
def test_strip_scan_kinds_and_padded_rows(device, oracle, rows, cols, pitch, offset, dtype, exclusive, reverse, prod):
    check(device, oracle, rows, cols, dtype, seed=rows + offset, pitch=pitch, offset=offset, prod=prod,
          exclusive=exclusive, reverse=reverse)


# Every chunk's look-back totals its missing predecessors from the input.
@pytest.mark.parametrize("limits", [(0, 0), (1, 1)])
@pytest.mark.parametrize("dtype", [np.uint32, np.float32])
@pytest.mark.parametrize("rows,cols,reverse", [(1400, 32, False), (1200, 66, True), (900, 257, False)])
def test_strip_scan_under_forced_fallbacks(device, oracle, limits, dtype, rows, cols, reverse):
    with wait_limits(*limits):
        check(device, oracle, rows, cols, dtype, seed=rows, reverse=reverse, exclusive=reverse)


# f32 values over 46 powers of two, the second half of the rows the negated
# first in another order, so that the last outputs are what the f64 sums
# rounded: any other order of the chunk totals shows in the bits.
def _rounding_sensitive(rows, cols, pitch, offset):
    rng = np.random.default_rng(rows + cols)
    half = rows // 2
    x = np.zeros((rows, pitch), np.float32)
    x[:half] = (rng.uniform(-1, 1, (half, pitch)) * np.exp2(rng.integers(0, 46, (half, pitch)))).astype(np.float32)
    x[half:2 * half] = -x[rng.permutation(half)]
    return np.concatenate([np.zeros(offset, np.float32), x.ravel()])


@pytest.mark.parametrize("rows,cols,pitch,offset,exclusive,reverse", [
    (8_192, 32, 32, 0, False, False), (7_001, 45, 47, 3, True, False), (50_000, 64, 64, 0, False, True),
    (60_000, 100, 100, 0, True, True), (8_193, 255, 255, 1, False, False), (700_000, 33, 33, 0, False, True),
    (400_000, 64, 64, 0, True, False), (200_000, 130, 131, 0, False, False)])
def test_f32_strips_below_256_lines_give_the_same_bits_in_every_run(device, oracle, rows, cols, pitch, offset, exclusive, reverse):
    lay = Layout.try_new([rows, cols], [pitch, 1], offset)
    x = device.upload(_rounding_sensitive(rows, cols, pitch, offset))
    out = device.alloc_zeroed(np.float32, offset + rows * pitch)

    def run():
        SCAN.scan_axis_into(device, hx.CumSumOp, StridedView(x, lay), 0,
                            hx.ScanDirection.Reverse if reverse else hx.ScanDirection.Forward, StridedView(out, lay),
                            hx.ScanKind.Exclusive if exclusive else hx.ScanKind.Inclusive)
        return device.download_owned(out).view(np.uint32)

    first = run()
    for _ in range(10):
        assert np.array_equal(run(), first)
    for limits in ((0, 0), (1, 1)):  # waiters total missing chunks themselves
        with wait_limits(*limits):
            assert np.array_equal(run(), first), limits


# Taken by the fixed scratch, but with more status words than it holds as
# strips are first cut: [94200, 1279] takes longer chunks, the others several
# launches, each from the totals of the one before.  Rows at multiples of
# `every` hold column mod 7 + 1, all others 0.
@pytest.mark.parametrize("rows,cols,dtype,exclusive,reverse", [
    (94_200, 1279, np.float32, False, False), (4_000_003, 64, np.float32, False, False),
    (3_600_001, 65, np.float32, True, True), (7_400_000, 64, np.uint32, False, False)])
def test_noalloc_scan_whose_strips_exceed_the_scratch(device, rows, cols, dtype, exclusive, reverse):
    every = 100_000 if rows > 1_000_000 else 3_000
    assert _ffi.lib().hx_noalloc_scratch_bytes() == 8 << 20
    lay = Layout.c_contiguous([rows, cols])
    x, out = device.alloc_zeroed(dtype, rows * cols), device.alloc_zeroed(dtype, rows * cols)
    weight = (np.arange(cols) % 7 + 1).astype(dtype)
    for r in range(0, rows, every):
        device.write_sub_buffer(x, r * cols, weight)
    SCAN.scan_axis_into_noalloc(device, hx.CumSumOp, StridedView(x, lay), 0,
                                hx.ScanDirection.Reverse if reverse else hx.ScanDirection.Forward,
                                StridedView(out, lay), hx.ScanKind.Exclusive if exclusive else hx.ScanKind.Inclusive)
    marks = np.zeros(rows, np.int64)
    marks[::every] = 1
    count = _numpy_scan(marks[:, None], False, exclusive, reverse)[:, 0].astype(dtype)
    got = device.download_owned(out).reshape(rows, cols)
    for c in range(cols):
        assert np.array_equal(got[:, c], count * weight[c]), c
