"""Axis-0 reductions at the edges of their launch forms: the shortest axis that
is split, one-launch blocks of 64 and of 256 outputs, column tiles with a fold
of few and of many outputs, and column counts of every remainder of 4.
Integers, min, max and argmax are compared bit for bit with numpy, f32 sums
within 2*ceil(log2 n)*eps*sum|terms|."""
from __future__ import annotations

import numpy as np
import pytest

import hephaestus_amd as hx
from hephaestus_amd import Layout, StridedView

pytestmark = pytest.mark.gpu

AXIS = hx.RocmAxisReductionOps()

# (lines, columns, distance between lines, offset of line 0)
VIEWS = [(32, 9, 9, 0), (33, 4, 4, 0), (33, 5, 5, 0), (34, 7, 9, 2), (200, 3, 3, 0), (64, 64, 64, 0), (65, 66, 67, 1),
         (1023, 97, 97, 0), (1024, 195, 195, 0), (1025, 198, 200, 3), (2000, 261, 261, 0), (4096, 101, 101, 0),
         (4097, 103, 103, 0), (300, 1023, 0, 5), (40, 49151, 49151, 0), (40, 49153, 49155, 1), (512, 65540, 65540, 0),
         (513, 65537, 65537, 0), (1100, 8199, 8199, 0), (1030, 10239, 10239, 0), (1030, 10241, 10241, 0),
         (4100, 10242, 10242, 0), (97, 1000, -1003, 96 * 1003), (33, 524290, 524290, 0)]


@pytest.mark.parametrize("lines,cols,pitch,offset", VIEWS)
def test_column_reductions(device, oracle, lines, cols, pitch, offset):
    size = offset + max(0, (lines - 1) * pitch) + cols
    lay = Layout.try_new([lines, cols], [pitch, 1], offset)
    at = np.lib.stride_tricks.as_strided

    def view(x):
        return at(x[offset:], (lines, cols), (4 * pitch, 4))

    def reduced(op, x, dtype):
        out = device.alloc_zeroed(dtype, cols)
        AXIS.reduce_axis_into(device, op, StridedView(x, lay), 0, StridedView(out, Layout.c_contiguous([1, cols])))
        return device.download_owned(out)

    i = oracle.uniform_int(size, seed=lines + cols, lo=-50, hi=50, dtype=np.int32)
    iv, ib = view(i), device.upload(i)
    assert np.array_equal(reduced(hx.SumOp, ib, np.int32), iv.sum(axis=0, dtype=np.int32))
    assert np.array_equal(reduced(hx.MinOp, ib, np.int32), iv.min(axis=0))
    assert np.array_equal(reduced(hx.ArgMaxOp, ib, np.uint32), iv.argmax(axis=0))  # many ties: the first wins
    f = oracle.uniform_real(size, seed=lines, lo=-1.0, hi=1.0)
    fv, fb = view(f), device.upload(f)
    exact = fv.sum(axis=0, dtype=np.float64)
    bound = 2 * max(1, (lines - 1).bit_length()) * 2.0**-23 * np.abs(fv).sum(axis=0, dtype=np.float64)
    got = reduced(hx.SumOp, fb, np.float32)
    assert np.all(np.abs(got - exact) <= bound + 2.0**-24 * np.abs(exact))
    assert np.array_equal(got, reduced(hx.SumOp, fb, np.float32))
    f[offset + (lines // 2) * pitch + cols - 1] = np.nan  # the last column's, from the middle line
    fv, fb = view(f), device.upload(f)
    got = reduced(hx.SumOp, fb, np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(fv.sum(axis=0)))
    assert np.array_equal(reduced(hx.MaxOp, ib, np.int32), iv.max(axis=0))
