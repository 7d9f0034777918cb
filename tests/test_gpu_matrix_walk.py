"""Full reductions, dots and norms of matrices whose rows lie apart (slices,
padded, reversed and repeated rows): every row-end remainder, rows of one to
many 16-byte units, and from a few elements to several whole trips of every
thread.  Integers, min, max and argmax are compared bit for bit with numpy,
f32 sums within 2*ceil(log2 n)*eps*sum|terms|."""
from __future__ import annotations

import numpy as np
import pytest

import hephaestus_amd as hx
from hephaestus_amd import Layout, StridedView

pytestmark = pytest.mark.gpu

FULL = hx.RocmFullReductionOps()
ONE = Layout.c_contiguous([1])


def close(got, terms):
    terms = np.asarray(terms, np.float64)
    bound = 2 * max(1, (terms.size - 1).bit_length()) * 2.0**-23 * np.abs(terms).sum()
    return abs(float(got) - terms.sum()) <= bound + 2.0**-24 * abs(terms.sum())


# (rows, cols, distance between rows, offset of row 0)
VIEWS = [(3, 4, 5, 0), (2, 5, 9, 3), (5, 6, 6 + 2, 1), (7, 7, 10, 2), (40, 8, 11, 1), (1000, 9, 9 + 4, 0), (3, 4097, 4100, 1),
         (517, 130, 131, 5), (2049, 259, 300, 1), (700, 4094, 4096, 4097), (100000, 19, 23, 2), (11, 6, -8, 80), (9, 6, 0, 1),
         (1, 1000003, 7, 1)]


@pytest.mark.parametrize("rows,cols,pitch,offset", VIEWS)
def test_matrix_views(device, oracle, rows, cols, pitch, offset):
    size = offset + max(0, (rows - 1) * pitch) + cols
    lay = Layout.try_new([rows, cols], [pitch, 1], offset)
    at = offset + np.arange(rows)[:, None] * pitch + np.arange(cols)

    def reduced(op, x, dtype, prologue=None):
        out = device.alloc_zeroed(dtype, 1)
        FULL.reduce_full_into(device, op, StridedView(device.upload(x), lay), StridedView(out, ONE), prologue=prologue)
        return device.download_owned(out)[0]

    def argmax(x):
        index, value = device.alloc_zeroed(np.uint32, 1), device.alloc_zeroed(x.dtype, 1)
        FULL.argmax_full_into(device, StridedView(device.upload(x), lay), index, value)
        return device.download_owned(index)[0], device.download_owned(value)[0]

    f = oracle.uniform_real(size, seed=rows, lo=-1.0, hi=1.0)
    g = oracle.uniform_real(size, seed=cols, lo=-1.0, hi=1.0)
    i = oracle.uniform_int(size, seed=rows + cols, lo=-1000, hi=1000, dtype=np.int32)
    u = oracle.uniform_int(size, seed=rows + 7, lo=0, hi=2**32 - 1)
    fv, gv, iv, uv = f[at], g[at], i[at], u[at]
    assert close(reduced(hx.SumOp, f, np.float32), fv)
    assert close(reduced(hx.SumOp, f, np.float32, prologue=(0.5, 0.25)), fv.astype(np.float64) * 0.5 + 0.25)
    assert reduced(hx.SumOp, i, np.int32) == iv.sum(dtype=np.int32)
    assert reduced(hx.ProdOp, u | 1, np.uint32) == np.multiply.reduce((uv | 1).ravel(), dtype=np.uint32)
    assert reduced(hx.MinOp, i, np.int32) == iv.min() and reduced(hx.MaxOp, u, np.uint32) == uv.max()
    for x, v in ((f, fv), (i % 5, iv % 5)):  # many ties among the latter: the first wins
        index, value = argmax(x)
        assert index == np.argmax(v.ravel()) and value == v.max()
    a, b = StridedView(device.upload(f), lay), StridedView(device.upload(g), lay)
    assert close(device.download_owned(hx.dot(device, a, b))[0], fv.astype(np.float64) * gv)
    assert close(device.download_owned(hx.norm_l1(device, a))[0], np.abs(fv))
    assert np.isclose(device.download_owned(hx.norm_l2(device, a))[0], np.linalg.norm(fv.astype(np.float64)), rtol=1e-6)
    assert device.download_owned(hx.norm_max(device, a))[0] == np.abs(fv).max()
    w = StridedView(device.upload(u), lay)
    assert device.download_owned(hx.dot(device, w, w))[0] == np.multiply(uv, uv).sum(dtype=np.uint32)


def test_dot_of_matrices_with_rows_at_different_distances(device, oracle):
    rows, cols = 333, 1001
    x = oracle.uniform_real(rows * 1003 + 8, seed=1, lo=-1.0, hi=1.0)
    y = oracle.uniform_real(rows * 1200, seed=2, lo=-1.0, hi=1.0)
    a, b = Layout.try_new([rows, cols], [1003, 1], 3), Layout.try_new([rows, cols], [-1200, 1], (rows - 1) * 1200 + 5)
    xv = x[3:3 + rows * 1003].reshape(rows, 1003)[:, :cols].astype(np.float64)
    yv = y.reshape(rows, 1200)[::-1, 5:5 + cols]
    got = device.download_owned(hx.dot(device, StridedView(device.upload(x), a), StridedView(device.upload(y), b)))[0]
    assert close(got, xv * yv)


@pytest.mark.parametrize("special", [np.nan, np.inf, -np.inf])
def test_special_values_at_a_row_end_are_taken_once_and_only_inside(device, special):
    """The last unit of a row re-reads up to three elements of the unit before
    it; the padding around the rows holds values that must not be seen."""
    rows, cols, pitch = 50, 1001, 1004
    x = np.full(rows * pitch, np.float32(3e38))
    inside = x.reshape(rows, pitch)[:, :cols]
    inside[:] = 1.0
    inside[7, 997:] = [2.0, 3.0, special, 5.0]
    lay = Layout.try_new([rows, cols], [pitch, 1], 0)
    out = device.alloc_zeroed(np.float32, 1)
    FULL.reduce_full_into(device, hx.SumOp, StridedView(device.upload(x), lay), StridedView(out, ONE))
    got, want = device.download_owned(out)[0], inside.sum(dtype=np.float64)
    assert np.array_equal(got, np.float32(want), equal_nan=True)
    index, value = device.alloc_zeroed(np.uint32, 1), device.alloc_zeroed(np.float32, 1)
    FULL.argmax_full_into(device, StridedView(device.upload(x), lay), index, value)
    at = 7 * cols + (999 if special == np.inf else 1000)
    assert device.download_owned(index)[0] == at and device.download_owned(value)[0] == inside.ravel()[at]
