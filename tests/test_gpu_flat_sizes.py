"""Flat full reductions on both sides of the sizes from and to which a thread
keeps four loads in flight, and in the remainders between.  Integers, max and
argmax bit for bit, f32 sums within 2*ceil(log2 n)*eps*sum|x|."""
from __future__ import annotations

import numpy as np
import pytest

import hephaestus_amd as hx
from hephaestus_amd import Layout, StridedView

pytestmark = pytest.mark.gpu

FULL = hx.RocmFullReductionOps()
ONE = Layout.c_contiguous([1])


@pytest.mark.parametrize("n", [(1 << 21) - 1, 1 << 21, (1 << 21) + 5, 5000011, 3 * (1 << 23) + 3, 1 << 26, (1 << 26) + 1])
def test_flat_sizes(device, oracle, n):
    def reduced(op, x, dtype):
        out = device.alloc_zeroed(dtype, 1)
        FULL.reduce_full_into(device, op, StridedView(x, Layout.c_contiguous([n])), StridedView(out, ONE))
        return device.download_owned(out)[0]

    u = oracle.uniform_int(n, seed=n, lo=0, hi=2**32 - 1)
    d = device.upload(u)
    assert reduced(hx.SumOp, d, np.uint32) == u.sum(dtype=np.uint32)
    assert reduced(hx.MaxOp, d, np.uint32) == u.max()
    f = oracle.uniform_real(n, seed=n, lo=-1.0, hi=1.0)
    f[n - 1] = f[n // 3] = 2.0  # the first of two maxima wins
    e = device.upload(f)
    bound = 2 * (n - 1).bit_length() * 2.0**-23 * np.abs(f).sum(dtype=np.float64)
    assert abs(float(reduced(hx.SumOp, e, np.float32)) - f.sum(dtype=np.float64)) <= bound
    index = device.alloc_zeroed(np.uint32, 1)
    FULL.argmax_full_into(device, StridedView(e, Layout.c_contiguous([n])), index)
    assert device.download_owned(index)[0] == n // 3
