"""Axis-0 reductions at the edges of the rule that gives a lane four outputs or
one: output counts that are no multiple of 4 around 2^18 at up to 32 lines,
around 2^20 elements, with last groups of 8 and 9 outputs, of 768
lines, and of 640, 10240
and 3 * 2^23 elements beyond 1024 lines.  And more outputs than a launch of blocks
takes."""
from __future__ import annotations

import numpy as np
import pytest

import hephaestus_amd as hx
from hephaestus_amd import Layout, StridedView

import test_gpu_column_blocks as blocks
from test_gpu_large import _slice

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lines,cols,pitch", [
    (17, (1 << 18) - 1, (1 << 18) - 1), (32, (1 << 18) + 1, (1 << 18) + 2), (33, 31_775, 31_775), (33, 31_777, 31_777),
    (257, 73, 75), (257, 72 + 1, 73), (1000, 201, 201), (768, 203, 203), (769, 202, 203), (300, 70, 71), (1025, 11, 13), (5000, 639, 639),
    (5000, 641, 641), (4999, 641, 643), (1100, 10_239, 10_239), (1100, 10_241, 10_241), (195_000, 129, 129),
    (195_200, 130, 131), (300_000, 7, 9)])
def test_outputs_per_lane(device, oracle, lines, cols, pitch):
    blocks.test_column_reductions(device, oracle, lines, cols, pitch, 0)


def test_more_outputs_than_one_launch_of_blocks_takes(device):
    """64 lines that are one line (stride 0) of 2^31 outputs: blocks of 256
    outputs would be 2^32 work-items."""
    outputs, lines = 1 << 31, 64
    x, out = device.alloc_zeroed(np.uint32, outputs), device.alloc_uninitialized(np.uint32, outputs)
    marks = {0: 3, 1: 5, (1 << 30) + 17: 7, outputs - 1: 11}
    for at, value in marks.items():
        device.write_sub_buffer(x, at, np.array([value], np.uint32))
    hx.RocmAxisReductionOps().reduce_axis_into(
        device, hx.SumOp, StridedView(x, Layout.try_new([lines, outputs], [0, 1], 0)), 0,
        StridedView(out, Layout.c_contiguous([1, outputs])))
    for at, value in marks.items():
        first = min(max(at - 2, 0), outputs - 8)
        want = [lines * marks.get(first + i, 0) for i in range(8)]
        assert _slice(device, out, first, 8).tolist() == want, at
    x.free()
    out.free()
