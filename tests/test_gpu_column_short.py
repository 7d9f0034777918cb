"""Axis-0 reductions of few lines: up to 32 lines are walked whole, one launch
and no partials; from 33 one-launch blocks."""
from __future__ import annotations

import numpy as np
import pytest

import hephaestus_amd as hx
from hephaestus_amd import Layout, StridedView

import test_gpu_column_blocks as blocks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lines,cols,pitch", [(16, 4096, 4096), (17, 63, 63), (17, 2049, 2049), (18, 205_844, 205_846),
                                              (31, 1000, 1003), (32, 100_001, 100_001), (32, 64, 64), (33, 1000, 1000)])
def test_few_lines_are_one_launch(device, oracle, lines, cols, pitch):
    x, out = device.alloc_zeroed(np.float32, lines * pitch), device.alloc_zeroed(np.float32, cols)
    plan = hx.RocmAxisReductionOps().prepare_reduce_axis_into(
        device, hx.SumOp, StridedView(x, Layout.try_new([lines, cols], [pitch, 1], 0)), 0,
        StridedView(out, Layout.c_contiguous([1, cols])))
    assert plan.workspace_bytes() == 0
    blocks.test_column_reductions(device, oracle, lines, cols, pitch, 0)


@pytest.mark.parametrize("cols", [1, 3, 64, 1001])
def test_no_lines(device, cols):
    """An empty reduced axis: the identity, one launch."""
    x, out = device.alloc_zeroed(np.uint32, 0), device.upload(np.full(cols, 7, np.uint32))
    ops = hx.RocmAxisReductionOps()
    views = StridedView(x, Layout.c_contiguous([0, cols])), StridedView(out, Layout.c_contiguous([1, cols]))
    assert ops.prepare_reduce_axis_into(device, hx.SumOp, views[0], 0, views[1]).workspace_bytes() == 0
    ops.reduce_axis_into(device, hx.SumOp, views[0], 0, views[1])
    assert not device.download_owned(out).any()
