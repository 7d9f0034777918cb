"""Recorded scans that need no status words are one graph node (no clear in
front): lines that one tile holds, column scans of one tile or one chunk.
Prepared plans and hx_scan_noalloc, replayed with new inputs; an eager
dispatch of the plan, which may be cut in other tiles, runs in between."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import hephaestus_amd as hx
from hephaestus_amd import Layout, StridedView

from test_gpu_capture import Capture, Stream, _hip

pytestmark = pytest.mark.gpu

SCAN = hx.RocmScanOps()

# (rows, cols, axis, nodes): 8192 elements are the longest ragged line kept
# in one tile, whole tiles to 32768; 16384 / 3 and 32768 / 24 rows are one row tile, 224
# rows one chunk of a strip.
SHAPES = [(1, 2049, 1, 1), (3, 4096, 1, 1), (1, 5000, 1, 1), (40, 8192, 1, 1), (1, 8193, 1, 2), (1, 16384, 1, 1),
          (2, 32768, 1, 1), (1, 32769, 1, 2), (100, 3, 0, 1), (600, 20, 0, 1), (60, 255, 0, 1), (224, 64, 0, 1),
          (225, 64, 0, 2)]


def _nodes(capture):
    count = ctypes.c_size_t()
    assert _hip().hipGraphGetNodes(capture.graph, None, ctypes.byref(count)) == 0
    return count.value


@pytest.mark.parametrize("dtype", [np.uint32, np.float32])
@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("rows,cols,axis,nodes", SHAPES)
def test_nodes_of_a_recorded_scan(device, oracle, rows, cols, axis, nodes, noalloc, dtype):
    lay = Layout.c_contiguous([rows, cols])
    n = rows * cols
    x, y = device.alloc_zeroed(dtype, n), device.alloc_zeroed(dtype, n)
    args = (device, hx.CumSumOp, StridedView(x, lay), axis, hx.ScanDirection.Forward, StridedView(y, lay),
            hx.ScanKind.Inclusive)
    plan = None if noalloc else SCAN.prepare_scan_axis(*args)
    stream = Stream()
    try:
        capture = Capture(stream)
        with capture:
            if noalloc:
                SCAN.scan_axis_into_noalloc(*args, stream.value)
            else:
                plan.dispatch(stream.value)
        try:
            assert _nodes(capture) == nodes
            for rep in range(3):
                # integers below 2^8: f32 sums are exact
                host = oracle.uniform_int(n, seed=rep + n, lo=0, hi=255).astype(dtype)
                want = np.add.accumulate(host.reshape(rows, cols), axis=axis, dtype=dtype).ravel()
                device.write_buffer(x, host)
                capture.replay()
                assert np.array_equal(device.download_owned(y), want), rep
                device.write_buffer(y, np.zeros(n, dtype))
                (SCAN.scan_axis_into if noalloc else plan.dispatch)(*(args if noalloc else ()))
                assert np.array_equal(device.download_owned(y), want), rep
        finally:
            capture.destroy()
    finally:
        stream.close(device)
