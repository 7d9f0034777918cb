"""hx_scan_noalloc takes a scan by its figure and then runs it in the fixed
scratch: whatever is taken has to fit.  Host arithmetic only (no GPU)."""
from __future__ import annotations

import ctypes
import random

import numpy as np
import pytest

import hephaestus_amd as hx
from hephaestus_amd import Layout, _ffi
from hephaestus_amd.device import hx_dtype

SCRATCH = 8 << 20


def sizes(dtype, rows, cols, pitch, axis=0, skip=0):
    lay = Layout.try_new([rows, cols], [pitch, 1], 0)
    view = ctypes.byref(_ffi.layout_struct(lay))
    needs, uses = ctypes.c_uint64(), ctypes.c_uint64()
    n = rows * pitch
    _ffi.check(_ffi.lib().hx_debug_scan_noalloc_bytes(hx_dtype(dtype), 1 << 40, n, view, axis,
                                                      (1 << 44) + 4 * skip, n, view,
                                                      ctypes.byref(needs), ctypes.byref(uses)))
    return needs.value, uses.value


def taken_fits(dtype, rows, cols, pitch, axis=0, skip=0):
    needs, uses = sizes(dtype, rows, cols, pitch, axis, skip)
    assert uses <= SCRATCH or needs > SCRATCH, (dtype, rows, cols, pitch, axis, skip, needs, uses)
    return needs <= SCRATCH


@pytest.fixture(scope="module", autouse=True)
def _library():
    hx.load_native()


@pytest.mark.parametrize("rows,cols,pitch", [(91_729, 1279, 1279), (94_200, 1279, 1279), (97_560, 1279, 1279),
                                             (90_000, 1280, 1283), (65_000, 1790, 1790), (50_000, 2303, 2303),
                                             (4_000_003, 64, 64), (3_600_001, 65, 65), (30_000_000, 200, 203)])
def test_f32_scans_near_the_limit_are_taken(rows, cols, pitch):
    assert taken_fits(np.float32, rows, cols, pitch)


@pytest.mark.parametrize("dtype,rows,cols", [(np.uint32, 65536, 4096), (np.uint32, 1 << 20, 256),
                                             (np.float32, 2_684_354, 100), (np.float32, 98_161, 1279)])
def test_larger_scans_are_rejected(dtype, rows, cols):
    assert sizes(dtype, rows, cols, cols)[0] > SCRATCH


def test_every_scan_that_is_taken_fits():
    rng = random.Random(7)
    for _ in range(20_000):
        cols = round(2 ** rng.uniform(0, 20))
        rows = round(2 ** rng.uniform(0, 32 - np.log2(cols)))
        dtype = rng.choice((np.float32, np.uint32, np.int32))
        taken_fits(dtype, rows, cols, cols + rng.choice((0, 0, 1, 3, 4, 32)), rng.randrange(2), rng.choice((0, 0, 1)))
