"""Column scans at the edges of the rule that gives wide matrices rows of 1 KiB
in place of strips: one round of blocks (at most 240 rows, 65536 columns, more
than 2^23 elements), two of whole lines (more than 49152 columns, 2^24
elements), and matrices of 5 * 2^24 (f32 3 * 2^25) elements whose rows are no
whole 128-byte lines.  And of the rule for 8 rows a lane: 224 rows up to 2^26
elements, 112 beyond.  Compared as the strips are."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_fallbacks import wait_limits
from test_gpu_strips import check

pytestmark = pytest.mark.gpu

# (rows, cols, pitch, offset)
ROUNDS = [(200, 41_943, 41_943, 0), (200, 41_944, 41_944, 0), (240, 65_535, 65_536, 0), (240, 65_536, 65_537, 1),
          (241, 65_536, 65_536, 0), (257, 65_536, 65_536, 0), (257, 65_536, 65_568, 32), (257, 65_537, 65_537, 0),
          (480, 49_184, 49_184, 0), (480, 49_152, 49_152, 0), (481, 50_016, 50_016, 0)]
FEW_ROWS = [(224, 80_001, 80_001, 0), (225, 80_001, 80_001, 0), (224, 299_600, 299_601, 3), (112, 600_003, 600_003, 0),
            (113, 600_003, 600_003, 0), (90, 200_032, 200_032, 0), (65, 300_001, 300_004, 0)]


@pytest.mark.parametrize("dtype", [np.uint32, np.float32])
@pytest.mark.parametrize("rows,cols,pitch,offset", ROUNDS + FEW_ROWS)
def test_edges_of_the_rules(device, oracle, rows, cols, pitch, offset, dtype):
    check(device, oracle, rows, cols, dtype, seed=rows + cols, pitch=pitch, offset=offset)


@pytest.mark.parametrize("rows,cols,dtype", [(10_240, 8191, np.uint32), (10_240, 8193, np.uint32),
                                             (160, 524_287, np.int32), (161, 524_287, np.int32), (12_290, 8193, np.float32),
                                             (384, 262_143, np.float32), (385, 262_143, np.float32)])
def test_shared_lines_beyond_the_caches(device, oracle, rows, cols, dtype):
    check(device, oracle, rows, cols, dtype, seed=cols)


@pytest.mark.parametrize("prod", [False, True])
@pytest.mark.parametrize("exclusive,reverse", [(True, False), (False, True), (True, True)])
@pytest.mark.parametrize("dtype", [np.int32, np.float32])
@pytest.mark.parametrize("rows,cols,pitch,offset", [(239, 36_001, 36_003, 1), (300, 57_344, 57_344, 0)])
def test_kinds(device, oracle, rows, cols, pitch, offset, dtype, exclusive, reverse, prod):
    check(device, oracle, rows, cols, dtype, seed=rows, pitch=pitch, offset=offset, prod=prod, exclusive=exclusive,
          reverse=reverse)


# Every tile's look-back totals its missing predecessors from the input.
@pytest.mark.parametrize("limits", [(0, 0), (1, 1)])
@pytest.mark.parametrize("dtype", [np.uint32, np.float32])
def test_forced_fallbacks(device, oracle, limits, dtype):
    with wait_limits(*limits):
        check(device, oracle, 480, 49_184, dtype, seed=3)
