"""Axis-0 reductions at the edges of the rule that gives a lane four outputs or
one: output counts that are no multiple of 4 around 2^18 at up to 32 lines,
around 2^20 elements, with last groups of 8 and 9 outputs, and of 640, 10240
and 3 * 2^23 elements beyond 1024 lines."""
from __future__ import annotations

import pytest

import test_gpu_column_blocks as blocks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lines,cols,pitch", [
    (17, (1 << 18) - 1, (1 << 18) - 1), (32, (1 << 18) + 1, (1 << 18) + 2), (33, 31_775, 31_775), (33, 31_777, 31_777),
    (257, 73, 75), (257, 72 + 1, 73), (1000, 201, 201), (300, 70, 71), (1025, 11, 13), (5000, 639, 639),
    (5000, 641, 641), (4999, 641, 643), (1100, 10_239, 10_239), (1100, 10_241, 10_241), (195_000, 129, 129),
    (195_200, 130, 131), (300_000, 7, 9)])
def test_outputs_per_lane(device, oracle, lines, cols, pitch):
    blocks.test_column_reductions(device, oracle, lines, cols, pitch, 0)
