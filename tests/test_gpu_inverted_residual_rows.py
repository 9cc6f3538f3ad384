"""Inverted residual blocks with one buffer of each kind in LDS (csrc/inverted_residual.hip), at the edges of their strips and tiles, against
the oracle: as the other blocks in test_gpu_inverted_residual.py."""
import numpy as np
import pytest

import test_gpu_inverted_residual as whole
from test_gpu_inverted_residual import g, vm  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu

# As test_gpu_inverted_residual.BLOCKS, with the kernel that tests/test_inverted_residual_rows_cpu.py finds each to take: tiles of the projection
# per wavefront, tiles of expanded channels per interval, K steps.  Both strides, rows that do not fill the last strip, one interval and
# the channels of a last one that are not there, rows of no whole 8 or 16.
BLOCKS = [
    ((90, (16, 96, 24), 23, 112, 2, np.uint8, 77, (13, 200, 128), False, True, 0, False), (1, 1, 1)),
    ((64, (24, 144, 24), 56, 56, 1, np.int8, -9, (13, 0, 5), True, False, 1, True), (2, 1, 1)),
    ((64, (24, 72, 40), 27, 53, 1, np.uint8, 0, (0, 255, 0), True, True, 0, False), (2, 1, 1)),
    ((128, (32, 192, 32), 28, 28, 1, np.int8, 100, (255, 9, 117), False, False, 2, False), (1, 2, 1)),
    ((150, (17, 33, 17), 31, 61, 1, np.uint8, 255, (128, 128, 3), True, True, 2, True), (2, 1, 1)),
    ((60, (48, 96, 20), 37, 74, 1, np.uint8, 4, (60, 61, 62), True, True, 0, False), (1, 1, 3)),
    ((100, (32, 32, 16), 45, 112, 2, np.int8, 0, (0, 0, 128), False, True, 0, True), (2, 1, 1)),
    ((40, (64, 128, 32), 41, 60, 2, np.uint8, 131, (31, 0, 90), True, True, 0, True), (1, 2, 3)),
    ((90, (32, 64, 32), 27, 25, 2, np.int8, -128, (0, 0, 0), False, True, 0, False), (1, 2, 1)),
]


@pytest.mark.parametrize("block", [b for b, _ in BLOCKS])
def test_one_buffer(g, oracle, monkeypatch, block):  # noqa: F811
    monkeypatch.setattr(whole, "BLOCKS", [block])
    whole.test_single_blocks(g, oracle, 0)
