"""GPU parity of the persistent GEMM's tile widths (csrc/gemm_pp.hip), bit for bit.

SHAPES holds, for every width of pp_width (csrc/tile_plan.h), shapes that schedule 0 runs in
one launch of that width (tests/test_ring_plan.py checks the choice on the CPU): partial tiles
in both directions, less than one K stage (128) and a tail inside a stage, one round and
several tiles per CU. The comparisons are those of tests/test_gpu_ring.py.
"""

import pytest

from tests import test_gpu_ring

pytestmark = pytest.mark.gpu

SHAPES = [
    (128, 653, 6760, 32), (128, 2592, 9240, 32), (128, 1556, 9240, 128), (128, 1038, 6024, 416),
    (160, 769, 8368, 32), (160, 772, 8352, 128), (160, 2592, 6024, 160),
    (160, 1297, 6024, 1056), (192, 2592, 12456, 32), (192, 775, 10408, 128),
    (192, 2333, 4416, 160), (192, 1038, 9240, 1056), (224, 769, 12344, 128),
    (224, 769, 12304, 160),
    # rows that do not start on 16 bytes: narrower stores
    (160, 643, 10988, 3200), (192, 962, 11716, 3200), (224, 964, 13684, 3200),
]


@pytest.mark.parametrize("width,m,n,k", SHAPES)
def test_widths_match_the_plain_tiling_and_the_oracle(ops, width, m, n, k):
    test_gpu_ring.test_ring_tiles_match_the_plain_tiling_and_the_oracle(ops, width, m, n, k)
