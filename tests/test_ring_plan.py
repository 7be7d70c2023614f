"""Schedule 0's choice between the ring kernel and the others (gemm_choice in
csrc/tile_plan.h), compiled on the CPU with g++: every ring tile is picked by one of the
shapes that tests/test_gpu_ring.py runs on the GPU, and shapes worked out by hand from the
round times go where they should."""

import shutil
import subprocess

import pytest

from tests.conftest import PKG
from tests.test_gpu_gemm import SWITCHES, WIDE_SHAPES
from tests.test_gpu_pp_width import SHAPES as PP_SHAPES
from tests.test_gpu_ring import SHAPES

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "tile_plan.h"
using namespace ci8;
int main(int argc, char** argv) {
  for (int i = 1; i + 4 < argc; i += 5) {
    const char op = argv[i + 4][0];  // f: fused or biased, w: with INT32 products, u: neither
    const int m = atoi(argv[i]), n = atoi(argv[i + 1]), k = atoi(argv[i + 2]), cus = atoi(argv[i + 3]);
    const GemmChoice c = gemm_choice(m, n, k, cus, op == 'f', op == 'w');
    const int width = pp_width(m, n, k, cus).bn;
    switch (c.kernel) {
      case GemmKernel::kSmall: std::puts("small 0 0"); break;
      case GemmKernel::kRing:
        std::printf("ring %d %d\n", kRingTiles[c.ring].bm, kRingTiles[c.ring].bn);
        break;
      case GemmKernel::kPersistent:  // width, columns of 224-wide tiles before the 160-wide ones
        std::printf("persistent %d %d\n", width, width == kPlanBN ? pp_plan(m, n, cus).n_head : 0);
        break;
      case GemmKernel::kWide256: std::puts("wide 256 0"); break;
      case GemmKernel::kWide224: std::puts("wide 224 0"); break;
    }
  }
  std::printf("%d\n", kRingTileCount);
  return 0;
}
"""


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    folder = tmp_path_factory.mktemp("ring_plan")
    (folder / "plan.cpp").write_text(PROGRAM)
    subprocess.run([gxx, "-std=c++17", "-O1", f"-I{PKG / 'csrc'}", str(folder / "plan.cpp"), "-o",
                    str(folder / "plan")], check=True)

    def run(cases):
        args = [str(v) for case in cases for v in case]
        lines = subprocess.run([str(folder / "plan"), *args], check=True, capture_output=True,
                               text=True).stdout.split("\n")
        return [(kind, int(a), int(b)) for kind, a, b in map(str.split, lines[: len(cases)])], \
            int(lines[len(cases)])

    return run


def test_every_ring_tile_has_a_gpu_shape(choose):
    for op in "fw":  # cutlass_channel_mm's products come from the same tile
        got, count = choose([(m, n, k, 256, op) for _, m, n, k in SHAPES])
        for (tile, m, n, k), choice in zip(SHAPES, got):
            assert choice == ("ring", *tile), (m, n, k, op)
    assert len({tile for tile, *_ in SHAPES}) == count


def test_persistent_widths_have_gpu_shapes(choose):
    got, _ = choose([(m, n, k, 256, "f") for _, m, n, k in PP_SHAPES])
    assert got == [("persistent", width, 0) for width, *_ in PP_SHAPES]
    assert {width for width, *_ in PP_SHAPES} == {224, 192, 160, 128}


def test_kernels_of_the_gemm_tests(choose):
    got, _ = choose([(m, n, k, 256, "f") for _, _, m, n, k, _ in SWITCHES])
    assert got == [("persistent", width, split) for width, split, *_ in SWITCHES]
    got, _ = choose([(m, n, k, 256, call) for _, call, m, n, k in WIDE_SHAPES])
    assert got == [("wide", width, 0) for width, *_ in WIDE_SHAPES]
    # test_wide_tiles_where_they_fill_the_rounds; the large tilings without their rivals
    got, _ = choose([(256, 11264, 256, 256, "f"), (200, 34816, 128, 256, "f"),
                     (1024, 2560, 544, 256, "f")])
    assert got[0][0] == "ring" and got[1][:2] == ("persistent", 160)
    assert got[2][0] == "ring"


def test_256_wide_tiles_take_no_k_tail(choose):
    """With one they take two to three times as long: 403 us for the second with products, 210 by
    the ring kernel."""
    got, _ = choose([(4096, 4096, 1152, 256, "f"), (4096, 4096, 1056, 256, "f"),
                     (1335, 10392, 9568, 256, "w")])
    assert got[0] == ("wide", 256, 0)
    assert got[1][:2] != ("wide", 256) and got[2][0] == "ring"


def test_choices_by_hand(choose):
    cases = [
        # M = 4096, N = 17408, K = 5120: 1,248 persistent tiles, 4 + 0.75 + 0.25 * 224 / 256
        # rounds of 52.7 us = 263 us; 22 x 109 = 2,398 tiles of 192 x 160, 9.37 + rounds of
        # 38.7 us = 363 us.
        (4096, 17408, 5120, 256, "f"),
        # M = 128, N = K = 4096: 256 small-M tiles of 64 x 32, one round: 7.9 us; 256 ring
        # tiles of 32 x 64: 8.9 us.
        (128, 4096, 4096, 256, "f"),
        # M = 1024, N = 5120, K = 17408: 256 tiles of 128 x 160, one round, 90.8 us; 92
        # persistent tiles of 224 take 0.84 of a round of 157 us, 160 of 128 0.91 of 120 us.
        (1024, 5120, 17408, 256, "f"),
        # M = 768, N = 17408, K = 5120: 234 persistent tiles, 0.98 of a round: 53 us; ring
        # tiles take 2 rounds or more.
        (768, 17408, 5120, 256, "f"),
        # The same with an INT32 copy, which the persistent kernel does not write.
        (768, 17408, 5120, 256, "w"),
        # M = 2048, N = 5120, K = 17408: 256 tiles of 256 x 160, one round, 129 us; 184 of 224
        # 0.93 of a round of 157 us, 216 of 192 0.96 of one of 141 us.
        (2048, 5120, 17408, 256, "f"),
        # Rows that do not start on 16 bytes: 232 persistent tiles of 128 take 12.9 us by their
        # rounds and 13.6 more for 7.5 million outputs and 0.98 rounds, 464 ring tiles of 128 x
        # 128 19.6 (measured: 26.7 us, 18.9).
        (1018, 7340, 1088, 256, "f"),
        # With products, 10.7 million outputs: 192 x 128 ring tiles 64 us and 17 for them, 204
        # tiles of 224 in one round 67.7 and 13.9, 5% off (measured: 120 us, 94).
        (2870, 3716, 5088, 256, "w"),
        # Level by the times, measured 4.60 and 4.54 us by the small-M kernel, 4.86 by the ring.
        (186, 1496, 1312, 256, "f"),
        (127, 2068, 1408, 256, "f"),
        # One partial round of short tiles: 40, 20 and 174 small-M tiles of 16 x 16 take 2.2 us and
        # 242 of 16 x 32 2.5 (measured: 2.1-2.3 us by the small-M kernel, 2.9-3.7 by the ring; the
        # last after its quantization 5.1 and 5.8-6.1).
        (7, 640, 192, 256, "f"),
        (1, 320, 384, 256, "w"),
        (43, 928, 288, 256, "w"),
        (167, 704, 128, 256, "f"),
        # K = 288: 216 ring tiles of 128 x 128, 120 persistent tiles of 128 (measured: 7.6 us, 9.0).
        (1080, 2992, 288, 256, "f"),
    ]
    got, _ = choose(cases)
    assert got[0] == ("persistent", 224, 0)
    assert got[1] == ("small", 0, 0)
    assert got[2] == ("ring", 128, 160)
    assert got[3] == ("persistent", 224, 0)
    assert got[4][0] == "ring"
    assert got[5] == ("persistent", 160, 0)
    assert got[6][0] == "ring"
    assert got[7] == ("wide", 224, 0)
    assert got[8:14] == [("small", 0, 0)] * 6
    assert got[14][0] == "ring"
