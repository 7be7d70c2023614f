"""GPU parity of the grouped ring kernel (csrc/grouped_ring.hip), bit-exact against the oracle.

SHAPES holds, for every tile of the kernel, shapes that grouped_summed_mm runs on it (the
choice is checked on the CPU below): partial tiles, K tails inside a stage (copies crossing
group boundaries mid-row), one stage per group, fewer stages than ring slots in all, several
tiles per CU, the most groups whose row scales fit a tile's LDS and one more, and M >= 1024
with M % 4 != 0 or a row scale tensor off 16-byte alignment.
"""

import shutil
import subprocess

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.conftest import PKG
from tests.helpers import bf16_bits, guard_intact, to_dev, with_guard
from tests.test_gpu_grouped import TWO_WAVES_SHAPES, grouped_inputs

SHAPES = [
    # tile, groups, m, n, k
    ((32, 64), 2, 15, 824, 320), ((32, 64), 1, 70, 64, 64), ((32, 64), 128, 40, 132, 32),
    ((64, 64), 3, 292, 1636, 160), ((64, 64), 2, 653, 940, 64), ((96, 64), 4, 238, 4276, 320),
    ((64, 96), 4, 1077, 1428, 416), ((64, 128), 2, 732, 2212, 576), ((96, 128), 2, 1485, 2036, 320),
    ((128, 96), 3, 866, 3388, 320), ((128, 128), 4, 749, 4132, 32), ((128, 128), 2, 932, 3444, 448),
    ((160, 128), 3, 1179, 3240, 224), ((192, 128), 4, 1129, 4708, 128), ((0, 0), 129, 40, 132, 32),
]

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "tile_plan.h"
using namespace ci8;
int main(int argc, char** argv) {
  for (int i = 1; i + 5 < argc; i += 6) {
    const int t = grouped_ring_tile(atoi(argv[i]), atoi(argv[i + 1]), atoi(argv[i + 2]),
                                    atoi(argv[i + 3]), atoi(argv[i + 4]), atoi(argv[i + 5]) != 0);
    std::printf("%d %d\n", t < 0 ? 0 : kGroupedTiles[t].bm, t < 0 ? 0 : kGroupedTiles[t].bn);
  }
  std::printf("%d\n", kGroupedTileCount);
  return 0;
}
"""


def test_tile_choices(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    (tmp_path / "plan.cpp").write_text(PROGRAM)
    subprocess.run([gxx, "-std=c++17", "-O1", f"-I{PKG / 'csrc'}", str(tmp_path / "plan.cpp"), "-o",
                    str(tmp_path / "plan")], check=True)
    # By hand: M = 2048, N = 4096, G = 4, K = 4096 fills one round with 256 x 128 tiles (115
    # us; 512 ring tiles of 128 x 128 take 159), which run unless the call rules them out;
    # without a CU count nothing is chosen.
    by_hand = [(2048, 4096, 4096, 4, 256, 1), (2048, 4096, 4096, 4, 256, 0), (64, 4096, 4096, 4, 0, 0)]
    two_waves = [(m, n, k, g, 256, 1) for g, m, n, k in [*TWO_WAVES_SHAPES, (3, 1028, 3600, 384)]]
    cases = [(m, n, k, g, 256, 0) for _, g, m, n, k in SHAPES] + by_hand + two_waves
    lines = subprocess.run([str(tmp_path / "plan"), *(str(v) for c in cases for v in c)], check=True,
                           capture_output=True, text=True).stdout.split("\n")
    got = [tuple(map(int, line.split())) for line in lines[: len(cases)]]
    assert got[: len(SHAPES)] == [s[0] for s in SHAPES]
    assert got[len(SHAPES)] == (0, 0) and got[len(SHAPES) + 1] != (0, 0)
    assert got[len(SHAPES) + 2] == (0, 0)
    assert got[len(SHAPES) + len(by_hand):] == [(0, 0)] * len(two_waves)
    assert all(m >= 1024 and m % 4 == 0 and n % 4 == 0 for m, n, *_ in two_waves)
    assert len({s[0] for s in SHAPES} - {(0, 0)}) == int(lines[len(cases)])


@pytest.mark.gpu
@pytest.mark.parametrize("tile,g,m,n,k", SHAPES)
def test_ring_tiles_match_the_oracle(ops, tile, g, m, n, k):
    rng = np.random.default_rng(g * 100003 + m * 101 + n + k)
    a_np, w_np, sa_np, sw_np = grouped_inputs(rng, g, m, n, k, signed_scales=True)
    # Row scales one FP32 off 16-byte alignment: the kernel reads them one by one, and the
    # 256 x 128 tiles, which need them aligned, are ruled out at M >= 1024 too.
    sa = to_dev(np.concatenate([np.zeros(1, np.float32), sa_np.reshape(-1)]))[1:].view(g, m)
    out, buf = with_guard((m, n), torch.bfloat16, float("nan"))
    print(f"grouped ring tile {tile} g={g} m={m} n={n} k={k}", flush=True)
    ops.grouped_summed_mm(to_dev(a_np), to_dev(w_np), sa, to_dev(sw_np), out)
    torch.cuda.synchronize()
    assert guard_intact(buf, float("nan"))
    assert np.array_equal(bf16_bits(out), O.grouped_summed_mm(a_np, sa_np, w_np, sw_np))
