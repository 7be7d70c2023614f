"""GPU parity of the GGUF Q8_0 ring kernel (csrc/gguf_ring.hip).

SHAPES holds, for every tile of the kernel, shapes that gguf_q8_packed_mm runs on it (the
choice is checked on the CPU below): partial tiles, K tails inside a stage of 128 or 256
values, fewer K stages than ring slots, several tiles per CU, groups, padded rows with NaN in
the padding (which must not reach any sum), and scalar stores (N % 4 != 0). Every element is
held to the bound of tests/test_gpu_gguf_q8.py: one BF16 ulp plus K * 2^-24 * sum |x wq|, the
rounding of any FP32 summation order.
"""

import shutil
import subprocess

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.conftest import PKG
from tests.helpers import bf16_bits, guard_intact, to_dev, with_guard
from tests.test_gpu_gguf_q8 import LARGE_CASES, RING_CASES, SPAN_CASES, check

SHAPES = [
    # tile, m, groups, n, k, row padding
    ((16, 16), 11, 3, 1126, 2240, 8), ((16, 16), 892, 1, 3, 64, 0), ((16, 32), 49, 1, 1633, 1344, 0),
    ((16, 32), 16, 1, 8192, 2304, 0), ((32, 32), 361, 3, 199, 704, 24), ((32, 32), 17, 1, 8188, 320, 8),
    ((64, 32), 239, 2, 826, 2496, 0), ((64, 64), 346, 1, 1052, 448, 8), ((96, 64), 153, 2, 2836, 384, 0),
    ((128, 64), 614, 1, 2770, 704, 8), ((128, 96), 758, 3, 1219, 2176, 8), ((128, 128), 1028, 1, 3140, 3136, 0),
]

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "tile_plan.h"
using namespace ci8;
int main(int argc, char** argv) {
  for (int i = 1; i + 4 < argc; i += 5) {
    const int t = gguf_ring_tile(atoi(argv[i]), atoi(argv[i + 1]), atoi(argv[i + 2]),
                                 atoi(argv[i + 3]), atoi(argv[i + 4]));
    const int rows = gguf_large_rows(atoi(argv[i]), atoi(argv[i + 1]), atoi(argv[i + 3]), 256);
    std::printf("%d %d %d\n", t < 0 ? 0 : kGgufTiles[t].bm, t < 0 ? 0 : kGgufTiles[t].bn, rows);
  }
  std::printf("%d\n", kGgufTileCount);
  return 0;
}
"""


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    """(m, n, k, groups, cus) cases -> chosen (bm, bn), (0, 0) for none; the tile count; the rows
    of the large tiles (gguf_q8.hip) that run the case if it is none and m > 16."""
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    folder = tmp_path_factory.mktemp("gguf_plan")
    (folder / "plan.cpp").write_text(PROGRAM)
    subprocess.run([gxx, "-std=c++17", "-O1", f"-I{PKG / 'csrc'}", str(folder / "plan.cpp"), "-o",
                    str(folder / "plan")], check=True)

    def run(cases):
        lines = subprocess.run([str(folder / "plan"), *(str(v) for c in cases for v in c)], check=True,
                               capture_output=True, text=True).stdout.split("\n")
        got = [tuple(map(int, line.split())) for line in lines[: len(cases)]]
        return [g[:2] for g in got], int(lines[len(cases)]), [g[2] for g in got]

    return run


def test_tile_choices(choose):
    # By hand: M = 2048, N = K = 4096 runs 256 tiles of 256 x 128, one round, 66.9 us, 512
    # ring tiles of 128 x 128 two of 42.0; M = 1, N = K = 4096 16 channels a CU: 6.7 against
    # 7.5 us for 256 tiles of 16 x 16; without a CU count nothing is chosen.
    # M <= 16 shapes that the span kernel was measured to run up to 19% faster (us, span / ring):
    # 6.8 / 8.1, 4.8 / 5.7, 8.0 / 8.8, 9.0 / 10.1, 9.6 / 10.4, 6.5 / 7.2, 3.35 / 3.68.
    span = [(2, 3437, 3136, 2, 256), (12, 7022, 1344, 1, 256), (3, 6198, 3712, 1, 256),
            (1, 6023, 4992, 1, 256), (16, 8038, 2112, 2, 256), (6, 8168, 2240, 1, 256),
            (14, 502, 320, 1, 256)]
    by_hand = [(2048, 4096, 4096, 1, 256), (1, 4096, 4096, 1, 256), (64, 4096, 4096, 1, 0), *span]
    cases = [(m, n, k, g, 256) for _, m, g, n, k, _ in SHAPES] + by_hand
    # K > 8192 (us, the other kernels / ring): 135.6 / 80.1, 139.3 / 68.6, 59.7 / 48.9.
    long_k = [(3, 11877, 8704, 4, 256), (1, 8674, 9152, 4, 256), (5, 12024, 9600, 2, 256)]
    assert choose(long_k)[0] == [(16, 32)] * 3
    # One K stage, up to 16 channels a CU: 3.23 / 3.01, 3.42 / 3.06, 3.21 / 3.06.
    short_k = [(2, 520, 256, 1, 256), (3, 3532, 256, 1, 256), (10, 200, 64, 2, 256)]
    assert choose(short_k)[0] == [(16, 16)] * 3
    # 64 and more channels a CU: 51.5 / 45.5, 47.0 / 43.2, 46.7 / 42.4; past M = 8 51.1 / 55.8, 33.9 / 36.2.
    many = [(2, 8078, 7168, 4, 256), (5, 7284, 6912, 4, 256), (3, 4029, 5824, 8, 256),
            (12, 7257, 7488, 4, 256), (16, 5339, 5952, 4, 256)]
    assert choose(many)[0] == [(16, 32)] * 3 + [(0, 0)] * 2
    got, count, _ = choose(cases)
    assert got[: len(SHAPES)] == [s[0] for s in SHAPES]
    assert got[len(SHAPES):] == [(0, 0)] * len(by_hand)
    assert len({s[0] for s in SHAPES}) == count


def test_cases_of_the_other_kernels(choose):
    """The cases of test_gpu_gguf_q8.py run the kernels that they are listed under."""
    got, *_ = choose([(m, n, k, g, 256) for m, g, n, k, _ in RING_CASES])
    assert (0, 0) not in got
    got, *_ = choose([(m, n, k, g, 256) for m, g, n, k, _ in SPAN_CASES])
    assert set(got) == {(0, 0)}
    got, _, rows = choose([(m, n, k, g, 256) for _, m, g, n, k, _ in LARGE_CASES])
    assert set(got) == {(0, 0)}
    assert rows == [case[0] for case in LARGE_CASES]


def test_launches_fit_32_bit_work_item_counts(choose):
    """HIP refuses 2^32 work-items or more along x. A tile of which a call would need that many
    (512 threads each; the most rows the operator takes, and hundreds of groups that share x
    through small strides) is never chosen, the largest count that fits is."""
    m, n = 65535 * 32, 3
    cases = [(m, n, k, g, 256) for g in (256, 511, 512, 1000, 65535) for k in (64, 1024, 2048, 4096)]
    got, *_ = choose(cases)
    for (*_, groups, _), (bm, bn) in zip(cases, got):
        blocks = -(-m // bm) * -(-n // bn) * groups if bm else 0
        assert blocks * 512 < 2**32, (groups, bm, bn)
    assert got[cases.index((m, n, 2048, 511, 256))] != (0, 0)
    assert got[cases.index((m, n, 2048, 512, 256))] == (0, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("tile,m,groups,n,k,pad", SHAPES)
def test_ring_tiles(ops, tile, m, groups, n, k, pad):
    from consumer_int8 import gguf

    rng = np.random.default_rng(m * 31 + n + k)
    row = groups * k + pad
    x_full = O.f32_to_bf16(rng.standard_normal((m, row)).astype(np.float32))
    x_full[:, groups * k:] = 0x7FC0  # NaN
    x_np = x_full[:, : groups * k].reshape(m, groups, k)
    codes_np = rng.integers(-128, 128, (groups, n, k)).astype(np.int8)
    scales_np = (rng.random((groups, n, k // 32)) * 0.02).astype(np.float16).view(np.uint16)
    x = torch.as_strided(to_dev(x_full), (m, groups, k), (row, k, 1))
    out, buf = with_guard((m, groups, n), torch.bfloat16, float("nan"))
    print(f"gguf ring tile {tile} m={m} groups={groups} n={n} k={k} pad={pad}", flush=True)
    gguf.q8_packed_mm(x, to_dev(codes_np), to_dev(scales_np).view(torch.float16), out)
    torch.cuda.synchronize()
    assert guard_intact(buf, float("nan"))
    check(bf16_bits(out), x_np, codes_np, scales_np, rel_norm=0.001)


@pytest.mark.gpu
def test_ring_special_values(ops):
    """An infinite scale gives what the rounded weights give: infinities of the codes' sign
    (NaN for a zero code); a NaN activation reaches its own row only."""
    from consumer_int8 import gguf

    m, n, k = 34, 40, 320
    rng = np.random.default_rng(9)
    x_np = O.f32_to_bf16(rng.standard_normal((m, 1, k)).astype(np.float32))
    x_np[5, 0, 300] = 0x7FC0
    codes_np = rng.integers(1, 128, (1, n, k)).astype(np.int8)
    codes_np[0, 7, 290] = 0
    scales = (rng.random((1, n, k // 32)) * 0.02).astype(np.float16)
    scales[0, 7, 9] = scales[0, 8, 0] = np.inf
    x = to_dev(x_np)
    x[:, 0, 288:] = x[:, 0, 288:].abs()
    x[:, 0, :32] = -x[:, 0, :32].abs()
    out = torch.empty(m, 1, n, device="cuda", dtype=torch.bfloat16)
    gguf.q8_packed_mm(x, to_dev(codes_np), to_dev(scales.view(np.uint16)).view(torch.float16), out)
    torch.cuda.synchronize()
    got = out[:, 0].float().cpu().numpy()
    others = np.delete(np.arange(m), 5)
    assert np.isnan(got[5]).all()
    assert np.isnan(got[others, 7]).all() and np.isneginf(got[others, 8]).all()
    assert np.isfinite(np.delete(got[others], [7, 8], axis=1)).all()
