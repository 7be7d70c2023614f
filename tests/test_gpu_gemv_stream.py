"""GPU parity of channel_gemv's stream kernel (csrc/gemv_stream.hip).

SHAPES holds, for every tile width (8 * copies channels) and x height (4, 8 or 16 rows) of the
kernel, shapes that channel_gemv runs on it (the choice is checked on the CPU below): ragged
N, half last channel blocks, K tails inside a stage, fewer stages than waves, and more than one
round of tiles. Every element is held to test_gpu_gemv.py's bound (one BF16 ulp plus the
rounding of any FP32 summation order).
"""

import shutil
import subprocess

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.conftest import PKG
from tests.helpers import bf16_bits, guard_intact, randn_bf16, to_dev, with_guard
from tests.test_gpu_gemv import QUAD_SHAPES, RESIDENT_SHAPES, SPAN_SHAPES, check_gemv

SHAPES = [
    # copies, m, n, k
    (1, 5, 2001, 2064), (1, 16, 37, 128), (1, 1, 1023, 8320), (2, 8, 4000, 2064), (2, 9, 4095, 4096),
    (3, 6, 4861, 256), (3, 16, 4864, 2176), (4, 13, 8190, 5136), (5, 12, 10001, 5120),
    (6, 1, 12003, 8320), (7, 3, 14001, 8208), (8, 4, 16001, 8208), (9, 2, 18001, 8208),
    (5, 7, 19000, 8224), (3, 4, 5120, 17408),
    (1, 5, 999, 16), (2, 16, 3622, 80), (1, 8, 366, 944),
    # past 96 MB: nontemporal copies
    (7, 9, 27001, 4096), (6, 5, 24501, 4224), (5, 16, 18433, 8192), (9, 12, 34817, 3072 + 1152), (6, 1, 11801, 8576),
]

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "tile_plan.h"
int main(int argc, char** argv) {
  for (int i = 1; i + 3 < argc; i += 4)
    std::printf("%d\n", ci8::gemv_stream_copies(atoi(argv[i]), atoi(argv[i + 1]), atoi(argv[i + 2]),
                                                atoi(argv[i + 3])));
  std::printf("%d\n", ci8::kStreamMaxCopies);
  return 0;
}
"""


def test_choices(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    (tmp_path / "plan.cpp").write_text(PROGRAM)
    subprocess.run([gxx, "-std=c++17", "-O1", f"-I{PKG / 'csrc'}", str(tmp_path / "plan.cpp"), "-o",
                    str(tmp_path / "plan")], check=True)
    others = [(1, 4096, 4096, 256), (4, 17408, 5120, 256), (8, 8192, 8192, 256),
              (16, 17408, 5120, 256), (5, 512, 512, 0),
              (8, 28672, 8192, 256), (8, 28672, 4096, 256), (16, 28672, 4112, 256),
              # measured up to 22% slower on the stream kernel
              (1, 26801, 9280, 256), (1, 3755, 8832, 256), (2, 7846, 9984, 256),
              (10, 1684, 1040, 256), (5, 2481, 7824, 256), (14, 4839, 1808, 256),
              (9, 5000, 1616, 256), (11, 8630, 7056, 256), (8, 5102, 6416, 256),
              (9, 5036, 3456, 256), (6, 586, 5776, 256), (5, 129, 7584, 256),
              *((*s, 256) for s in SPAN_SHAPES + QUAD_SHAPES + RESIDENT_SHAPES)]
    # measured up to 12% faster on it
    taken = [(14, 5047, 5568, 256), (8, 1866, 1984, 256), (2, 6352, 17408, 256),
             (1, 6352, 17408, 256), (1, 5120, 17408, 256), (3, 2088, 9712, 256),
             (16, 366, 944, 256), (8, 924, 6480, 256),
             (10, 4373, 16, 256)]
    cases = [(m, n, k, 256) for _, m, n, k in SHAPES] + others + taken
    lines = subprocess.run([str(tmp_path / "plan"), *(str(v) for c in cases for v in c)], check=True,
                           capture_output=True, text=True).stdout.split()
    got = [int(v) for v in lines]
    assert got[: len(SHAPES)] == [s[0] for s in SHAPES]
    assert got[len(SHAPES): len(cases) - len(taken)] == [0] * len(others)
    assert all(got[len(cases) - len(taken): len(cases)])
    assert {s[0] for s in SHAPES} == set(range(1, got[len(cases)] + 1))


@pytest.mark.gpu
@pytest.mark.parametrize("copies,m,n,k", SHAPES)
def test_stream_widths(ops, copies, m, n, k):
    rng = np.random.default_rng(m * 31 + n + k)
    x_bits = randn_bf16(rng, (m, k))
    w = rng.integers(-128, 128, (n, k)).astype(np.int8)
    s_bits = O.f32_to_bf16((rng.random(n) * 0.002).astype(np.float32))
    out, buf = with_guard((m, n), torch.bfloat16, float("nan"))
    print(f"stream gemv copies={copies} m={m} n={n} k={k}", flush=True)
    ops.channel_gemv(to_dev(x_bits), to_dev(w), to_dev(s_bits), out)
    torch.cuda.synchronize()
    assert guard_intact(buf, float("nan"))
    check_gemv(bf16_bits(out), x_bits, w, s_bits)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 6])
def test_long_rows_with_x_off_16_bytes(ops, m):
    """x at a 4-byte offset keeps the kernels that load it that way."""
    n, k = 300, 8208
    rng = np.random.default_rng(m)
    x_bits = randn_bf16(rng, (m, k))
    w = rng.integers(-128, 128, (n, k)).astype(np.int8)
    s_bits = O.f32_to_bf16((rng.random(n) * 0.002).astype(np.float32))
    x = to_dev(np.concatenate([np.zeros(2, np.uint16), x_bits.reshape(-1)]))[2:].view(m, k)
    out = torch.empty(m, n, device="cuda", dtype=torch.bfloat16)
    ops.channel_gemv(x, to_dev(w), to_dev(s_bits), out)
    torch.cuda.synchronize()
    check_gemv(bf16_bits(out), x_bits, w, s_bits)


@pytest.mark.gpu
def test_special_values(ops):
    """A NaN activation reaches its own row only; an infinite channel scale gives that
    channel's infinities, also with a K tail; other rows and channels stay finite."""
    m, n, k = 6, 50, 2128
    rng = np.random.default_rng(3)
    x = to_dev(randn_bf16(rng, (m, k))).abs() + 0.125
    x[2, k - 1] = float("nan")
    w = torch.from_numpy(rng.integers(1, 128, (n, k)).astype(np.int8)).cuda()
    s = torch.full((n,), 0.01, device="cuda", dtype=torch.bfloat16)
    s[7] = float("inf")
    out = torch.empty(m, n, device="cuda", dtype=torch.bfloat16)
    ops.channel_gemv(x, w, s, out)
    torch.cuda.synchronize()
    got = out.float().cpu().numpy()
    rows, channels = np.delete(np.arange(m), 2), np.delete(np.arange(n), 7)
    assert np.isnan(got[2]).all()
    assert np.isposinf(got[rows, 7]).all()
    assert np.isfinite(got[np.ix_(rows, channels)]).all()
