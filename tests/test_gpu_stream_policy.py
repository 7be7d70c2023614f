"""The streaming kernels' cache policies and waves per row (csrc/stream_policy.h, quantize.hip,
silu.hip, allspark.hip): outputs past a few MB (written through), inputs past the L2s (32 MiB,
nontemporal loads) and inputs and outputs past the MALL together (256 MiB, nontemporal loads
and stores) must give the bits that the same rows give in small calls, which
tests/test_gpu_quantize.py, test_gpu_silu.py and test_gpu_allspark.py hold against the oracle;
rows at the edges of the eight-wave rules must equal the oracle's. The policy of a call is
checked on the CPU.
"""

import shutil
import subprocess

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.conftest import PKG
from tests.helpers import guard_intact, host, to_dev, with_guard

CACHED, WRITE_THROUGH, NT_LOADS, NT = range(4)
QUANTIZE, SILU = 2 << 20, 0

# 6.0 MB, 33.6 MB and 34 MB in (odd packs), 539 MB in.
LARGE = [(1030, 3048), (1030, 16328), (2083, 8200), (15500, 17400)]

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "stream_policy.h"
int main(int argc, char** argv) {
  for (int i = 1; i + 2 < argc; i += 3)
    std::printf("%d\n", int(ci8::stream_policy(atoll(argv[i]), atoll(argv[i + 1]), atoll(argv[i + 2]))));
  std::printf("%lld %lld\n", (long long)ci8::kQuantizeWriteThrough,
              (long long)ci8::kSiluWriteThrough);
  return 0;
}
"""


def test_policies(tmp_path):
    """Bytes in, bytes out and the output size from which on to write through. A stored output
    is left dirty in the L2s only while it is small, and is nontemporal only where the MALL
    cannot hold it beside the input."""
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    (tmp_path / "policy.cpp").write_text(PROGRAM)
    subprocess.run([gxx, "-std=c++17", "-O1", f"-I{PKG / 'csrc'}", str(tmp_path / "policy.cpp"), "-o",
                    str(tmp_path / "policy")], check=True)
    cases = [
        (2 * 128 * 4096, 128 * 4096, QUANTIZE, CACHED),  # quantize_rows [128, 4096]
        (2 * 512 * 5120, 512 * 5120, QUANTIZE, WRITE_THROUGH),
        (2 * 2048 * 5120, 2048 * 5120, QUANTIZE, WRITE_THROUGH),
        (2 * 4096 * 5120, 4096 * 5120, QUANTIZE, NT_LOADS),
        (2 * 16384 * 5120, 16384 * 5120, QUANTIZE, NT_LOADS),
        (2 * 16384 * 8704, 16384 * 8704, QUANTIZE, NT),
        (4 * 17408, 2 * 17408, SILU, WRITE_THROUGH),  # silu_mul [1, 2 x 17408]
        (4 * 4096 * 8704, 2 * 4096 * 8704, SILU, NT_LOADS),
        (4 * 4096 * 17408, 2 * 4096 * 17408, SILU, NT),
        (4 * 4096 * 17408, 4096 * 17408, QUANTIZE, NT),  # silu_mul_quantize
    ]
    args = [str(v) for *sizes, _ in cases for v in sizes]
    lines = subprocess.run([str(tmp_path / "policy"), *args], check=True, capture_output=True,
                           text=True).stdout.split("\n")
    assert [int(v) for v in lines[: len(cases)]] == [want for *_, want in cases]
    assert lines[len(cases)] == f"{QUANTIZE} {SILU}"


def bf16(rows, width):
    g = torch.Generator(device="cuda").manual_seed(rows + width)
    return torch.randn(rows, width, generator=g, device="cuda").bfloat16()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,k", LARGE)
def test_large_quantize_rows_equals_small_calls(ops, rows, k):
    x = bf16(rows, k)
    codes, buf = with_guard((rows, k), torch.int8, 99)
    scales = torch.empty(rows, device="cuda")
    ops.quantize_rows(x, codes, scales)
    step = min(500, 2**21 // k)  # parts below the write-through size
    part = torch.empty(step, k, device="cuda", dtype=torch.int8)
    part_scales = torch.empty(step, device="cuda")
    for r in range(0, rows, step):
        c = min(step, rows - r)
        ops.quantize_rows(x[r : r + c], part[:c], part_scales[:c])
        assert torch.equal(codes[r : r + c], part[:c])
        assert torch.equal(scales[r : r + c], part_scales[:c])
    assert guard_intact(buf, 99)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,k", [(300, 8704), (970, 8704), (485, 17408), (15500, 17408)])
def test_large_silu_equals_small_calls(ops, rows, k):
    x = bf16(rows, 2 * k)
    codes, buf = with_guard((rows, k), torch.int8, 99)
    act, act_buf = with_guard((rows, k), torch.bfloat16, float("nan"))
    scales = torch.empty(rows, device="cuda")
    ops.silu_mul_quantize(x, codes, scales)
    ops.silu_mul(x, act)
    part = torch.empty(100, k, device="cuda", dtype=torch.int8)
    part_act = torch.empty(100, k, device="cuda", dtype=torch.bfloat16)
    part_scales = torch.empty(100, device="cuda")
    for r in range(0, rows, 100):
        c = min(100, rows - r)
        ops.silu_mul_quantize(x[r : r + c], part[:c], part_scales[:c])
        ops.silu_mul(x[r : r + c], part_act[:c])
        assert torch.equal(codes[r : r + c], part[:c])
        assert torch.equal(act[r : r + c], part_act[:c])
        assert torch.equal(scales[r : r + c], part_scales[:c])
    assert guard_intact(buf, 99) and guard_intact(act_buf, float("nan"))


@pytest.mark.gpu
@pytest.mark.parametrize("n,k", [(32 * 500 + 16, 17408), (32 * 250 + 16, 17408)])
def test_large_unpack_allspark_equals_small_calls(ops, n, k):
    padded = (n + 31) // 32 * 32
    g = torch.Generator(device="cuda").manual_seed(n)
    packed = torch.randint(1, 256, (padded, k), generator=g, device="cuda", dtype=torch.uint8)
    packed_scales = torch.rand(padded, generator=g, device="cuda").bfloat16()
    weight, buf = with_guard((n, k), torch.int8, 99)
    scales = torch.empty(n, device="cuda", dtype=torch.bfloat16)
    ops.unpack_allspark(packed, packed_scales, weight, scales)
    for r in range(0, n, 3200):
        c = min(3200, n - r)
        part = torch.empty(c, k, device="cuda", dtype=torch.int8)
        part_scales = torch.empty(c, device="cuda", dtype=torch.bfloat16)
        end = r + (c + 31) // 32 * 32
        ops.unpack_allspark(packed[r:end], packed_scales[r:end], part, part_scales)
        assert torch.equal(weight[r : r + c], part)
        assert torch.equal(scales[r : r + c], part_scales)
    assert guard_intact(buf, 99)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,k", [(256, 2568), (256, 4104), (257, 4104), (256, 8192),
                                    (1024, 8200), (1025, 8200), (3, 12296), (5, 20480),
                                    (2, 20488)])
def test_waves_per_row_match_the_oracle(ops, rows, k):
    x = bf16(rows, k)
    codes, buf = with_guard((rows, k), torch.int8, 99)
    scales = torch.empty(rows, device="cuda")
    ops.quantize_rows(x, codes, scales)
    want, want_scales = O.quantize_rows(host(x.view(torch.int16)).view(np.uint16))
    assert np.array_equal(host(codes), want) and np.array_equal(host(scales), want_scales)
    assert guard_intact(buf, 99)
