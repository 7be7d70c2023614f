"""The streaming kernels' cache policies and waves per row (csrc/ci8_device.h, quantize.hip,
silu.hip, allspark.hip) on the GPU: inputs past the L2s (32 MiB, nontemporal loads) and
outputs past the MALL (256 MiB, nontemporal stores) must give the bits that the same rows give
in small calls, which tests/test_gpu_quantize.py, test_gpu_silu.py and test_gpu_allspark.py
hold against the oracle; rows at the edges of the eight-wave rules must equal the oracle's.
"""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.helpers import guard_intact, host, to_dev, with_guard

pytestmark = pytest.mark.gpu

# 33.6 MB in, 34 MB in and odd packs, 269.7 MB of codes.
LARGE = [(1030, 16328), (2083, 8200), (15500, 17400)]


def bf16(rows, width):
    g = torch.Generator(device="cuda").manual_seed(rows + width)
    return torch.randn(rows, width, generator=g, device="cuda").bfloat16()


@pytest.mark.parametrize("rows,k", LARGE)
def test_large_quantize_rows_equals_small_calls(ops, rows, k):
    x = bf16(rows, k)
    codes, buf = with_guard((rows, k), torch.int8, 99)
    scales = torch.empty(rows, device="cuda")
    ops.quantize_rows(x, codes, scales)
    part = torch.empty(500, k, device="cuda", dtype=torch.int8)
    part_scales = torch.empty(500, device="cuda")
    for r in range(0, rows, 500):
        c = min(500, rows - r)
        ops.quantize_rows(x[r : r + c], part[:c], part_scales[:c])
        assert torch.equal(codes[r : r + c], part[:c])
        assert torch.equal(scales[r : r + c], part_scales[:c])
    assert guard_intact(buf, 99)


@pytest.mark.parametrize("rows,k", [(970, 8704), (485, 17408), (15500, 17408)])
def test_large_silu_equals_small_calls(ops, rows, k):
    x = bf16(rows, 2 * k)
    codes, buf = with_guard((rows, k), torch.int8, 99)
    act, act_buf = with_guard((rows, k), torch.bfloat16, float("nan"))
    scales = torch.empty(rows, device="cuda")
    ops.silu_mul_quantize(x, codes, scales)
    ops.silu_mul(x, act)
    part = torch.empty(250, k, device="cuda", dtype=torch.int8)
    part_act = torch.empty(250, k, device="cuda", dtype=torch.bfloat16)
    part_scales = torch.empty(250, device="cuda")
    for r in range(0, rows, 250):
        c = min(250, rows - r)
        ops.silu_mul_quantize(x[r : r + c], part[:c], part_scales[:c])
        ops.silu_mul(x[r : r + c], part_act[:c])
        assert torch.equal(codes[r : r + c], part[:c])
        assert torch.equal(act[r : r + c], part_act[:c])
        assert torch.equal(scales[r : r + c], part_scales[:c])
    assert guard_intact(buf, 99) and guard_intact(act_buf, float("nan"))


@pytest.mark.parametrize("n,k", [(32 * 500 + 16, 17408)])
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
