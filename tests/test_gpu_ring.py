"""GPU parity of the ring GEMM (csrc/gemm_ring.hip), bit-exact.

SHAPES holds, for every tile of the kernel, a shape that schedule 0 runs on it
(tests/test_ring_plan.py checks the choice on the CPU), with partial tiles in both
directions, K tails inside a stage, fewer K stages than ring slots, an odd and an even
number of stages, and several tiles per CU. The output of fused_channel_mm, channel_mm and
cutlass_channel_mm must equal the 256 x 32 tiling's (schedule 5), and the INT32 products the
oracle's.
"""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.helpers import bf16_bits, guard_intact, host, to_dev, with_guard

SHAPES = [
    ((32, 64), 343, 956, 1568), ((32, 64), 33, 5460, 288), ((32, 96), 190, 3300, 576),
    ((32, 96), 13, 16756, 160), ((64, 48), 334, 1476, 1696), ((64, 64), 353, 2452, 1120),
    ((64, 64), 37, 13132, 1472), ((64, 80), 938, 1188, 1920), ((64, 96), 375, 4028, 1984),
    ((64, 128), 669, 2780, 1888), ((96, 96), 1234, 1560, 1856), ((128, 80), 501, 4104, 1696),
    ((96, 128), 473, 5228, 928), ((128, 128), 328, 10808, 1728), ((128, 128), 297, 8468, 416),
    ((128, 160), 1061, 3724, 1056), ((128, 160), 293, 10948, 800), ((160, 160), 401, 10260, 2080),
    ((192, 128), 521, 8196, 1184), ((192, 160), 521, 10948, 800),
]


def inputs(m, n, k):
    rng = np.random.default_rng(m * 31 + n + k)
    a = rng.integers(-127, 128, (m, k)).astype(np.int8)
    w = rng.integers(-128, 128, (n, k)).astype(np.int8)
    sa = rng.uniform(1e-3, 1e-1, m).astype(np.float32)
    sw = O.f32_to_bf16(rng.uniform(1e-3, 1e-2, n).astype(np.float32))
    return rng, a, w, sa, sw


@pytest.mark.gpu
@pytest.mark.parametrize("tile,m,n,k", SHAPES)
def test_ring_tiles_match_the_plain_tiling_and_the_oracle(ops, tile, m, n, k):
    rng, a_np, w_np, sa_np, sw_np = inputs(m, n, k)
    a, w, sa, sw = to_dev(a_np), to_dev(w_np), to_dev(sa_np), to_dev(sw_np)
    print(f"ring tile {tile} m={m} n={n} k={k}", flush=True)
    ref = torch.empty(m, n, device="cuda", dtype=torch.bfloat16)
    ops.fused_channel_mm(a, w, sa, sw, ref, 5)
    out, buf = with_guard((m, n), torch.bfloat16, float("nan"))
    ops.fused_channel_mm(a, w, sa, sw, out, 0)
    biased, biased_buf = with_guard((m, n), torch.bfloat16, float("nan"))
    ops.channel_mm(a, to_dev((w_np.view(np.uint8) ^ 0x80)), sa, sw, biased)
    full, full_buf = with_guard((m, n), torch.bfloat16, float("nan"))
    acc, acc_buf = with_guard((m, n), torch.int32, -(2**31))
    ops.cutlass_channel_mm(a, w, sa, sw, acc, full)
    torch.cuda.synchronize()
    want = bf16_bits(ref)
    for got, guard in ((out, buf), (biased, biased_buf), (full, full_buf)):
        assert np.array_equal(bf16_bits(got), want)
        assert guard_intact(guard, float("nan"))
    assert guard_intact(acc_buf, -(2**31))
    rows = np.unique(np.concatenate([[0, m - 1], rng.integers(0, m, 24)]))
    products = a_np[rows].astype(np.float64) @ w_np.astype(np.float64).T  # exact: below 2^53
    assert np.array_equal(host(acc)[rows], products.astype(np.int64))


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,offset", [(353, 2451, 1120, 0), (669, 2778, 192, 0), (343, 956, 96, 1)])
def test_ring_scalar_stores(ops, m, n, k, offset):
    """channel_mm with n % 4 != 0 or a channel scale off 8-byte alignment: the epilogue
    loads and stores single values."""
    _, a_np, w_np, sa_np, sw_np = inputs(m, n, k)
    sw = to_dev(np.concatenate([sw_np[:1]] * offset + [sw_np]))[offset:]
    out, buf = with_guard((m, n), torch.bfloat16, float("nan"))
    print(f"ring scalar stores m={m} n={n} k={k} offset={offset}", flush=True)
    ops.channel_mm(to_dev(a_np), to_dev(w_np.view(np.uint8) ^ 0x80), to_dev(sa_np), sw, out)
    torch.cuda.synchronize()
    assert guard_intact(buf, float("nan"))
    assert np.array_equal(bf16_bits(out), O.fused_channel_mm(a_np, w_np, sa_np, sw_np))


@pytest.mark.gpu
def test_ring_in_graph_replays(ops):
    """Captured once, replayed on other activations, with eager work in between."""
    m, n, k = 669, 2780, 1888
    _, a_np, w_np, sa_np, sw_np = inputs(m, n, k)
    a, w, sa, sw = to_dev(a_np), to_dev(w_np), to_dev(sa_np), to_dev(sw_np)
    out, ref = (torch.empty(m, n, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    ops.fused_channel_mm(a, w, sa, sw, out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.fused_channel_mm(a, w, sa, sw, out)
    for rep in range(3):
        a.neg_() if rep else None
        out.fill_(float(rep))
        ops.fused_channel_mm(a, w, sa, sw, ref, 5)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(bf16_bits(out), bf16_bits(ref)), rep
