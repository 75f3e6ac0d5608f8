"""INT4-g128 x INT8 group sums at their largest, on every tile height.

All activations at one extreme and all levels at the other: each 128-K group
sums to +-128 * 127 * 15, and K groups of it with a power-of-two scale are exact
in fp32, so the fp32 output is known exactly.
"""
import pytest
import torch

from test_gpu_parity import pk  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(33, 128, 128), (2048, 1024, 256), (4100, 1024, 384), (7500, 1024, 256), (9000, 3072, 128)])
@pytest.mark.parametrize("level,zero,x", [(15, 0, -127), (0, 15, -127), (15, 0, 127), (3, 3, 127)])
def test_extreme_group_sums(pk, m, n, k, level, zero, x):  # noqa: F811
    q = torch.full((n, k // 8), 0, dtype=torch.int32, device="cuda")
    q.view(torch.uint8).fill_(level * 17)
    scale = torch.full((n, k // 128), 2.0**-6, dtype=torch.float16, device="cuda")
    zeros = torch.full((n, k // 128), float(zero), dtype=torch.float16, device="cuda")
    x8 = torch.full((m, k), x, dtype=torch.int8, device="cuda")
    # one different element a row, so that rows and columns are told apart
    rows = torch.arange(m, device="cuda")
    x8[rows, rows % k] = (rows % 7 - 3).to(torch.int8)
    xs = torch.full((m,), 0.5, device="cuda")
    out = torch.empty((m, n), device="cuda")
    pk.call("pk_linear_int4g128_a8", x8, xs, q, scale, zeros, None, out, 1, m, n, k)
    want = (x8.double().sum(1) * (level - zero) * 2.0**-7)[:, None].expand(m, n)
    assert torch.equal(out.double(), want)
