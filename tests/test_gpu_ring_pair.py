"""Small grids two K-steps per barrier, and GLU on small grids: every output row
equals, bit for bit, the same row of a launch large enough for the persistent
engines (which accumulate each output over K in the same order)."""
import numpy as np
import pytest

from test_gpu_parity import pk  # noqa: F401

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
LARGE = 40960


def operands(fmt, m, n, k):
    g = torch.Generator(device="cuda")
    g.manual_seed(m * 7 + n + k)
    if fmt == 1:
        a = torch.randint(-127, 128, (LARGE, k), generator=g, device="cuda", dtype=torch.int8)
        b = torch.randint(-127, 128, (n, k), generator=g, device="cuda", dtype=torch.int8)
    else:
        a = torch.randn((LARGE, k), generator=g, device="cuda").to(torch.float8_e4m3fn).view(torch.uint8)
        b = torch.randn((n, k), generator=g, device="cuda").to(torch.float8_e4m3fn).view(torch.uint8)
    return a, b, torch.rand(LARGE, generator=g, device="cuda"), torch.rand(n, generator=g, device="cuda") * 0.01


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("m,n,k", [(1, 128, 256), (31, 144, 512), (33, 1024, 768), (96, 1024, 4096), (65, 4096, 2560), (500, 3072, 1024),
                                   (750, 1024, 4096), (496, 4096, 768), (40, 1024, 640)])
def test_rows_equal_large_grid(pk, fmt, m, n, k):  # noqa: F811
    a, b, rs, ws = operands(fmt, m, n, k)
    tile = pk.gemm_tile(fmt, pk.EPI_F16, m, n, True)
    assert tile[0] in (32, 64) and tile[2] > 2
    for epi, dtype in ((pk.EPI_F16, torch.float16), (pk.EPI_F32, torch.float32), (pk.EPI_F8, torch.uint8)):
        small = torch.full((m + 1, n), 77, dtype=dtype, device="cuda")
        large = torch.zeros((LARGE, n), dtype=dtype, device="cuda")
        pk.gemm(fmt, epi, a, b, m, n, k, small, w_scales=ws, row_scales=rs)
        pk.gemm(fmt, epi, a, b, LARGE, n, k, large, w_scales=ws, row_scales=rs)
        assert torch.equal(small[:m], large[:m]), f"epilogue {epi}"
        assert bool((small[m] == 77).all())
    res = torch.randn((m, n), device="cuda").half()
    out, ref = res.clone(), torch.zeros((LARGE, n), dtype=torch.float16, device="cuda")
    ref[:m] = res
    pk.gemm(fmt, pk.EPI_F16, a, b, m, n, k, out, w_scales=ws, row_scales=rs, residual=out, out_scale=0.5, res_scale=1.0)
    pk.gemm(fmt, pk.EPI_F16, a, b, LARGE, n, k, ref, w_scales=ws, row_scales=rs, residual=ref, out_scale=0.5, res_scale=1.0)
    assert torch.equal(out, ref[:m])


@pytest.mark.parametrize("m,valid", [(16, 9), (250, 250), (752, 741), (1500, 1500)])
def test_glu_small_grids(pk, m, valid):  # noqa: F811
    a, b, rs, ws = operands(0, m, 2048, 1024)
    small = torch.full((m + 1, 1024), 77, dtype=torch.float16, device="cuda")
    large = torch.zeros((LARGE, 1024), dtype=torch.float16, device="cuda")
    pk.call("pk_conv_glu_fp8", a, b, ws, rs, small, m, valid)
    pk.call("pk_conv_glu_fp8", a, b, ws, rs, large, LARGE, LARGE)
    assert torch.equal(small[:valid], large[:valid])
    assert not small[valid:m].any() and bool((small[m] == 77).all())


def test_integer_sums(pk):  # noqa: F811
    """INT8 through the pairs against exact integer products."""
    m, n, k = 70, 256, 1024
    a, b, _, _ = operands(1, m, n, k)
    acc = torch.empty((m, n), dtype=torch.int32, device="cuda")
    pk.call("pk_linear_int8_accumulate", a, b, acc, m, n, k)
    ref = a[:m].cpu().numpy().astype(np.int64) @ b.cpu().numpy().astype(np.int64).T
    assert np.array_equal(acc.cpu().numpy(), ref)
