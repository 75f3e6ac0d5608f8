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


@pytest.mark.parametrize("m,k", [(1, 640), (96, 128), (96, 640), (250, 384), (500, 640), (752, 1152), (1500, 640)])
def test_glu_odd_steps(pk, m, k):  # noqa: F811
    """GLU through pk_gemm with K an odd multiple of 128: the plain ring on 32-row
    tiles, the two-waves-per-SIMD ring on 64- and 128-row ones."""
    n, glu = 2048, 6
    assert pk.gemm_tile(0, glu, m, n)[0] in (32, 64, 128)
    a, b, rs, ws = operands(0, m, n, k)
    small = torch.full((m + 1, n // 2), 77, dtype=torch.float16, device="cuda")
    large = torch.zeros((LARGE, n // 2), dtype=torch.float16, device="cuda")
    pk.gemm(0, glu, a, b, m, n, k, small, w_scales=ws, row_scales=rs, ldo=n // 2)
    pk.gemm(0, glu, a, b, LARGE, n, k, large, w_scales=ws, row_scales=rs, ldo=n // 2)
    assert torch.equal(small[:m], large[:m]) and bool((small[m] == 77).all()) and bool(small[:m].any())


def test_integer_sums(pk):  # noqa: F811
    """INT8 through the pairs against exact integer products."""
    m, n, k = 70, 256, 1024
    a, b, _, _ = operands(1, m, n, k)
    acc = torch.empty((m, n), dtype=torch.int32, device="cuda")
    pk.call("pk_linear_int8_accumulate", a, b, acc, m, n, k)
    ref = a[:m].cpu().numpy().astype(np.int64) @ b.cpu().numpy().astype(np.int64).T
    assert np.array_equal(acc.cpu().numpy(), ref)


@pytest.mark.parametrize("m,k", [(16, 128), (272, 256), (528, 384), (16400, 512), (8208, 4096)])
def test_sparse_contract_stages(pk, m, k):  # noqa: F811
    """The sparse contract's three-stage ring across tiles: one to four K-steps
    (fewer than stages, and not a multiple of them), several tiles a workgroup,
    ragged rows.  Exact inputs (0, +-1 activations, +-2^i weights, scales a power
    of two), so the fp16 result is known: max|err| = 0."""
    g = torch.Generator(device="cuda")
    g.manual_seed(m + k)
    dense = torch.zeros((m, k // 4, 4), device="cuda")
    pos = torch.randint(0, 3, (m, k // 4), generator=g, device="cuda")
    first, second = pos, torch.full_like(pos, 3)
    val = torch.randint(-1, 2, (2, m, k // 4), generator=g, device="cuda").float()
    dense.scatter_(2, first[..., None], val[0][..., None]).scatter_(2, second[..., None], val[1][..., None])
    codes = val.permute(1, 2, 0).reshape(m, k // 2).to(torch.float8_e4m3fn).view(torch.uint8)
    nib = (first | (second << 2)).to(torch.uint8)
    meta = (nib[:, 0::2] | (nib[:, 1::2] << 4)).contiguous()
    buf = torch.cat([codes.reshape(-1), meta.reshape(-1)])
    w = torch.randint(-2, 3, (1024, k), generator=g, device="cuda").float()
    scales = torch.full((1024,), 0.125, device="cuda")
    out = torch.randint(-8, 9, (m, 1024), generator=g, device="cuda").half()
    want = out.double() + 0.5 * (dense.reshape(m, k).double() @ w.double().t()) * 0.125 / 16.0
    pk.call("pk_ffn_contract_fp8_sparse", buf, w.to(torch.float8_e4m3fn).view(torch.uint8), scales, out, m, k)
    assert torch.equal(out, want.half())
