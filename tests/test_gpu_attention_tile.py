"""The short form past 128 rows at the edges of its kernels' tiles, against the oracle
(ragged last tiles, windows narrower than the model's, fewer valid rows than rows, on
the wave kernel and on the fp32 tile kernel), and values that are not finite, which may
reach only the queries whose window holds them (oracle run on the finite values for the
others).  Bar: max|err| <= 1e-2 * RMS(oracle), that of the short form's other tests."""
import numpy as np
import pytest

from test_gpu_attention import TOL, dev, host, inputs, orc, pk  # noqa: F401

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def run(pk, args, rows, padded, valid, left, right):  # noqa: F811
    out = torch.full((padded, 1024), 0x5A5A, dtype=torch.int16, device="cuda")
    pk.call("pk_local_relpos_attention", *[dev(a) for a in args], out, rows, padded, valid, left, right)
    return host(out).view(np.float16)


@pytest.mark.parametrize("padded,rows,valid,left,right", [
    (129, 129, 129, 128, 128), (145, 140, 150, 128, 128), (300, 300, 271, 128, 128), (272, 272, 272, 128, 1), (160, 160, 160, 0, 128),
    (200, 200, 17, 100, 37), (400, 399, 390, 7, 3), (144, 144, 0, 128, 128)])
def test_tile_edges(pk, orc, padded, rows, valid, left, right):  # noqa: F811
    q, k, v, pos, bu, bv = inputs(900 + padded + left, max(padded, valid))
    got = run(pk, (q, k, v, pos, bu, bv), rows, padded, valid, left, right)
    live = min(rows, valid, padded)
    assert not got[live:].view(np.uint16).any()
    if live == 0:
        return
    ref = orc.local_attention_short(q, k, v, pos, bu, bv, rows, valid_rows=valid, left=left, right=right)
    g, r = got[:live].astype(np.float64), ref[:live].astype(np.float64)
    assert np.abs(g - r).max() <= TOL * np.sqrt((r ** 2).mean())


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_tile_non_finite_values(pk, orc, bad):  # noqa: F811
    padded, left, right, at = 192, 20, 9, 100
    q, k, v, pos, bu, bv = inputs(77, padded)
    spoilt = v.copy()
    spoilt[at, 5::7] = bad
    got = run(pk, (q, k, spoilt, pos, bu, bv), padded, padded, padded, left, right).astype(np.float64)
    ref = orc.local_attention_short(q, k, v, pos, bu, bv, padded, valid_rows=padded, left=left, right=right).astype(np.float64)
    sees = (np.arange(padded) - left <= at) & (at <= np.arange(padded) + right)
    cols = np.arange(1024) % 1024
    hit = np.zeros(1024, bool)
    hit[5::7] = True
    clean = ~(sees[:, None] & hit[cols][None, :])
    assert not np.isfinite(got[~clean]).any()
    assert np.isfinite(got[clean]).all()
    assert np.abs(got - ref)[clean].max() <= TOL * np.sqrt((ref ** 2).mean())


@pytest.mark.parametrize("rows,edge", [(16, True), (2048, False), (2064, True), (8208, True), (16400, False), (32784, True), (49168, False),
                                       (65536, True), (65552, True)])
def test_value_quantizer_row_sizes(pk, orc, rows, edge):  # noqa: F811
    """Rows at and one step past what a workgroup of each size holds, with
    near-ties (multiples of half a step), infinities and NaN: bit for bit."""
    gen = torch.Generator().manual_seed(rows)
    vt = torch.randn((1024, rows), generator=gen).half()
    vt[1::5] = (torch.randint(-14, 15, vt[1::5].shape, generator=gen) * 0.5).half()  # v / s at half-integers
    vt[1::5, 0] = 7.0
    vt[7, rows // 2], vt[12, 3], vt[12, 4], vt[17], vt[22] = float("nan"), float("inf"), float("nan"), 0, 6e-8
    vt = vt.numpy()
    el = rows * 1024
    out = torch.full((el + el // 2 + 4096,), 0xAB, dtype=torch.uint8, device="cuda")
    if edge:
        pk.call("pk_quantize_value_int4_register", dev(vt), out, el, 56.0, rows - 3)
    else:
        pk.call("pk_quantize_value_int4", dev(vt), out, el, 56.0)
    ref = orc.quantize_value_int4(vt, 56.0, edge_only=edge, valid_rows=rows - 3 if edge else rows, fill=0xAB)
    # a NaN quantizes to 0 (the oracle's conversion of NaN to int is not defined)
    for f, r in np.argwhere(np.isnan(vt)):
        ref[el + (f * rows + r) // 2] &= 0x0F if r & 1 else 0xF0
    np.testing.assert_array_equal(host(out), ref)


@pytest.mark.parametrize("padded,rows,valid,left,right", [
    (400, 399, 390, 95, 3), (512, 512, 500, 0, 128), (448, 447, 440, 60, 37), (352, 352, 352, 128, 0), (529, 529, 529, 128, 70),
    (1024, 1024, 1023, 101, 19)])
def test_tile_narrow_windows(pk, orc, padded, rows, valid, left, right):  # noqa: F811
    """Windows narrower than the model's in calls that take the tile kernel."""
    test_tile_edges(pk, orc, padded, rows, valid, left, right)


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_tile_non_finite_values_short_form(pk, orc, bad):  # noqa: F811
    """As test_tile_non_finite_values, in a call that takes the tile kernel."""
    padded, left, right = 416, 70, 40
    q, k, v, pos, bu, bv = inputs(78, padded)
    spoilt = v.copy()
    for at in (0, 200, 415):
        spoilt[at, 5::7] = bad
    got = run(pk, (q, k, spoilt, pos, bu, bv), padded, padded, padded, left, right).astype(np.float64)
    ref = orc.local_attention_short(q, k, v, pos, bu, bv, padded, valid_rows=padded, left=left, right=right).astype(np.float64)
    sees = np.zeros(padded, bool)
    for at in (0, 200, 415):
        sees |= (np.arange(padded) - left <= at) & (at <= np.arange(padded) + right)
    hit = np.zeros(1024, bool)
    hit[5::7] = True
    clean = ~(sees[:, None] & hit[None, :])
    assert not np.isfinite(got[~clean]).any()
    assert np.isfinite(got[clean]).all()
    assert np.abs(got - ref)[clean].max() <= TOL * np.sqrt((ref ** 2).mean())


@pytest.mark.parametrize("rows,valid,right", [(496, 600, 0), (490, 600, 0), (496, 500, 2), (512, 4096, 0)])
def test_tile_keys_end_with_the_window(pk, orc, rows, valid, right):  # noqa: F811
    """valid_rows past the rows of Q, K and V, which end with the last key of the last
    query's window."""
    left, keys = 128, min(valid, rows + right)
    q, k, v, pos, bu, bv = inputs(500 + rows + right, keys)
    got = run(pk, (q[:rows], k, v, pos, bu, bv), rows, rows, valid, left, right)
    ref = orc.local_attention_short(q, k, v, pos, bu, bv, rows, valid_rows=keys, left=left, right=right)
    g, r = got.astype(np.float64), ref[:rows].astype(np.float64)
    assert np.abs(g - r).max() <= TOL * np.sqrt((r ** 2).mean())


@pytest.mark.parametrize("rows,at", [(752, 3), (752, 750), (4000, 100), (4000, 3990), (15008, 40)])
def test_boundary_tiles_non_finite_values(pk, orc, rows, at):  # noqa: F811
    """NaN bytes of the long form's e4m3 V (the tc form) in a boundary tile's keys
    reach the queries whose window holds them and no others of the boundary."""
    q, k, v, pos, bu, bv = inputs(600 + at, rows)
    value = torch.empty((1024, rows), dtype=torch.uint8, device="cuda")
    pk.call("pk_quantize_fp8_fixed_transpose", dev(v), value, rows, 56.0)
    outs = []
    for spoil in (False, True):
        if spoil:
            value[5::7, at] = 0x7F
        out = torch.empty((rows, 1024), dtype=torch.int16, device="cuda")
        pk.call("pk_local_relpos_attention_tc_scores", dev(q), dev(k), dev(v), value, dev(pos), dev(bu), dev(bv), out, rows, rows, rows,
                128, 128, rows)
        outs.append(host(out).view(np.float16).astype(np.float64))
    clean_run, got = outs
    hit = np.zeros(1024, bool)
    hit[5::7] = True
    sees = np.abs(np.arange(rows) - at) <= 128
    # queries of the fp32 boundary tiles: below the first whole window, past the last
    edge = (np.arange(rows) < 128) | (np.arange(rows) >= 16 * ((rows - 144) // 16 + 1))
    assert np.isnan(got[np.ix_(sees & edge, hit)]).all()
    other = edge[:, None] & ~(sees[:, None] & hit[None, :])
    assert np.isfinite(got[other]).all()
    # the same sums in another order (fp32), rounded to fp16
    assert np.abs(got - clean_run)[other].max() <= 2 ** -10 * np.abs(clean_run[other]).max()
