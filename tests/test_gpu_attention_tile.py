"""The fp32 attention tile kernel at the edges of its tiles, against the oracle:
the short form past 128 rows (ragged last tiles, windows narrower than the model's,
fewer valid rows than rows), and values that are not finite, which may reach only the
queries whose window holds them (oracle run on the finite values for the others).
Bar: max|err| <= 1e-2 * RMS(oracle), that of the short form's other tests."""
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
