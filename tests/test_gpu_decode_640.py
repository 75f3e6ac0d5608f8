"""The 64-workgroup decode kernel of the model's width (H = 640) at the edges of
its layout, against the oracle: joint rows below, at and past the 16 a
workgroup owns (1024), at its most (1088) and one past it (the general kernel),
eight durations, fewer frames than a window, an encoder stride above the width.
Tokens, final frame and joint steps are exact, the prediction within 1e-4."""
import numpy as np
import pytest

from test_gpu_parity import decode_case, dev, host, orc, pk  # noqa: F401

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("form", ["fp16", "long"])
@pytest.mark.parametrize("T,D,frames,stride,int8", [
    (1019, 5, 60, 640, True), (1080, 8, 60, 648, True), (1081, 8, 40, 640, False), (3, 1, 7, 640, False), (1025, 5, 1, 642, True),
    (1025, 5, 33, 640, False)])
def test_decode_640_edges(pk, orc, form, T, D, frames, stride, int8):  # noqa: F811
    H = 640
    lstm, proj, wj, bj, enc, emb = decode_case(H, T, D, frames, 4000 + T + frames, int8)
    joint = (*orc.quantize_int8_rows(wj), bj) if int8 else (wj, None, bj)
    wide = np.zeros((frames, stride), np.float16)
    wide[:, :H] = enc
    toks = torch.zeros(frames * 10 + 1, dtype=torch.int32, device="cuda")
    res = torch.zeros(4, dtype=torch.int32, device="cuda")
    wbytes = pk.lib.pk_tdt_decode_workspace_bytes(H)
    work = torch.full((wbytes // 4,), -1, dtype=torch.int32, device="cuda")  # the call overwrites it
    d = [dev(a) for a in lstm]
    tail = (dev(proj[0]), dev(proj[1]), dev(joint[0]), int(int8), None if joint[1] is None else dev(joint[1]), dev(bj), H, T, D, 10,
            toks, toks.numel(), res, work, wbytes)
    if form == "fp16":
        pk.call("pk_tdt_decode", dev(wide), frames, stride, dev(emb), *d, *tail)
        ref_toks, ref_frame, ref_pred = orc.tdt_decode(enc, emb, lstm, proj, joint, T, D)
    else:
        table = torch.zeros((T - 1, 4 * H), dtype=torch.float16, device="cuda")
        pk.launch_linear(dev(emb), d[0], None, None, table, T - 1, 4 * H, H)
        pk.call("pk_tdt_decode_long", dev(wide), frames, stride, table, *d[1:], *tail)
        ref_toks, ref_frame, ref_pred = orc.tdt_decode_long(enc, host(table), lstm[1:], proj, joint, T, D)
    count, frame, status, steps = (int(v) for v in host(res))
    assert status == 0 and (count, frame) == (len(ref_toks), ref_frame) and steps >= count
    assert np.array_equal(host(toks)[:count], ref_toks)
    pred = host(work).view(np.float32)[1032 + 8 * H:1032 + 9 * H]
    assert np.max(np.abs(pred - ref_pred)) <= 1e-4 * max(1.0, float(np.max(np.abs(ref_pred))))
