"""Frames whose joint scores are all NaN (an infinite encoder feature against weights
of 0) in the scan and in both decoders: token 0 with duration 0, as
pk_joint_gemv and the oracle decide, up to max_symbols of them a frame."""
import numpy as np
import pytest

from test_gpu_parity import decode_case, dev, host, orc, pk  # noqa: F401

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
BAD = (0, 9, 10, 30)  # frames with the infinite feature


def spoilt(H, T, D, frames, seed, int8):
    case = list(decode_case(H, T, D, frames, seed, int8))
    lstm, proj, wj, bj, enc, emb = case
    wj[:, 3] = 0
    enc[[f for f in BAD if f < frames], 3] = np.inf
    return lstm, proj, wj, bj, enc, emb


@pytest.mark.parametrize("form", ["fp16", "long"])
@pytest.mark.parametrize("H,T,int8", [(640, 1025, True), (640, 1081, False), (512, 1025, True), (128, 200, False)])
def test_decode(pk, orc, form, H, T, int8):  # noqa: F811
    D, frames = 5, 37
    lstm, proj, wj, bj, enc, emb = spoilt(H, T, D, frames, 6000 + H + T, int8)
    joint = (*orc.quantize_int8_rows(wj), bj) if int8 else (wj, None, bj)
    toks = torch.zeros(frames * 10 + 1, dtype=torch.int32, device="cuda")
    res = torch.zeros(4, dtype=torch.int32, device="cuda")
    wbytes = pk.lib.pk_tdt_decode_workspace_bytes(H)
    work = torch.zeros(wbytes // 4, dtype=torch.int32, device="cuda")
    d = [dev(a) for a in lstm]
    tail = (dev(proj[0]), dev(proj[1]), dev(joint[0]), int(int8), None if joint[1] is None else dev(joint[1]), dev(bj), H, T, D, 10,
            toks, toks.numel(), res, work, wbytes)
    if form == "fp16":
        pk.call("pk_tdt_decode", dev(enc), frames, H, dev(emb), *d, *tail)
        ref_toks, ref_frame, _ = orc.tdt_decode(enc, emb, lstm, proj, joint, T, D)
    else:
        table = torch.zeros((T - 1, 4 * H), dtype=torch.float16, device="cuda")
        pk.launch_linear(dev(emb), d[0], None, None, table, T - 1, 4 * H, H)
        pk.call("pk_tdt_decode_long", dev(enc), frames, H, table, *d[1:], *tail)
        ref_toks, ref_frame, _ = orc.tdt_decode_long(enc, host(table), lstm[1:], proj, joint, T, D)
    count, frame, status, _ = (int(v) for v in host(res))
    assert status == 0 and (count, frame) == (len(ref_toks), ref_frame)
    assert np.array_equal(host(toks)[:count], ref_toks)
    assert list(ref_toks[:10]) == [0] * 10  # frame 0 is one of them


@pytest.mark.parametrize("int8", [False, True])
def test_scan_and_gemv(pk, orc, int8):  # noqa: F811
    H, T, D, frames = 640, 1025, 5, 20
    _, _, wj, bj, enc, _ = spoilt(H, T, D, frames, 6100, int8)
    w, s = orc.quantize_int8_rows(wj) if int8 else (wj, None)
    pred = (np.random.default_rng(3).standard_normal(H) * 0.3).astype(np.float32)
    args = (dev(w), int(int8), None if s is None else dev(s), dev(bj), dev(enc), dev(pred))
    decision = torch.full((1, 2), -1, dtype=torch.int32, device="cuda")
    scores = torch.zeros((1, T + D), device="cuda")
    pk.call("pk_joint_gemv", *args, scores, decision, T + D, H, T, D, 1, H)
    assert np.isnan(host(scores)).all() and host(decision).tolist() == [[0, 0]]
    state = torch.zeros(4, dtype=torch.int32, device="cuda")
    work = torch.zeros(2304, dtype=torch.int32, device="cuda")
    pk.call("pk_joint_scan", *args, T + D, H, T, D, frames, H, 10, state, work)
    assert host(state).tolist() == [0, 1, 0, 1]  # token 0, still at frame 0, one symbol
