"""parakeet_linear.call beyond the launches its table holds: entry points without a
stream argument, a stream handle given in its place, and how wrong names and
argument counts are refused.  Nothing here launches a kernel."""
import ctypes

import numpy as np
import pytest

import parakeet_linear as pk

torch = pytest.importorskip("torch")


def test_entries_without_a_stream():
    out = torch.zeros(7, dtype=torch.int64)
    pk.call("pk_exl3_layout", 1000, 640, 4, out, stream=0)
    ref = np.zeros(7, np.uint64)
    assert pk.lib.pk_exl3_layout(1000, 640, 4, ref.ctypes.data) == 0
    assert out.tolist() == ref.tolist()
    pk.call("pk_estimate_linear", 1, 1000, 640, 0, out, stream=0)
    assert out[:6].tolist() == [1000, 640, 1024, 640, 1024 * 640, 640 * 4]
    with pytest.raises(pk.PkError, match="pk_exl3_layout: status -.*bpw"):
        pk.call("pk_exl3_layout", 1000, 640, 9, out, stream=0)


def test_entries_ending_in_another_argument():
    pk.call("pk_gemm_k_split", pk.FMT_G128A8, pk.EPI_F32, 750, 1024, 4096, stream=0)
    with pytest.raises(pk.PkError, match="pk_gemm_k_split: status -4"):
        pk.call("pk_gemm_k_split", 99, pk.EPI_F32, 750, 1024, 4096, stream=0)


def test_stream_handle_in_its_place():
    # rows = -1 is refused before any launch
    for args, kw in (((None, None, 1.0, -1), {"stream": 0}), ((None, None, 1.0, -1, 0), {"stream": 0})):
        with pytest.raises(pk.PkError, match="negative element count"):
            pk.call("pk_quantize_fp8", *args, **kw)


def test_wrong_names_and_counts_are_named():
    with pytest.raises(AttributeError, match="pk_no_such_entry"):
        pk.call("pk_no_such_entry", 1, stream=0)
    with pytest.raises((TypeError, ctypes.ArgumentError)):
        pk.call("pk_quantize_fp8", None, None, stream=0)
