"""The token of a decision key (csrc/pk_decision.hpp), compiled for the host: every
id comes back, and an empty key (a frame whose token scores are all NaN) is token
0, the decision of pk_joint_gemv and of the oracle, never an id past the table."""
import ctypes
import os
import subprocess

import numpy as np

from conftest import PKG


def test_key_token(tmp_path, oracle):
    src = tmp_path / "key.cpp"
    src.write_text('#include "pk_decision.hpp"\n'
                   'static_assert(pk::key_token(0u) == 0);\n'
                   'extern "C" int key_token(uint32_t low) { return pk::key_token(low); }\n')
    lib = tmp_path / "key.so"
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(PKG, "csrc"), str(src), "-o", str(lib)], check=True)
    fn = ctypes.CDLL(str(lib)).key_token
    fn.argtypes, fn.restype = [ctypes.c_uint32], ctypes.c_int
    for low in (0x0000, 0x1fff, 0xe001, 0xffff):  # duration and tag bits do not matter
        assert fn(low) == 0
        for tok in (0, 1, 1024, 65533, 65534):
            assert fn(((0xffff - tok) << 16) | low) == tok
    nan = np.full(1030, np.nan, np.float32)
    assert oracle.joint_decide(nan) == (0, 0)
