"""The short form's choice of kernel (csrc/pk_attention_rule.hpp), compiled for the
host: the wave kernel wherever the tile kernel was measured slower on 256 CUs
(narrow windows, few rows, a nearly empty last round of tiles), the tile kernel
where it was clearly faster."""
import ctypes
import os
import subprocess

import pytest

from conftest import PKG

# (live queries, keys a query sees), each measured both ways
WAVE = [(0, 0), (48, 48), (96, 96), (128, 128), (129, 129), (144, 144), (152, 152), (400, 64), (128, 128), (144, 129), (200, 129), (256, 129),
        (264, 129), (144, 65), (300, 65), (384, 81), (496, 33), (511, 11), (512, 1), (520, 129), (640, 161), (768, 129), (1024, 65),
        (1040, 81), (1536, 65), (4096, 65)]
TILE = [(176, 176), (256, 257), (300, 161), (300, 257), (392, 129), (392, 97), (496, 257), (511, 129), (520, 193), (640, 225), (768, 193),
        (1024, 129), (1024, 97), (1040, 257), (1536, 129), (2048, 161), (4096, 129)]


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    src, lib = d / "rule.cpp", d / "rule.so"
    src.write_text('#include "pk_attention_rule.hpp"\n'
                   'extern "C" int rule(int live, int keys, int cus) { return pk::short_takes_tile(live, keys, cus); }\n')
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(PKG, "csrc"), str(src), "-o", str(lib)], check=True)
    return ctypes.CDLL(str(lib)).rule


def test_rule(rule):
    assert [c for c in WAVE if rule(*c, 256)] == []
    assert [c for c in TILE if not rule(*c, 256)] == []
