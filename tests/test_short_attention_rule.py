"""The short form's choice of kernel (csrc/pk_attention_rule.hpp), compiled for the
host: the wave kernel wherever the tile kernel was measured slower on 256 CUs
(narrow windows, few rows, a nearly empty last round of tiles), the tile kernel
where it was clearly faster.  And the rows that a tile of the tile kernel loads:
only queries that have an output and keys that some query sees."""
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
                   'extern "C" int rule(int live, int keys, int cus) { return pk::short_takes_tile(live, keys, cus); }\n'
                   'extern "C" int last_key(int qb, int live, int valid, int right) { return pk::tile_last_key(qb, live, valid, right); }\n'
                   'extern "C" int key_row(int key, int last) { return pk::tile_key_row(key, last); }\n'
                   'extern "C" int query_row(int query, int live) { return pk::tile_query_row(query, live); }\n')
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(PKG, "csrc"), str(src), "-o", str(lib)], check=True)
    return ctypes.CDLL(str(lib))


def test_rule(rule):
    assert [c for c in WAVE if rule.rule(*c, 256)] == []
    assert [c for c in TILE if not rule.rule(*c, 256)] == []


@pytest.mark.parametrize("rows,padded,valid,left,right", [
    (496, 496, 600, 128, 0), (496, 496, 600, 128, 37), (300, 300, 271, 128, 128), (272, 272, 272, 128, 1), (512, 512, 2**31 - 1, 128, 0),
    (400, 399, 390, 95, 3), (145, 140, 150, 128, 128), (17, 32, 40, 0, 0), (1, 16, 1, 128, 128), (33, 64, 64, 7, 128)])
def test_tile_rows(rule, rows, padded, valid, left, right):
    """Every load of a tile (272 key columns, 16 queries) stays in the rows that the
    wave kernel reads: queries below `live`, keys in some live query's window.  valid
    may exceed padded; K of 496 rows with valid = 600 and no right context ends at
    key 495."""
    live = min(rows, padded, valid)
    for qb in range(0, live, 16):
        last_query = min(qb + 15, live - 1)
        lo, hi = max(0, qb - left), min(valid - 1, last_query + right)
        last = rule.last_key(qb, live, valid, right)
        assert last == hi
        for col in range(272):
            row = rule.key_row(qb - left + col, last)
            assert lo <= row <= hi
            if lo <= qb - left + col <= hi:
                assert row == qb - left + col
        for q in range(16):
            assert rule.query_row(qb + q, live) == min(qb + q, live - 1)


def test_tile_kernel_takes_its_rows_from_there():
    text = open(os.path.join(PKG, "csrc", "pk_attention_tile.hpp")).read()
    assert "p.valid_rows - 1" not in text and "p.padded_rows - 1" not in text
    assert text.count("tile_key_row(") == 2 and text.count("tile_query_row(") == 1 and text.count("tile_last_key(") == 1
