"""The long form's cell functions (csrc/pk_cell.hpp), compiled for the host, against
the oracle's bit for bit: the kernels evaluate the same IEEE operations, quotients as
divisions, since one ulp can move an INT8 rounding and with it a token."""
import ctypes
import os
import re
import subprocess

import numpy as np

from conftest import PKG

SRC = os.path.join(PKG, "csrc")


def test_cell_functions_are_the_oracles(tmp_path, oracle):
    src = tmp_path / "cell.cpp"
    src.write_text('#include "pk_cell.hpp"\n'
                   'extern "C" void run(const float* v, int n, float* e, float* s, float* t, float* gs, float* gt) {\n'
                   '    for (int i = 0; i < n; ++i) {\n'
                   '        e[i] = pk::det_exp(v[i]); s[i] = pk::det_sigmoid(v[i]); t[i] = pk::det_tanh(v[i]);\n'
                   '        gs[i] = pk::det_gate(v[i], false); gt[i] = pk::det_gate(v[i], true);\n'
                   '    }\n}\n')
    lib = tmp_path / "cell.so"
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-Wno-unknown-pragmas", "-I", SRC, str(src),
                    "-o", str(lib)], check=True)
    run = ctypes.CDLL(str(lib)).run
    rng = np.random.default_rng(5)
    v = np.concatenate([rng.standard_normal(4000) * s for s in (1e-6, 0.01, 1.0, 5.0, 60.0)]
                       + [np.linspace(-0.7, 0.7, 4001), [0.0, -0.0, 104, -104, 89, -89, 200, -200, np.inf, -np.inf, np.nan]]).astype(np.float32)
    out = [np.empty_like(v) for _ in range(5)]
    run(*[a.ctypes.data_as(ctypes.c_void_p) if isinstance(a, np.ndarray) else a for a in (v, v.size, *out)])
    orc = oracle.lib()
    exp = np.array([orc.orc_det_exp(float(x)) for x in v], np.float32)
    one = np.float32(1)
    with np.errstate(over="ignore"):
        sig = one / (one + np.array([orc.orc_det_exp(float(-x)) for x in v], np.float32))
    tanh = np.array([orc.orc_det_tanh(float(x)) for x in v], np.float32)
    for got, ref in zip(out, (exp, sig, tanh, sig, tanh)):
        num = ~np.isnan(ref)
        assert np.isnan(got[~num]).all() and np.array_equal(got[num].view(np.uint32), ref[num].view(np.uint32))


def test_decoder_takes_the_cell_from_there():
    text = open(os.path.join(SRC, "pk_decode.hip")).read()
    assert '#include "pk_cell.hpp"' in text
    assert not re.search(r"__builtin_amdgcn_rcp|div_rn|det_exp", text)
