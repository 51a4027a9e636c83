"""CPU: the wave-wide binary GCD inversion (zkwasm-prover_amd/csrc/inv_wave.h),
host branch, with the checks and inputs of test_inv_bingcd."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from test_inv_bingcd import HERE, MODS, ROOT, _int, _limbs, _values


@pytest.fixture(scope="module")
def iw(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("iw") / "libiw.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "zkwasm-prover_amd", "csrc"),
                    os.path.join(HERE, "inv_bingcd", "check_wave.cpp"), "-o", out], check=True)
    L = ctypes.CDLL(out)
    L.ib_inv.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int]
    return L


@pytest.mark.parametrize("field", [0, 1])
def test_inverse_identity(iw, field):
    M = MODS[field]
    corr = pow(2, (32 - iw.ib_bits()) * iw.ib_steps(), M)
    for y in _values(M, 21 + field, 20000):
        v = np.zeros(8, dtype=np.uint32)
        assert iw.ib_inv(v.ctypes.data, _limbs(y).ctypes.data, field) == 1, y
        assert _int(v) < M
        assert y * _int(v) * corr % M == 1, y


@pytest.mark.parametrize("field", [0, 1])
def test_zero_is_reported(iw, field):
    v = np.zeros(8, dtype=np.uint32)
    assert iw.ib_inv(v.ctypes.data, _limbs(0).ctypes.data, field) == 0
