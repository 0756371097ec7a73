"""The quotient and remainder that turn a work unit into its tile and pass
(zillumgl_amd/csrc/zgl_math.h divUniform), against whole-number division: around every
multiple that its rounded reciprocal could miss, up to the largest 31-bit numerator."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("div") / "div_probe.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC",
                    os.path.join(HERE, "native", "div_probe.cpp"), "-o", out], check=True)
    L = C.CDLL(out)
    ip = C.POINTER(C.c_int32)
    L.probe_div.argtypes = [ip, C.c_int32, ip, ip, C.c_int64]
    L.probe_div.restype = None

    def run(n, d):
        q, r = np.empty_like(n), np.empty_like(n)
        L.probe_div(n.ctypes.data_as(ip), d, q.ctypes.data_as(ip), r.ctypes.data_as(ip), n.size)
        return q, r
    return run


@pytest.mark.parametrize("d", [1, 2, 3, 7, 64, 65, 240, 255, 641, 2048, 65535, 65536, 65537, 2**30 + 1, 2**31 - 1])
def test_quotient_and_remainder(probe, d):
    top = 2**31 - 1
    k = np.unique(np.concatenate([np.arange(0, 2000), np.random.default_rng(d).integers(0, top // d + 1, 20000),
                                  np.arange(max(0, top // d - 2000), top // d + 1)])).astype(np.int64)
    n = (k[:, None] * d + np.array([-2, -1, 0, 1, 2])).ravel()
    n = np.concatenate([n, np.array([top - 1, top])])
    n = np.unique(n[(n >= 0) & (n <= top)])
    q, r = probe(n.astype(np.int32), d)
    assert np.array_equal(q.astype(np.int64), n // d)
    assert np.array_equal(r.astype(np.int64), n % d)
