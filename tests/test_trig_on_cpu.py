"""The double-precision trigonometry of device_trig.h, compiled for the host, against numpy's
double functions rounded to float: equal wherever the double result is not within its own error
of the middle between two floats (at most one argument in 10^6), and then one unit apart."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("trig") / "libtrig_emu.so")
    subprocess.check_call(["/opt/rocm/bin/hipcc", "-O2", "-std=c++17", "-fPIC", "-shared", "--offload-arch=gfx950", "-ffp-contract=off",
                           "-fno-fast-math", os.path.join(HERE, "emu", "trig_emu.hip"), "-o", lib])
    return C.CDLL(lib)


def test_trig_rounds_like_the_double_functions(emu):
    rs = np.random.RandomState(3)
    n = 1 << 20
    x = np.concatenate([rs.uniform(-7, 7, n), rs.uniform(-1e-3, 1e-3, n)]).astype(np.float32)
    y = np.concatenate([rs.uniform(-1, 1, n), 1 - 10.0 ** rs.uniform(-7, 0, n)]).astype(np.float32)
    edge = np.array([0.0, -0.0, 1.0, -1.0, np.pi / 4, np.pi / 2, np.pi, 2 * np.pi, -np.pi / 4, 0.41421357], np.float32)
    zero = np.array([0.0, -0.0, 0.0, -0.0], np.float32)
    x = np.concatenate([x, edge, np.ones_like(edge), zero])
    y = np.concatenate([y, np.ones_like(edge), np.clip(edge, -1, 1), zero[[0, 0, 1, 1]]])
    out = np.zeros((len(x), 4), np.float32)
    emu.emu_trig(x.ctypes.data_as(C.c_void_p), y.ctypes.data_as(C.c_void_p), C.c_int64(len(x)), out.ctypes.data_as(C.c_void_p))
    xd, yd = x.astype(np.float64), y.astype(np.float64)
    for k, want in enumerate([np.sin(xd), np.cos(xd), np.arccos(yd), np.arctan2(yd, xd)]):
        want = want.astype(np.float32)
        assert np.mean(out[:, k] != want) <= 1e-6, k
        assert np.array_equal(np.signbit(out[:, k]), np.signbit(want)), k
        assert np.all(np.abs(out[:, k] - want) <= np.spacing(np.abs(want))), k


def test_trig_passes_nan_on(emu):
    x, y = np.array([np.nan, 0.5], np.float32), np.array([0.5, 1.0000001], np.float32)
    out = np.zeros((2, 4), np.float32)
    emu.emu_trig(x.ctypes.data_as(C.c_void_p), y.ctypes.data_as(C.c_void_p), C.c_int64(2), out.ctypes.data_as(C.c_void_p))
    assert np.isnan(out[0, [0, 1, 3]]).all() and np.isnan(out[1, 2])
