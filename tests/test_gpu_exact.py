"""The short correctly rounded quotients and roots (gbr_exact.h) on the GPU:
reciprocals and roots over every float of their range, quotients over all that
the texture level of detail and the noise model's last step can form and over
2^30 drawn pairs of each other range (tests/cpp/exact_sweep.hip)."""
import ctypes
import os

import numpy as np
import pytest

from habitat_sim_amd import hip

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "_build", "libexact_sweep.so")


class Result(ctypes.Structure):
    _fields_ = [("checked", ctypes.c_uint64), ("bad", ctypes.c_uint64), ("a", ctypes.c_uint32), ("b", ctypes.c_uint32)]


def _sweep(name, *args):
    hip.hip()  # the runtime that the library uses
    res = Result()
    assert getattr(ctypes.CDLL(LIB), name)(*args, ctypes.byref(res)) == 0
    a, b = np.array([res.a, res.b], np.uint32).view(np.float32)
    assert res.bad == 0, f"{name}: {res.bad} of {res.checked} differ, for instance {a!r}, {b!r}"
    return res.checked


def test_every_reciprocal():
    assert _sweep("exact_rcp") == 2 * (252 * (1 << 23) + 1)


def test_every_root():
    assert _sweep("exact_sqrt") == 160 * (1 << 23) + 1


def test_quotients_of_the_level_of_detail():
    assert _sweep("exact_div_log2") == 1 << 23


def test_quotients_of_the_noise_model():
    num = np.float32(np.float32(35.130) * np.float32(8.0))
    assert _sweep("exact_div_integers", ctypes.c_float(num), ctypes.c_uint64(1 << 23)) == 1 << 23


@pytest.mark.parametrize("name,a,b,q", [
    ("the header's whole range", (-100, 125), (-126, 125), (-125, 126)),
    ("depth over factor of the noise model", (-10, 3), (-17, 2), (-14, 20)),
    ("vector component over length", (-60, 29), (-30, 29), (-90, 0)),
    ("distance over range of a light", (-30, 29), (-30, 29), (-60, 60)),
    ("attenuation over squared distance", (-48, 0), (0, 60), (-108, 0)),
    ("linear depth", (-60, 59), (-60, 59), (-60, 60))])
def test_drawn_quotients(name, a, b, q):
    n = 1 << 30
    checked = _sweep("exact_div", ctypes.c_uint64(len(name)), ctypes.c_uint64(n), (ctypes.c_int * 6)(*a, *b, *q))
    assert checked > n // 4, checked
