"""The FP32 limiters as medians with 0 (csrc/physics.hpp tmed3: MonCen's half slope, minmod, the limited PPM
offsets) against their branch forms in numpy float32, on random pairs and pairs on each switch."""
import ctypes as C
import os

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "glmmhdturb_amd", "_build", "liblimitercheck.so")
f = np.float32


def _pairs(kind):
    r = np.random.default_rng(9)
    a = (r.standard_normal(20000) * 10.0 ** r.uniform(-6, 3, 20000)).astype(f)
    b = (r.standard_normal(20000) * 10.0 ** r.uniform(-6, 3, 20000)).astype(f)
    if kind == "switch":
        w = r.integers(0, 8, a.size)
        b = np.choose(w, [a, f(2) * a, f(0.5) * a, f(3) * a, a / f(3), -a, np.zeros_like(a), np.nextafter(a, f(np.inf))]).astype(f)
        a = np.where(r.random(a.size) < 0.05, f(0), a)
    return a, b


@pytest.mark.parametrize("kind", ["random", "switch"])
def test_f32_limiters_equal_their_branch_forms(kind):
    if not os.path.exists(LIB):
        pytest.skip("host limiter build is missing (tests/native)")
    lib = C.CDLL(LIB)
    a, b = _pairs(kind)
    out = [np.empty_like(a) for _ in range(4)]
    ptr = [x.ctypes.data_as(C.POINTER(C.c_float)) for x in (a, b, *out)]
    lib.lc_limiters_f32(*ptr, C.c_long(a.size))
    same = np.sign(a) * np.sign(b) > 0
    small = np.minimum(np.abs(a), np.abs(b))
    half = np.minimum(small, f(0.25) * np.abs(a + b))
    assert np.array_equal(out[0], np.where(same, np.copysign(half, a), f(0)))                       # MonCen / 2
    assert np.array_equal(out[1], np.where(same, np.copysign(small, a), f(0)))                      # minmod
    for k, (x, y) in enumerate(((a, b), (b, a))):                                                   # PPM offsets
        assert np.array_equal(out[2 + k], np.where(same, np.copysign(np.minimum(np.abs(x), f(2) * np.abs(y)), x), f(0)))
