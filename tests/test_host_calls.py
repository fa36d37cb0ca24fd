"""The library's host code over a stand-in for the HIP runtime (tests/native/fake_hip.cpp): what it launches, waits
for and frees, in which order, and what is left when a call fails.  No GPU."""
import ctypes as C
import os
import re

import pytest

from glmmhdturb_amd import Params, _lib, step_args

LIB = os.path.join(os.path.dirname(_lib.HERE), "glmmhdturb_amd", "_build", "libhostcheck.so")


class Host:
    """The library and the stand-in's log."""

    def __init__(self, cus=256, occ=2):
        if not os.path.exists(LIB):
            pytest.skip("host build over the stand-in runtime is missing (tests/native)")
        self.lib = _lib.load(LIB)
        self.lib.fh_log.restype = C.c_char_p
        self.lib.fh_live.restype = C.c_long
        self.lib.fh_live.argtypes = [C.c_void_p]
        self.lib.fh_reset(cus, occ)

    def log(self, start=0):
        return [self.lib.fh_log(i).decode() for i in range(start, self.lib.fh_log_size())]

    def fail(self, function, nth=1):
        self.lib.fh_fail(function.encode(), nth)


def planes(n=9, base=0x10000000):
    arr, _ = _lib.plane_array([base + 0x100000 * v for v in range(n)])
    return arr


def test_a_new_contexts_slots_are_zero_on_every_stream():
    """They are cleared on the null stream, which a caller's non-blocking stream does not wait for."""
    h = Host()
    ctx = h.lib.glm_create(16, 16, 16, 8)
    log = h.log()
    at = [i for i, x in enumerate(log) if x.startswith("memset")]
    assert at and any(x in ("sync (nil)", "sync device") for x in log[at[-1] + 1:])
    h.lib.glm_destroy(ctx)
