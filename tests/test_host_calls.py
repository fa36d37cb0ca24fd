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


def boxes(n=3, edge=32):
    out = (_lib.GLMEnsBox * n)()
    for b, x in enumerate(out):
        x.nx = x.ny = x.nz = edge
        for v in range(9):
            x.u0[v], x.u1[v] = 0x20000000 + 0x1000000 * b + 0x10000 * v, 0x40000000 + 0x1000000 * b + 0x10000 * v
        x.boxlen, x.courant, x.ch_scale, x.turb_T = 1.0, 0.3, 0.25, 1.0
    return out


def ensemble(h, bx):
    e = h.lib.glm_ens_create(len(bx), bx, C.byref(step_args(Params(N=32, nz=32), 1.0, 0.0)), 8)
    assert e
    return e


def march(line):
    m = re.search(r"boxes (\S+) tiles (\S+) total (\d+)", line)
    return int(m[1], 16), int(m[2], 16), int(m[3])


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("call", [("hipMalloc", 1), ("hipMalloc", 2), ("hipMemcpy", 1), ("hipMemcpy", 2)])
def test_a_failed_configure_leaves_the_ensemble_as_it_was(call, graph):
    """The next sweep runs the old layout, whose tables are still allocated and of its size."""
    h = Host()
    bx = boxes()
    e = ensemble(h, bx)
    if graph:
        assert h.lib.glm_ens_graph(e, 1) == 0
    assert h.lib.glm_ens_step(e, 1) == 0
    before = march([x for x in h.log() if "ens_march" in x][-1])
    h.fail(*call)
    assert h.lib.glm_ens_configure(e, 1, 0, 1) != 0
    assert h.lib.glm_ens_step(e, 1) == 0
    after = march([x for x in h.log() if "ens_march" in x][-1])
    assert after == before
    assert h.lib.fh_live(after[0]) > 0 and h.lib.fh_live(after[1]) == 8 * after[2]
    # and a configure that succeeds replaces them
    assert h.lib.glm_ens_configure(e, 1, 0, 1) == 0
    assert h.lib.glm_ens_step(e, 1) == 0
    new = march([x for x in h.log() if "ens_march" in x][-1])
    assert new[2] > before[2] and h.lib.fh_live(new[1]) == 8 * new[2] and h.lib.fh_live(new[0]) > 0
    h.lib.glm_ens_destroy(e)


def test_current_buffers_are_the_devices_after_a_failed_sweep():
    """The step control has flipped the buffers when the march behind it cannot be launched."""
    h = Host()
    bx = boxes(2)
    e = ensemble(h, bx)
    out, _ = _lib.plane_array([0] * 9)
    for sweep in range(3):
        h.fail("hipLaunchKernel", 1 + sweep % 2)   # the control, the march, the control
        assert h.lib.glm_ens_step(e, 1) != 0
        n = h.lib.glm_ens_sweeps(e)
        assert n == (0, 1, 1)[sweep]
        for b in range(2):
            assert h.lib.glm_ens_current(e, b, out) == 0
            assert list(out) == list(bx[b].u1 if n % 2 else bx[b].u0)
    assert h.lib.glm_ens_reset(e) == 0 and h.lib.glm_ens_current(e, 0, out) == 0 and list(out) == list(bx[0].u0)
    h.lib.glm_ens_destroy(e)


def test_waiting_calls_return_through_words_of_their_own():
    """Two threads that wait for different results of one context do not get each other's."""
    h = Host()
    start = len(h.log())
    ctx = h.lib.glm_create(16, 16, 16, 8)
    mapped = [x.split() for x in h.log(start) if x.startswith("malloc")][-1]
    base, size = int(mapped[1], 16), int(mapped[2])
    a = step_args(Params(N=16, nz=16, gamma=1.4), 1e-3, 0.0, want_cfl=True)
    out = C.c_double()
    assert h.lib.glm_step(ctx, planes(), planes(base=0x30000000), C.byref(a)) == 0
    assert h.lib.glm_cfl_max(ctx, C.byref(out)) == 0
    assert h.lib.glm_ctot_max(ctx, planes(), C.byref(a), C.byref(out)) == 0
    assert h.lib.glm_step_adjoint(ctx, planes(), planes(base=0x30000000), planes(base=0x50000000), C.byref(a), None) == 0
    assert h.lib.glm_adjoint_force_dot(ctx, 1, C.byref(out)) == 0
    words = [int(x.split("host ")[1], 16) for x in h.log() if "publish_u64" in x]
    assert len(set(words)) == len(words) == 3
    assert all(base + 8 * _lib.NDIAG <= w <= base + size - 8 for w in words)   # behind the diagnostics
    h.lib.glm_destroy(ctx)


def test_the_reverse_step_fits_the_device_it_finds():
    """Fewer CUs: the HLLD adjoint's grid is what is resident, the marches take longer chunks."""
    grids = {}
    for cus in (256, 64):
        h = Host(cus, 1)
        ctx = h.lib.glm_create(64, 64, 64, 8)
        a = step_args(Params(N=64, nz=64, gamma=1.4), 1e-3, 0.0, riemann="hlld", recon="ppm")
        assert h.lib.glm_step_adjoint(ctx, planes(), planes(base=0x30000000), planes(base=0x50000000), C.byref(a), None) == 0
        for k in ("adj_riemann", "adj_front", "adj_back"):
            grids[k, cus] = int(re.search(r"grid (\d+)", [x for x in h.log() if k in x][-1])[1])
        h.lib.glm_destroy(ctx)
    assert grids["adj_riemann", 256] == 256 and grids["adj_riemann", 64] == 64
    assert grids["adj_front", 64] < grids["adj_front", 256] and grids["adj_back", 64] < grids["adj_back", 256]


# (boxes, forcing grid, kmax, one kernel): few planes of many terms each: separate passes; enough planes, either side
# of the line; planes of few terms, more of them in an ensemble; a plane past LDS
@pytest.mark.parametrize("n,g,kmax,one", [(1, 64, 3.0, False), (1, 64, 16.0, False), (1, 32, 5.0, False), (2, 64, 3.0, True),
                                          (3, 32, 8.0, True), (3, 32, 16.0, False), (4, 32, 16.0, True), (1, 128, 3.0, True),
                                          (1, 32, 3.0, True), (1, 16, 8.0, True), (8, 128, 16.0, False)])
def test_the_forcing_passes_are_joined_where_that_is_faster(n, g, kmax, one):
    h = Host()
    if n == 1:
        ctx = h.lib.glm_create(16, 16, 16, 8)
        assert h.lib.glm_ou_setup(ctx, g, 1.0, kmax, 0.5, 100, 0.0, 1.0, 7) == 0
        assert h.lib.glm_ou_advance(ctx) == 0
        h.lib.glm_destroy(ctx)
    else:
        bx = boxes(n)
        for x in bx:
            x.do_turb, x.g, x.ndt, x.kmin, x.kmax, x.amp = 1, g, 100, 1.0, kmax, 1.0
        e = ensemble(h, bx)
        assert h.lib.glm_ens_step(e, 1) == 0
        h.lib.glm_ens_destroy(e)
    passes = [re.search(r"ou_pass_[xyz]+", x)[0] for x in h.log() if "ou_pass_" in x]
    assert passes == (["ou_pass_x", "ou_pass_yz"] if one else ["ou_pass_x", "ou_pass_y", "ou_pass_z"])
