"""Kernel times (ksh_profile_*) of launches whose stream is gone by the time they are asked for: a path
engine's streams end with the call.  An event recorded on a destroyed stream counts for one of the stream
that lives at its address next, so the times have to be read before the stream is destroyed.  The test
opens captures on new streams (on addresses of the old ones among them), asks for the times, and closes
the captures: the launches are all counted, and no capture has been touched."""
import ctypes as C

import pytest

from gsstructuralanalysis_amd import _lib as L
from gsstructuralanalysis_amd import geometry as g

pytestmark = pytest.mark.gpu

KW = dict(method=0, max_iter=20, tol=1e-6, tol_f=1e-8, tol_u=1e-6, scaling=0.0, bifurcation_method=0)
THREAD_LOCAL, NON_BLOCKING = 1, 1
NAMES = [b"band_ldlt_batch_fp64", b"residual_elem", b"tangent_elem"]


def _profiled_run(sp, lib):
    lib.ksh_profile_reset()
    lib.ksh_profile_enable(1)
    try:
        sp.run_alm(2, 2e-3, precision=L.FP64, **KW)
    finally:
        lib.ksh_profile_enable(0)


def _counts(lib):
    out = []
    for name in NAMES:
        n, ms = C.c_int64(), C.c_double()
        L.check(lib.ksh_profile_query(name, C.byref(n), C.byref(ms)))
        out.append(n.value)
    return out


def test_times_of_destroyed_streams(ksh):
    from gsstructuralanalysis_amd.problem import ShellProblem
    hip, lib = C.CDLL("libamdhip64.so.7"), L.load()
    sp = ShellProblem(g.roof_problem(p=2, n=4))
    print(f"[case] kernel times of an ended engine, roof p=2 4x4 nfree={sp.nfree}", flush=True)
    _profiled_run(sp, lib)
    want = _counts(lib)
    assert all(n > 0 for n in want)
    _profiled_run(sp, lib)
    streams = []
    try:
        for _ in range(16):
            s = C.c_void_p()
            assert hip.hipStreamCreateWithFlags(C.byref(s), NON_BLOCKING) == 0
            assert hip.hipStreamBeginCapture(s, THREAD_LOCAL) == 0
            streams.append(s)
        assert _counts(lib) == want
    finally:
        ended = []
        for s in streams:
            graph = C.c_void_p()
            ended.append(hip.hipStreamEndCapture(s, C.byref(graph)))
            if graph:
                hip.hipGraphDestroy(graph)
            hip.hipStreamDestroy(s)
    assert ended == [0] * 16
