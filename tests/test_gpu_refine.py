"""Refinement residuals by column blocks (ksh_spmv.hip) at the edges of the 64-row and 64-column blocks:
orders below, at and past multiples of 64, half-widths below one block, and over two and three.

The mixed form (FP32 factor, FP64 residuals) runs an arc-length path whose solves are refined to 1e-9: no
solve may stall (with a wrong residual eight sweeps do not get there), Newton takes the
iterations of the FP64 form, and the path agrees with it to 1e-8, the bar of the forms' parity.
"""
import ctypes as C

import numpy as np
import pytest

from gsstructuralanalysis_amd import _lib as L
from gsstructuralanalysis_amd import geometry as g

pytestmark = pytest.mark.gpu

KW = dict(method=0, max_iter=20, tol=1e-6, tol_f=1e-8, tol_u=1e-6, scaling=0.0, bifurcation_method=0, keep_U=True)


@pytest.mark.parametrize("p,nx,ny", [(2, 3, 2), (2, 6, 2), (2, 8, 5), (3, 3, 4), (3, 6, 6), (3, 12, 4), (3, 17, 5)])
def test_mixed_refinement_at_block_edges(p, nx, ny, ksh):
    from gsstructuralanalysis_amd.problem import ShellProblem
    sp = ShellProblem(g.roof_problem(p=p, n=nx, ny=ny))
    print(f"[case] refinement p={p} {nx}x{ny} nfree={sp.nfree} bw={sp.bw}", flush=True)
    ref = sp.run_alm(4, 2e-3, precision=L.FP64, **KW)
    lib = L.load()
    lib.ksh_profile_reset()
    lib.ksh_profile_enable(1)
    try:
        mix = sp.run_alm(4, 2e-3, precision=L.FP32_IR, max_refine=8, refine_tol=1e-9, **KW)
    finally:
        lib.ksh_profile_enable(0)
    n, ms = C.c_int64(), C.c_double()
    lib.ksh_profile_query(b"fp64_refactor_stall", C.byref(n), C.byref(ms))
    assert n.value == 0
    assert mix["steps_done"] == ref["steps_done"] == 4
    assert np.array_equal(mix["iterations"], ref["iterations"])
    assert np.abs(mix["U"] - ref["U"]).max() <= 1e-8 * np.abs(ref["U"]).max()
