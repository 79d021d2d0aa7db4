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


@pytest.mark.parametrize("p,nx,ny", [(2, 3, 2), (2, 8, 5), (3, 3, 4), (3, 6, 6), (3, 17, 5)])
def test_fp32_matrix_refinement_at_block_edges(p, nx, ny, ksh):
    """K stored in FP32: the refinement against it reaches 1e-9 without a stall, and the path, whose residuals
    are FP64, agrees with the FP64 form to 1e-5 (an inexact Jacobian; the bar of that form's parity)."""
    from gsstructuralanalysis_amd.problem import ShellProblem
    sp = ShellProblem(g.roof_problem(p=p, n=nx, ny=ny))
    print(f"[case] refinement against FP32 K p={p} {nx}x{ny} nfree={sp.nfree} bw={sp.bw}", flush=True)
    ref = sp.run_alm(4, 2e-3, precision=L.FP64, **KW)
    lib = L.load()
    lib.ksh_profile_reset()
    lib.ksh_profile_enable(1)
    try:
        got = sp.run_alm(4, 2e-3, precision=L.FP32, max_refine=8, refine_tol=1e-9, **KW)
    finally:
        lib.ksh_profile_enable(0)
    n, ms = C.c_int64(), C.c_double()
    lib.ksh_profile_query(b"fp64_refactor_stall", C.byref(n), C.byref(ms))
    assert n.value == 0
    assert got["steps_done"] == ref["steps_done"] == 4 and (got["residue_f"] < 1e-8).all()
    assert np.abs(got["U"] - ref["U"]).max() <= 1e-5 * np.abs(ref["U"]).max()


def test_residuals_by_several_launches(ksh):
    """Batches whose partial sums exceed 512 MiB go by groups of matrices, one launch after the other over the
    same scratch: every instance gets the bits that it gets alone."""
    from gsstructuralanalysis_amd.problem import ShellProblem, run_alm_batch
    pt = g.roof_problem(p=3, n=48)
    z = pt.ctrl[:, 2].copy()
    sps = []
    for i in range(480):
        pt.ctrl[:, 2] = z * (1.0 + 1e-4 * i)
        sps.append(ShellProblem(pt))
    n, bw = sps[0].nfree, sps[0].bw
    each = -(-n // 64) * 64 * (1 + (bw + 127) // 64) * 8 * 2  # two right-hand sides a matrix
    first = (512 << 20) // each  # instance that the second launch begins with
    print(f"[case] {len(sps)} bands of {n} rows, half-width {bw}: {first} of them in the first launch", flush=True)
    assert first < len(sps) - 1
    kw = dict(KW, precision=L.FP32_IR, max_refine=8, refine_tol=1e-9)
    many, _ = run_alm_batch(sps, 1, 2e-3, **kw)
    for i in (0, first - 1, first, first + 1, len(sps) - 1):
        one = sps[i].run_alm(1, 2e-3, **kw)
        assert one["steps_done"] == 1
        for key in ("lambda", "U", "iterations"):
            assert np.array_equal(one[key], many[i][key]), (i, key)
