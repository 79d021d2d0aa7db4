"""The residual kernel at the edges of its waves, against the FP64 oracle: a wave takes 7 elements at
degree 2 and 4 at degree 3, so element counts of one, a full wave, one more, and remainders, with
and without a follower pressure.  Tolerance: the assembly parity bar, 1e-11 of max|R|.
"""
import numpy as np
import pytest

from gsstructuralanalysis_amd import geometry as g
from oracle.ok import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pressure", [0.0, -25.0])
@pytest.mark.parametrize("p,nx,ny", [(2, 1, 1), (2, 7, 1), (2, 4, 2), (2, 5, 3), (3, 1, 1), (3, 2, 2), (3, 5, 1), (3, 3, 3)])
def test_residual_wave_edges(p, nx, ny, pressure, ksh):
    from gsstructuralanalysis_amd.problem import ShellProblem
    pt = g.roof_problem(p=p, n=nx, ny=ny)
    pt.pressure = pressure
    print(f"[case] residual p={p} {nx}x{ny} pressure={pressure}", flush=True)
    sp, o = ShellProblem(pt), Oracle(pt)
    u = np.random.default_rng(11).standard_normal(o.nfree) * 3e-2
    for got, want in ((sp.residual(u, 0.7, conv=1), o.residual_alm(u, 0.7)), (sp.residual(u, 1.3, conv=0), o.residual_static(u, 1.3))):
        assert np.abs(got - want).max() <= 1e-11 * np.abs(want).max()
