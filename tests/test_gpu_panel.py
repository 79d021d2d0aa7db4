"""Panel kernels of the multi-workgroup factor (64-column diagonal blocks factored 16 columns at a time,
row tiles of 16) at the sizes where they can go wrong: orders around the multiples of 16 and 64, band
widths below one tile, below one panel and around the multiples of 16 and 32; and batches of uneven bands on
either side of the counts at which a launch changes (fused up to 8 bands, two row tiles a wave from 32).

Checked by the backward error of a solve with the factor, ||b - K x|| <= c eps G ||x||: G, the largest
entry of |L| |D| |L|^T of the oracle's factor, is what an unpivoted LDL^T's error is relative to (it is
max|K| for a definite matrix, and holds the growth of an indefinite one), and c = 8 bw + 64 covers one
rounding per product along a band row, for the factor and the two sweeps, and the blocked sums' own.
And by the pivots' signs against the oracle's; the three schedules (plain, lookahead, one fused launch a
step; two blocks a wave instead of the fused launches above 8 bands) give the same bits at every shape, in
the pivots and, by the solutions, in the stored rows, which in the fused schedule no pivot depends on."""
import numpy as np
import pytest

from gsstructuralanalysis_amd import _lib as L
from gsstructuralanalysis_amd import geometry as g
from oracle import ok
from oracle.ok import Oracle

pytestmark = pytest.mark.gpu

# (p, nx, ny): orders 6..3510 free dofs, half-widths 8..1307
SHAPES = [(2, 1, 2), (2, 1, 5), (2, 1, 20), (2, 2, 9), (2, 3, 2), (2, 4, 4), (3, 1, 6), (3, 2, 3), (3, 3, 12), (2, 8, 3), (3, 5, 5), (2, 9, 7),
          (3, 9, 4), (2, 29, 3), (3, 48, 3), (3, 51, 2), (3, 140, 2)]


def _growth(ref, n, bw):
    """max_i sum_k L_ik^2 |d_k|, the largest entry of |L| |D| |L|^T."""
    f = ref.ab.reshape(n, bw + 1)
    out = np.abs(f[:, 0]).copy()
    for k in range(n):
        m = min(bw, n - 1 - k)
        out[k + 1:k + 1 + m] += f[k, 1:1 + m] ** 2 * abs(f[k, 0])
    return out.max()


@pytest.mark.parametrize("p,nx,ny", SHAPES)
@pytest.mark.parametrize("prec", [L.FP64, L.FP32_IR])
def test_factor_at_tile_edges(p, nx, ny, prec, ksh, monkeypatch):
    from gsstructuralanalysis_amd.problem import BandMatrix, ShellProblem
    pt = g.roof_problem(p=p, n=nx, ny=ny, rho=1e3)
    o = Oracle(pt)
    print(f"[case] panel edges roof p={p} {nx}x{ny} nfree={o.nfree} bw={o.bw} prec={prec}", flush=True)
    sp = ShellProblem(pt)
    rng = np.random.default_rng(17)
    Kb = o.tangent_band(rng.standard_normal(o.nfree) * 1e-4)
    # an indefinite matrix too: the band minus a multiple of the mass that turns some pivots negative
    Mb = o.mass_band()
    shift = 1e-3 * np.abs(Kb).max() / np.abs(Mb).max()
    eps = np.finfo(np.float64 if prec == L.FP64 else np.float32).eps
    for ab in (Kb, Kb - shift * Mb):
        A = BandMatrix(sp, precision=prec)
        ds, xs = [], []
        b = rng.standard_normal(o.nfree)
        for schedule in ("2", "1", "0"):
            monkeypatch.setenv("KSH_LOOKAHEAD", schedule)
            A.upload(ab)
            A.set_inertia_guard(0.0)
            A.factor()
            ds.append(A.vector_d())
            xs.append(A.solve(b))
        assert np.array_equal(ds[0], ds[2]) and np.array_equal(ds[1], ds[2])
        assert np.array_equal(xs[0], xs[2]) and np.array_equal(xs[1], xs[2])
        ref = ok.BandLDLT(ab, o.nfree, o.bw)
        x = xs[2]
        r = b - ok.band_symv(ab, o.nfree, o.bw, x)
        assert np.linalg.norm(r) <= (8 * o.bw + 64) * eps * _growth(ref, o.nfree, o.bw) * np.linalg.norm(x)
        if prec == L.FP64:
            assert A.inertia()[0] == ref.negatives()[0]


@pytest.mark.parametrize("count", [8, 9, 31, 33])
@pytest.mark.parametrize("prec", [L.FP64, L.FP32_IR])
def test_schedules_of_uneven_batches(count, prec, ksh, monkeypatch):
    from gsstructuralanalysis_amd.problem import ShellProblem, run_alm_batch
    sizes = [(2, 1, 5), (2, 4, 4), (3, 3, 12), (2, 8, 3), (3, 5, 5), (2, 9, 7), (3, 9, 4), (3, 1, 6), (2, 2, 9), (3, 12, 6)]
    for p in (2, 3):  # a batch has one degree
        mine = [s for s in sizes if s[0] == p]
        sps = [ShellProblem(g.roof_problem(p=p, n=mine[i % len(mine)][1], ny=mine[i % len(mine)][2] + i // len(mine))) for i in range(count)]
        print(f"[case] schedules of {count} bands, orders {min(sp.nfree for sp in sps)}..{max(sp.nfree for sp in sps)}, "
              f"half-widths {min(sp.bw for sp in sps)}..{max(sp.bw for sp in sps)}, prec={prec}", flush=True)
        kw = dict(method=0, max_iter=20, tol=1e-6, tol_f=1e-8, tol_u=1e-6, scaling=0.0, bifurcation_method=0, keep_U=True, precision=prec)
        if prec != L.FP64:
            kw.update(max_refine=8, refine_tol=1e-9)
        runs = []
        for schedule in ("0", "1", "2"):
            monkeypatch.setenv("KSH_LOOKAHEAD", schedule)
            runs.append(run_alm_batch(sps, 2, 2e-3, **kw)[0])
        for run in runs[1:]:
            for a, b in zip(runs[0], run):
                assert a["steps_done"] == 2
                for key in ("lambda", "U", "negatives", "iterations"):
                    assert np.array_equal(a[key], b[key]), key
