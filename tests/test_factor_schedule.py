"""Host-side check of the multi-workgroup factor's schedules (CPU, no GPU).

The band LDL^T of gsstructuralanalysis_amd/csrc/ksh_factor_tiled.hip runs in panels of 64 columns.  Its
launches are made of these units:

  D  the diagonal block at c0: updated with the panel before (from its stored rows, or from rows that the
     unit solves itself), factored, stored; writes the panel's workspace slot;
  R  a tile of 16 rows below it: solved against the factored block and the slot, stored;
  T  a 32 x 32 block of the trailing window: updated with the panel's stored rows and pivots;
  F  a 64 x 64 tile of the window: the same with rows that the unit solves itself.

The plain schedule launches the R of a panel, then its T with the next D; the lookahead schedule the T of
the next panel's columns with the next D, then the next panel's R with the other T; the fused schedule one
launch a step: the next D, the F, and the R of the panel before.

The index arithmetic (parts of the update, tile and workgroup numbers, workspace slots) is the kernels' own:
ksh_factor_order.hpp, compiled here.  The entries that a unit reads and writes are restated below, with a
hash in the place of every value: a unit's output entries are hashes of all it reads.  On small shapes the
test checks that

  * the parts cover every block once, and a launch's workgroups every tile and block once;
  * no unit of a launch touches an entry or a workspace slot that another one writes;
  * every schedule ends with the hashes of the unscheduled algorithm (factor, solve all rows, update the
    whole window, next panel): each unit has read the right version of everything.

So the schedules order the same computations differently without a race, which is why the GPU tests
(test_gpu_lookahead.py, test_gpu_panel.py) find bit-identical factors."""
import subprocess

import numpy as np
import pytest

CSRC = __file__.rsplit("/tests/", 1)[0] + "/gsstructuralanalysis_amd/csrc"
NB, XCDS, ROW_WAVES, STEP_WAVES = 64, 8, 4, 8
PARTS = ("all", "next", "rest")

PROGRAM = r"""
#include <cstdio>
#include <initializer_list>
#include "ksh_factor_order.hpp"
using namespace ksh;
int main()
{
    for (int nbk = 0; nbk <= 45; ++nbk)
        for (int part : {kAll, kNext, kRest})
            for (int q = 0; q < trail_blocks(nbk, part); ++q) {
                int bi, bj;
                trail_decode(q, nbk, part, bi, bj);
                std::printf("part %d %d %d %d\n", nbk, part, bi, bj);
            }
    for (int p = 0; p < 1000; ++p) {
        int bi, bj;
        tri_decode(p, bi, bj);
        std::printf("tri %d %d\n", bi, bj);
    }
    for (int k = 0; k < 100; ++k) std::printf("slot %d\n", panel_slot(64 * k));
    std::printf("fused %d\n", kFusedBands);
    for (int n = 1; n <= 1024; ++n) std::printf("bucket %d %d\n", n, count_bucket(n));
    for (int active : {1, 3, 7, 8, 9, 16, 37, 256})
        for (int wg : {1, 2, 5})
            for (int h = 0; h < (int)band_grid(active, wg); ++h) {
                int band, local;
                workgroup_decode(h, active, wg, band, local);
                std::printf("wg %d %d %d %d %d\n", active, wg, h, band, local);
            }
    return 0;
}
"""


class Order:
    """The kernels' index arithmetic, as tables."""

    def __init__(self, text):
        self.parts, self.tri, self.slots, self.wg, self.buckets = {}, [], [], {}, {}
        for line in text.splitlines():
            kind, *v = line.split()
            v = [int(x) for x in v]
            if kind == "part":
                self.parts.setdefault((v[0], PARTS[v[1]]), []).append((v[2], v[3]))
            elif kind == "tri":
                self.tri.append((v[0], v[1]))
            elif kind == "slot":
                self.slots.append(v[0])
            elif kind == "fused":
                self.fused_bands = v[0]
            elif kind == "bucket":
                self.buckets.setdefault(v[1], []).append(v[0])
            else:
                self.wg.setdefault((v[0], v[1]), []).append(tuple(v[2:]))

    def blocks(self, nbk, part):
        return self.parts.get((nbk, part), [])


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    d = tmp_path_factory.mktemp("factor_order")
    src, exe = d / "order.cpp", d / "order"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-I", CSRC, "-o", str(exe), str(src)])
    return Order(subprocess.check_output([str(exe)], text=True))


# ---- values as hashes ---------------------------------------------------------------------------
M1, M2 = np.uint64(0x9E3779B97F4A7C15), np.uint64(0xBF58476D1CE4E5B9)


def mix(a, b):
    a, b = np.asarray(a, dtype=np.uint64), np.asarray(b, dtype=np.uint64)
    with np.errstate(over="ignore"):
        h = (a ^ (b * M1 + M2 + (a << np.uint64(6)) + (a >> np.uint64(3)))) * M2
        return h ^ (h >> np.uint64(29))


def fold(a):
    """One hash per row of a 2-d array (each entry hashed with its place, then their sum)."""
    with np.errstate(over="ignore"):
        return mix(mix(a, np.arange(a.shape[1])).sum(axis=1, dtype=np.uint64), 7)


class Band:
    """One band: V[i, j] the hash of entry (i, j); behind the entries, one cell per workspace slot."""

    def __init__(self, n, bw, nslots, seed):
        self.n, self.bw, self.nslots = n, bw, nslots
        i, j = np.indices((n, n))
        self.mask = (i >= j) & (i - j <= bw)
        rng = np.random.default_rng(seed)
        self.cells = np.zeros(n * n + nslots, dtype=np.uint64)
        self.cells[:n * n] = np.where(self.mask, rng.integers(1, 2 ** 63, (n, n), dtype=np.uint64), 0).ravel()

    def nr(self, c0):  # end of the panel's rows
        return min(self.n, c0 + NB + self.bw)


class Unit:
    """What a unit reads and writes of its band, by cell number."""

    def __init__(self, band, cells):
        self.B, self.cells = band, cells  # cells: the band's contents before the launch
        self.reads, self.writes, self.out = [], [], []

    def get(self, rows, cols):
        """Entries rows x cols inside the band (0 outside), noted as read."""
        n = self.B.n
        i, j = np.meshgrid(np.asarray(rows, int), np.asarray(cols, int), indexing="ij")
        ok = (i < n) & (j < n) & (i >= j) & (i - j <= self.B.bw)
        at = (i * n + j)[ok]
        self.reads.append(at)
        v = np.zeros(i.shape, dtype=np.uint64)
        v[ok] = self.cells[at]
        return v

    def put(self, i, j, v):
        ok = (i >= j) & (i - j <= self.B.bw)
        self.writes.append((i * self.B.n + j)[ok])
        self.out.append(v[ok])

    def slot(self, s):
        at = np.array([self.B.n ** 2 + s])
        self.reads.append(at)
        return self.cells[at][0]

    def put_slot(self, s, v):
        self.writes.append(np.array([self.B.n ** 2 + s]))
        self.out.append(np.array([v], dtype=np.uint64))

    # -- the arithmetic of the units
    def solve(self, c0, rows, slot):
        """L of the panel at c0 in these rows: from the unsolved rows, the factored block, the slot."""
        cols = np.arange(c0, c0 + NB)
        below = np.tril(np.ones((NB, NB), bool), -1)
        block = np.where(below, self.get(cols, cols), 0)
        h = mix(mix(fold(self.get(rows, cols)), fold(block.reshape(1, -1))[0]), self.slot(slot))
        L = mix(h[:, None], cols[None, :].astype(np.uint64))
        i, j = np.asarray(rows)[:, None], cols[None, :]
        return np.where((i < self.B.n) & (i - j <= self.B.bw), L, 0)

    def update(self, c0, rows, cols, Li, Lj):
        """Entries rows x cols of the window after the panel at c0, given L in the rows and columns."""
        at = np.arange(c0, c0 + NB) * (self.B.n + 1)
        self.reads.append(at)
        d = fold(self.cells[at].reshape(1, -1))[0]
        v = self.get(rows, cols)
        new = mix(mix(mix(v, fold(Li)[:, None]), fold(Lj)[None, :]), mix(d, c0))
        i, j = np.asarray(rows)[:, None], np.asarray(cols)[None, :]
        nr = self.B.nr(c0)  # outside the panel's rows L is zero and nothing changes
        return np.where((i < nr) & (j < nr), new, v)

    def factor(self, c0, v, slot):
        cols = np.arange(c0, min(c0 + NB, self.B.n))
        i, j = np.meshgrid(cols, cols, indexing="ij")
        low = (i >= j) & (i - j <= self.B.bw)
        h = fold(np.where(low, v, 0).reshape(1, -1))[0]
        self.put(i, j, mix(mix(h, i.astype(np.uint64)), j.astype(np.uint64)))
        if slot is not None:
            self.put_slot(slot, mix(h, 1))


def make_unit(spec, bands, snap, order):
    kind, b, c0 = spec[0], spec[1], spec[2]
    B = bands[b]
    u = Unit(B, snap[b])
    slot = lambda c: order.slots[c // NB] % B.nslots
    rows_of = lambda lo, hi: np.arange(lo, min(hi, B.n))
    if kind == "D":
        cols = rows_of(c0, c0 + NB)
        if spec[3] == "first":
            v = u.get(cols, cols)
        else:
            cp = c0 - NB
            L = u.solve(cp, cols, slot(cp)) if spec[3] == "solve" else u.get(cols, np.arange(cp, c0))
            v = u.update(cp, cols, cols, L, L)
        u.factor(c0, v, slot(c0))
    elif kind == "R":
        rows = np.arange(c0 + NB + 16 * spec[3], min(c0 + NB + 16 * spec[3] + 16, B.nr(c0)))
        L = u.solve(c0, rows, slot(c0))
        i, j = np.meshgrid(rows, np.arange(c0, c0 + NB), indexing="ij")
        u.put(i, j, L)
    else:
        edge = 32 if kind == "T" else NB
        bi, bj = spec[3]
        w0, nr, panel = c0 + NB, B.nr(c0), np.arange(c0, c0 + NB)
        rows = np.arange(w0 + edge * bi, min(w0 + edge * bi + edge, nr))
        cols = np.arange(w0 + edge * bj, min(w0 + edge * bj + edge, nr))
        if kind == "T":
            Li, Lj = u.get(rows, panel), u.get(cols, panel)
        else:
            Li, Lj = u.solve(c0, rows, slot(c0)), u.solve(c0, cols, slot(c0))
        new = u.update(c0, rows, cols, Li, Lj)
        i, j = np.meshgrid(rows, cols, indexing="ij")
        u.put(i, j, new)
    return u


# ---- the launches of the schedules ----------------------------------------------------------------
def active_at(ns, c):
    return sum(n > c for n in ns)  # bands are sorted, largest first


def row_units(bands, c0, waves, active):
    """R units of one launch's waves (one or two tiles each, two from 32 bands on), every tile once."""
    ntile = -(-max(B.bw for B in bands) // 16)
    per = 2 if active >= 32 else 1
    wg = -(-ntile // (waves * per))
    out = []
    for b in range(active):
        B, seen = bands[b], []
        for local in range(wg):
            for wave in range(waves):
                t0 = (local * waves + wave) * per
                if B.n <= c0 + NB or c0 + NB + 16 * t0 >= B.nr(c0):
                    continue
                left = -(-(B.nr(c0) - c0 - NB - 16 * t0) // 16)
                seen += range(t0, t0 + min(per, left))
        assert seen == list(range(-(-(B.nr(c0) - c0 - NB) // 16)))
        out += [("R", b, c0, t) for t in seen]
    return out


def trail_units(bands, c0, part, active, order, waves, nblk=1):
    """T units of one launch's waves: block numbers past the band's own are masked."""
    nbk_max = -(-max(B.bw for B in bands) // 32)
    wg = -(-len(order.blocks(nbk_max, part)) // (waves * nblk))
    out = []
    for b in range(active):
        B = bands[b]
        own = order.blocks(-(-(B.nr(c0) - c0 - NB) // 32), part)
        ps = [(local * nblk + s) * waves + wave for local in range(wg) for wave in range(waves) for s in range(nblk)]
        taken = [p for p in ps if p < len(own)]
        assert sorted(taken) == list(range(len(own)))
        out += [("T", b, c0, own[p]) for p in taken]
    return out


def plain(bands, order):
    ns = [B.n for B in bands]
    out = [[("D", b, 0, "first") for b in range(len(bands))]]
    c0 = 0
    while (np_ := active_at(ns, c0 + NB)) > 0:
        out.append(row_units(bands, c0, ROW_WAVES, np_))
        out.append([("D", b, c0 + NB, "update") for b in range(np_)] + trail_units(bands, c0, "all", np_, order, ROW_WAVES))
        c0 += NB
    return out


def lookahead(bands, order, nblk):
    ns = [B.n for B in bands]
    out = [[("D", b, 0, "first") for b in range(len(bands))]]
    np_ = active_at(ns, NB)
    if np_:
        out.append(row_units(bands, 0, ROW_WAVES, np_))
    c0 = 0
    while np_ > 0:
        out.append([("D", b, c0 + NB, "update") for b in range(np_)] + trail_units(bands, c0, "next", np_, order, ROW_WAVES))
        nxt = active_at(ns, c0 + 2 * NB)
        out.append((row_units(bands, c0 + NB, STEP_WAVES, nxt) if nxt else []) +
                   trail_units(bands, c0, "rest", np_, order, STEP_WAVES, nblk))
        np_ = nxt
        c0 += NB
    return out


def fused(bands, order):
    ns, maxbw = [B.n for B in bands], max(B.bw for B in bands)
    nt = -(-maxbw // NB)
    ntile = max(0, nt * (nt + 1) // 2 - 1)
    nrow = -(-(-(-maxbw // 16)) // ROW_WAVES)
    out = [[("D", b, 0, "first") for b in range(len(bands))]]
    c0 = 0
    while (np_ := active_at(ns, c0)) > 0:
        launch = []
        for b in range(np_):
            B = bands[b]
            if B.n > c0 + NB:
                launch.append(("D", b, c0 + NB, "solve"))
                tiles = [order.tri[g] for g in range(1, ntile + 1)]  # workgroup 0 has tile 0
                launch += [("F", b, c0, t) for t in tiles if c0 + NB + NB * t[0] < B.nr(c0)]
            if c0 > 0:
                cp = c0 - NB
                rows = [t for t in range(nrow * ROW_WAVES) if B.n > cp + NB and cp + NB + 16 * t < B.nr(cp)]
                launch += [("R", b, cp, t) for t in rows]
        out.append(launch)
        c0 += NB
    return out


def replay(launches, bands, order):
    for launch in launches:
        snap = [B.cells.copy() for B in bands]
        units = [make_unit(s, bands, snap, order) for s in launch]
        writer = [np.full(B.cells.size, -1) for B in bands]
        for k, (s, u) in enumerate(zip(launch, units)):
            at = np.concatenate(u.writes) if u.writes else np.array([], int)
            assert (writer[s[1]][at] == -1).all(), ("two units write an entry", s)
            writer[s[1]][at] = k
        for k, (s, u) in enumerate(zip(launch, units)):
            at = np.concatenate(u.reads)
            w = writer[s[1]][at]
            assert ((w == -1) | (w == k)).all(), ("a unit reads what another one of its launch writes", s)
        for s, u in zip(launch, units):
            for at, v in zip(u.writes, u.out):
                bands[s[1]].cells[at] = v


def unscheduled(B):
    """Factor, solve all rows, update the whole window, panel by panel."""
    for c0 in range(0, B.n, NB):
        cols = np.arange(c0, min(c0 + NB, B.n))
        u = Unit(B, B.cells)
        u.factor(c0, u.get(cols, cols), 0)
        apply_unit(u)
        if B.n <= c0 + NB:
            return
        rows, panel = np.arange(c0 + NB, B.nr(c0)), np.arange(c0, c0 + NB)
        if rows.size == 0:
            continue
        u = Unit(B, B.cells)
        L = u.solve(c0, rows, 0)
        i, j = np.meshgrid(rows, panel, indexing="ij")
        u.put(i, j, L)
        apply_unit(u)
        u = Unit(B, B.cells)
        L = u.get(rows, panel)
        i, j = np.meshgrid(rows, rows, indexing="ij")
        u.put(i, j, u.update(c0, rows, rows, L, L))
        apply_unit(u)


def apply_unit(u):
    for at, v in zip(u.writes, u.out):
        u.B.cells[at] = v


def bands_of(shape, nslots):
    return [Band(n, bw, nslots, seed) for seed, (n, bw) in enumerate(zip(*shape))]


SHAPES = [([300], [70]), ([200, 150, 64, 10], [100, 100, 40, 5]), ([129, 128, 65, 64, 63, 1], [130, 60, 64, 33, 31, 0]),
          ([400], [200]), ([97, 96], [96, 95]), ([260, 250], [31, 33]), ([420, 300], [250, 180]), ([500], [64]), ([330, 1], [17, 0])]


@pytest.mark.parametrize("shape", SHAPES)
def test_schedules_read_what_the_algorithm_reads(shape, order):
    ref = bands_of(shape, 1)
    for B in ref:
        unscheduled(B)
    for name, launches in (("plain", plain), ("lookahead", lambda b, o: lookahead(b, o, 1)),
                           ("lookahead, two blocks", lambda b, o: lookahead(b, o, 2)), ("fused", fused)):
        bands = bands_of(shape, 3)
        replay(launches(bands, order), bands, order)
        for B, R in zip(bands, ref):
            assert np.array_equal(B.cells[:B.n ** 2], R.cells[:R.n ** 2]), name


@pytest.mark.parametrize("nslots", [1, 2])
def test_fewer_workspace_slots_would_not_do(nslots, order):
    """The check sees a fused launch that would overwrite a slot it still reads."""
    bands = bands_of(([300], [70]), nslots)
    with pytest.raises(AssertionError):
        replay(fused(bands, order), bands, order)


def test_rows_stored_in_their_own_launch_would_race(order):
    """The check sees the fused schedule with a panel's rows stored while others still solve from them."""
    bands = bands_of(([300], [70]), 3)
    launches = fused(bands, order)
    launches[1] = launches[1] + [s for s in launches[2] if s[0] == "R"]
    with pytest.raises(AssertionError, match="writes"):
        replay(launches[:2], bands, order)


@pytest.mark.parametrize("nbk", range(0, 46))
def test_parts_cover_every_block_once(nbk, order):
    allb = {(i, j) for i in range(nbk) for j in range(i + 1)} - {(0, 0), (1, 0), (1, 1)}  # the next diagonal block's
    every, nxt, rest = (order.blocks(nbk, p) for p in PARTS)
    assert len(every) == len(allb) and set(every) == allb
    assert sorted(nxt + rest) == sorted(allb)
    assert all(bj <= 1 for _, bj in nxt) and all(bj >= 2 for _, bj in rest)


def test_tuning_buckets_end_where_the_schedule_changes(order):
    """Counts that share a tuned choice have the same launches under every schedule, and are within a factor
    of two of each other."""
    for counts in order.buckets.values():
        assert max(counts) <= order.fused_bands or min(counts) > order.fused_bands
        assert max(counts) <= 2 * min(counts)
    assert sorted(n for counts in order.buckets.values() for n in counts) == list(range(1, 1025))


def test_tile_numbers(order):
    assert order.tri == [(i, j) for i in range(60) for j in range(i + 1)][:1000]


# ---- XCD-aware workgroup -> (band, index) mapping of the trailing launches ---------------------
@pytest.mark.parametrize("active", [1, 3, 7, 8, 9, 16, 37, 256])
@pytest.mark.parametrize("wg", [1, 2, 5])
@pytest.mark.parametrize("ndiag", [0, 5, 8, 13])
def test_xcd_mapping_covers_every_band_workgroup_once(active, wg, ndiag, order):
    """Every (band, index) of a launch is taken by exactly one workgroup, the rest exit; with 8 or
    more bands a band's workgroups all sit on the XCD of its diagonal block's (id = band mod 8),
    also behind those of a launch that holds both (offset padded to a multiple of 8)."""
    pad = -(-ndiag // XCDS) * XCDS if active >= XCDS else ndiag
    seen = []
    for h, b, l in order.wg[(active, wg)]:
        if b < active:
            seen.append((b, l))
            if active >= XCDS:
                assert (pad + h) % XCDS == b % XCDS
    assert sorted(seen) == [(b, l) for b in range(active) for l in range(wg)]
