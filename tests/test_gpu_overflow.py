"""A cell that outgrows its bucket, in every way a rebuild can end: in the
list's last block (pair-only systems of up to 128 blocks), in a launch of its
own (larger ones), in the density loop's first block (EAM).  The host has to
learn of it, enlarge the buckets and build again, both in the entry points
and in the middle of fused steps."""
import copy

import numpy as np
import pytest

from imd_amd import imdg as G
from imd_amd import workloads as W

from helpers import (canon_pairs_gpu, canon_pairs_oracle, eam_tables,
                     emod_table, lj, oracle_eam, oracle_lj, rel_rms)
from test_gpu_tuning import TOL, _check_static

pytestmark = pytest.mark.gpu

PLACES = 32       # smallest bucket
LJ_MARGIN = 0.9   # list radius 3.4 sigma: 42 atoms of the crystal in a cell
LJ_CELL = 2.5 + LJ_MARGIN + 1e-6


def _fullest(x, s, ncell):
    """Atoms in the fullest cell of a periodic cube of ncell^3 cells."""
    w = np.mod(x / np.diag(s.box), 1.0)
    c = np.minimum((w * ncell).astype(int), ncell - 1)
    return np.bincount((c[:, 0] * ncell + c[:, 1]) * ncell + c[:, 2]).max()


def _in_box(s, ncell, cell, centre):
    """The block s in an empty box of ncell^3 cells, centred at `centre`
    (in cells)."""
    s.x = s.x - s.x.mean(axis=0) + np.asarray(centre) * cell
    s.box = np.diag([ncell * cell] * 3)
    return s


def _lj_cluster(cells, ncell, seed):
    s = W.fcc_system((cells,) * 3, 1.5496, [1.0], 0.0, seed, displace=0.02)
    return _in_box(s, ncell, LJ_CELL, (ncell // 2 + 0.5,) * 3)


LJ_SYSTEMS = {
    # 4,913 cells (no one-block sort), 2,048 atoms: the list's last block
    "one": [(8, 17)],
    "batch": [(8, 6), (7, 5)],
    # 19,652 atoms, 154 blocks: a launch of its own
    "large": [(17, 17)],
}


@pytest.mark.parametrize("precision", [G.FP64, G.MIXED])
@pytest.mark.parametrize("which", sorted(LJ_SYSTEMS))
def test_pair_only_overflow_static(which, precision):
    systems = [_lj_cluster(c, n, 70 + k)
               for k, (c, n) in enumerate(LJ_SYSTEMS[which])]
    for s, (_, n) in zip(systems, LJ_SYSTEMS[which]):
        assert _fullest(s.x, s, n) > PLACES
    with G.pair_context(lj(), systems, precision=precision,
                        nbl_margin=LJ_MARGIN) as gpu:
        for first in (True, False):      # the buckets fit the second time
            gpu.make_nblist() if not first else None
            gpu.calc_forces()
            pairs = gpu.pairs()
            a = gpu.atoms()
            at = 0
            for r, s in enumerate(systems):
                orc = oracle_lj(s, nbl_margin=LJ_MARGIN, timestep=0.002)
                orc.calc_forces()
                assert canon_pairs_gpu(pairs, r) == \
                    canon_pairs_oracle(orc.pairs())
                f = orc.atoms()["f"]
                d = a["f"][at:at + s.n] - f
                assert np.sqrt(np.mean(d * d) / np.mean(f * f)) <= \
                    TOL[precision][0]
                at += s.n


STEPS = 48


def _drifting(cells, ncell, cell, a, mass, dt, seed, gas=False):
    """A small cube that starts where eight cells meet and moves into the
    middle of one in 40 of the STEPS steps; gas: with one atom, out of reach of the
    others, in each cell the cube stays away from."""
    s = W.fcc_system((cells,) * 3, a, [mass], 0.0, seed, displace=0.02)
    mid = ncell // 2
    s = _in_box(s, ncell, cell, (mid,) * 3)
    if gas:
        g = np.stack(np.meshgrid(*[np.arange(ncell)] * 3, indexing="ij"),
                     -1).reshape(-1, 3)
        g = g[np.abs(g + 0.5 - mid).max(axis=1) > 2.0]
        s.x = np.concatenate([s.x, (g + 0.25) * cell])
        n = s.x.shape[0]
        s.type, s.mass = np.zeros(n, np.int32), np.full(n, mass)
        s.id = np.arange(n, dtype=np.int64)
    s.p = np.full(s.x.shape, 0.5 * cell / (40 * dt) * mass)
    return s


def _same_run(make, systems, dense, ncell, lanes, precision):
    """The run whose bucket overflows on the way has the trajectory of the
    same systems beside a dense one, which sets larger buckets."""
    got = []
    for extra in ([], [dense]):
        with make(systems + extra, precision) as gpu:
            gpu.set_tuning(lanes, 512, lanes, 512)
            gpu.run(STEPS)
            th = gpu.thermo_history(0, STEPS)
            got.append((gpu.atoms(), th[:, :len(systems), 0],
                        th[:, :len(systems), 6]))
    n = sum(s.n for s in systems)
    s = systems[0]
    assert _fullest(s.x, s, ncell) <= PLACES
    assert _fullest(got[1][0]["x"][:s.n], s, ncell) > PLACES
    for k in ("x", "p", "f", "epot", "rho"):
        assert np.array_equal(got[0][0][k][:n], got[1][0][k][:n]), k
    assert np.array_equal(got[0][1], got[1][1])
    assert np.array_equal(got[0][2], got[1][2])
    assert got[0][2][1:, 0].sum() > 0     # it rebuilt after the first step


@pytest.mark.parametrize("precision", [G.FP64, G.MIXED])
@pytest.mark.parametrize("which", ["one", "batch", "large"])
def test_pair_only_overflow_in_run(which, precision):
    ncell = {"one": 17, "batch": 6, "large": 27}[which]
    systems = [_drifting(3, ncell, LJ_CELL, 1.5496, 1.0, 0.002, 80 + k,
                         gas=which == "large")
               for k in range(2 if which == "batch" else 1)]
    dense = W.fcc_system((7, 7, 7), 1.5496, [1.0], 0.0, 90, displace=0.02)

    def make(sys_, prec):
        return G.pair_context(lj(), copy.deepcopy(sys_), precision=prec,
                              nbl_margin=LJ_MARGIN)

    _same_run(make, systems, dense, ncell, 2, precision)


@pytest.mark.parametrize("variant", ["fp64", "mixed", "spline", "eeam"])
def test_list_overflow_while_the_density_loop_runs(variant):
    """With EAM the first block of the density loop freezes the state when
    the list does not fit, while the other blocks start: the loops of several
    species, which take their tables' layout from LDS, run through it and the
    step is run again with the bits of a list that fits."""
    eam = eam_tables(nspecies=2, rc=5.5)
    s = W.alloy_slab((22, 21, 9), temp_k=900.0, seed=17)
    kw = dict(precision=G.MIXED if variant in ("mixed", "eeam") else G.FP64)
    if variant == "spline":
        kw["interpolation"] = G.INTERP_SPLINE
    if variant == "eeam":
        kw["emod"] = emod_table(2)
    got = []
    for size in (0.3, 2.5):   # the vacuum halves the estimate from the mean
        with G.eam_context(eam, [s], nbl_size=size, **kw) as gpu:
            gpu.set_tuning(2, 512, 2, 512)
            first = gpu.info()["kmax"]
            gpu.run(12)
            got.append((gpu.atoms(), gpu.thermo_history(0, 12)[..., :6]))
            assert (gpu.info()["kmax"] > first) == (size == 0.3)
    for k, v in got[0][0].items():
        assert np.array_equal(v, got[1][0][k]), k
    assert np.array_equal(got[0][1], got[1][1])


EAM_MARGIN = 4.0
EAM_CELL = 5.0 + EAM_MARGIN + 1e-6


@pytest.mark.parametrize("precision", [G.FP64, G.MIXED])
def test_overflow_after_deallocate(precision):
    """The list is given back and the next rebuild meets a cell that has
    outgrown its bucket: nothing may read the new, empty list memory.  Then
    calc_forces has the oracle's forces, and a fused run the bits of a context
    that starts there with buckets large enough."""
    eam = eam_tables()
    ncell, kw = 6, dict(precision=precision, nbl_margin=EAM_MARGIN)
    dense = W.eam_crystal(n_cells=8, temp_k=0.0, seed=91)
    for what in ("calc_forces", "run"):
        systems = [_drifting(3, ncell, EAM_CELL, 3.615, W.MASS_CU, W.FS,
                             84 + r) for r in range(2)]
        for s in systems:
            s.p *= 40.0          # to the middle of the cell in one step
            assert _fullest(s.x, s, ncell) <= PLACES
        with G.eam_context(eam, systems, **kw) as gpu:
            gpu.set_tuning(2, 512, 2, 512)
            gpu.calc_forces()
            gpu.move_atoms()
            gpu.deallocate_nblist()
            at = gpu.atoms()
            n = systems[0].n
            for r, s in enumerate(systems):
                s.x, s.p = (at[k][r * n:(r + 1) * n].copy() for k in "xp")
                assert _fullest(s.x, s, ncell) > PLACES
            if what == "calc_forces":
                gpu.calc_forces()
                got = gpu.atoms()
                for r, s in enumerate(systems):
                    orc = oracle_eam(s, eam, nbl_margin=EAM_MARGIN,
                                     timestep=W.FS)
                    orc.calc_forces()
                    assert canon_pairs_gpu(gpu.pairs(), r) == \
                        canon_pairs_oracle(orc.pairs())
                    assert rel_rms(got["f"][r * n:(r + 1) * n],
                                   orc.atoms()["f"]) <= TOL[precision][0]
                continue
            gpu.run(2)
            got = gpu.atoms()
        with G.eam_context(eam, systems + [dense], **kw) as gpu:
            gpu.set_tuning(2, 512, 2, 512)
            gpu.run(2)
            want = gpu.atoms()
        for k, v in got.items():
            assert np.array_equal(v, want[k][:2 * n]), k


SORTS = {
    # EAM, scan of the cells in the binning's last block and in its own launch
    "crystal": lambda: [W.eam_crystal(n_cells=14, temp_k=1200.0, seed=61)],
    "large": lambda: [W.eam_crystal(n_cells=42, temp_k=1200.0, seed=62)],
    "batch": lambda: [W.eam_crystal(n_cells=n, temp_k=t, seed=63 + n)
                      for n, t in ((5, 1.0), (8, 1500.0), (6, 900.0))],
    # 2,048 atoms in 13^3 cells: most of them empty, some beyond 32 atoms
    "cluster": lambda: [_in_box(W.eam_crystal(n_cells=8, temp_k=900.0,
                                              seed=64, displace=0.02),
                                13, EAM_CELL, (6.5, 6.5, 6.5))],
}


@pytest.mark.parametrize("graph", ["0", "1"])
@pytest.mark.parametrize("precision", [G.FP64, G.MIXED])
@pytest.mark.parametrize("which", sorted(SORTS))
def test_sort_without_buckets(which, precision, graph, monkeypatch):
    """Cells too many for buckets: the sort by place gives the bits of the
    sort through buckets, over fused steps with rebuilds and from captured
    ones."""
    margin = EAM_MARGIN if which == "cluster" else 0.4
    monkeypatch.setenv("IMDG_GRAPH", graph)
    got = []
    for limit in (None, "0"):
        if limit:
            monkeypatch.setenv("IMDG_BUCKET_LIMIT", limit)
        with G.eam_context(eam_tables(), SORTS[which](), precision=precision,
                           nbl_margin=margin) as gpu:
            gpu.run(40)
            th = gpu.thermo_history(0, 40)
            gpu.make_nblist()
            got.append((gpu.atoms(), th, gpu.pairs(), gpu.cells()))
    for k, v in got[0][0].items():
        assert np.array_equal(v, got[1][0][k]), k
    for a, b in zip(got[0][1:], got[1][1:]):
        assert np.array_equal(a, b)
    assert got[0][1][1:, :, 6].sum() > 0 or which == "cluster"


@pytest.mark.parametrize("precision", [G.FP64, G.MIXED])
@pytest.mark.parametrize("which", sorted(LJ_SYSTEMS))
def test_pair_only_sort_without_buckets(which, precision, monkeypatch):
    """The same for the pair-only systems whose buckets overflow, against
    runs whose buckets have grown."""
    systems = [_lj_cluster(c, n, 70 + k)
               for k, (c, n) in enumerate(LJ_SYSTEMS[which])]
    for s in systems:
        s.p = W.maxwell_momenta(np.random.default_rng(7), s.mass, 0.4)
    got = []
    for limit in (None, "0"):
        if limit:
            monkeypatch.setenv("IMDG_BUCKET_LIMIT", limit)
        with G.pair_context(lj(), systems, precision=precision,
                            nbl_margin=LJ_MARGIN) as gpu:
            gpu.run(60)
            got.append((gpu.atoms(), gpu.thermo_history(0, 60)))
    for k, v in got[0][0].items():
        assert np.array_equal(v, got[1][0][k]), k
    assert np.array_equal(got[0][1], got[1][1])
