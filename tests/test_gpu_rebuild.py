"""The rebuild chain: cells with more atoms than their bucket has places (a
dense cluster in an empty box: the buckets are sized from the mean and have
to grow, in calc_forces and in the middle of fused steps), the scan of the
cell counts in the binning's last block or in its own launch, and replicas
of which only some rebuild."""
import numpy as np
import pytest

from imd_amd import imdg as G
from imd_amd import workloads as W

from helpers import (canon_pairs_gpu, canon_pairs_oracle, eam_tables, lj,
                     oracle_eam, oracle_lj)
from test_gpu_tuning import TOL, _check_static

pytestmark = pytest.mark.gpu


def _cluster(temp=0.0):
    """A 6^3-cell block in a box 12 times as wide: 64 times fewer atoms per
    cell on average than in the block."""
    s = W.eam_crystal(n_cells=6, temp_k=temp, seed=8, displace=0.02)
    s.x = s.x + 100.0
    s.box = s.box * 12.0
    return s


@pytest.mark.parametrize("precision", [G.FP64, G.MIXED])
def test_bucket_overflow_static(precision):
    eam, s = eam_tables(), _cluster()
    # list radius 8 A: about 43 atoms in a full cell, 32 places in a bucket
    orc = oracle_eam(s, eam, nbl_margin=3.0, timestep=W.FS)
    orc.calc_forces()
    with G.eam_context(eam, [s], precision=precision, nbl_margin=3.0) as gpu:
        gpu.calc_forces()
        _check_static(gpu, orc, *TOL[precision])
        assert canon_pairs_gpu(gpu.pairs()) == canon_pairs_oracle(orc.pairs())


@pytest.mark.parametrize("precision", [G.FP64, G.MIXED])
@pytest.mark.parametrize("margin,kept", [(3.0, 1372), (0.4, 1372), (0.4, 1)])
def test_one_block_sort(margin, kept, precision):
    """A small system, whose steps begin with one block that finalizes the
    step before and sorts: 51 atoms a cell (more than the lanes that sort
    one), 13, and a single atom; static and over steps with rebuilds, whose
    records end with the last step's."""
    eam = eam_tables()
    s = W.eam_crystal(n_cells=7, temp_k=900.0, seed=31, displace=0.05)
    s.x, s.p, s.type, s.mass = (v[:kept] for v in (s.x, s.p, s.type, s.mass))
    orc = oracle_eam(s, eam, nbl_margin=margin, timestep=W.FS)
    orc.calc_forces()
    with G.eam_context(eam, [s], precision=precision,
                       nbl_margin=margin) as gpu:
        gpu.calc_forces()
        _check_static(gpu, orc, *TOL[precision])
        assert canon_pairs_gpu(gpu.pairs()) == canon_pairs_oracle(orc.pairs())
    runs = []
    for parts in ((40,), (1, 13, 26)):
        with G.eam_context(eam, [s], precision=precision,
                           nbl_margin=margin) as gpu:
            for n in parts:
                gpu.run(n)
            runs.append((gpu.atoms(), gpu.thermo_history(0, 40)))
    assert np.array_equal(runs[0][1], runs[1][1])
    assert np.array_equal(runs[0][1][:, 0, 0], np.arange(40))
    for k, v in runs[0][0].items():
        assert np.array_equal(v, runs[1][0][k]), k
    if margin == 0.4 and kept > 1:
        assert runs[0][1][1:, 0, 6].sum() > 0


def test_bucket_overflow_in_run():
    """The overflow met by fused steps: the missing steps are run again and
    the trajectory is that of a context whose buckets already fit."""
    eam, s = eam_tables(), _cluster(temp=300.0)
    got = []
    for first in (False, True):
        with G.eam_context(eam, [s], precision=G.FP64, nbl_margin=3.0) as gpu:
            if first:
                gpu.make_nblist()
            gpu.run(12)
            got.append((gpu.atoms(), gpu.thermo_history(0, 12)))
    for k, v in got[0][0].items():
        assert np.array_equal(v, got[1][0][k]), k
    assert np.array_equal(got[0][1][..., :6], got[1][1][..., :6])


# 27, 8,000 and 8,820 cells: the scan in the binning's last block up to 8,192
# cells, in its own launch beyond
@pytest.mark.parametrize("box", [(3, 3, 3), (20, 20, 20), (21, 21, 20)])
def test_scan_paths_match_oracle(box):
    eam = eam_tables()
    s = W.eam_crystal(n_cells=5, temp_k=300.0, seed=21, displace=0.05)
    edge = 5.4 + 1e-6
    if box != (3, 3, 3):
        s.x = s.x + np.array(box) * edge * 0.9   # across the faces
        s.box = np.diag(np.array(box) * edge)
    orc = oracle_eam(s, eam, nbl_margin=0.4, timestep=W.FS)
    orc.calc_forces()
    with G.eam_context(eam, [s], precision=G.FP64) as gpu:
        assert gpu.grid() == box
        gpu.calc_forces()
        _check_static(gpu, orc, *TOL[G.FP64])
        assert canon_pairs_gpu(gpu.pairs()) == canon_pairs_oracle(orc.pairs())


def test_some_replicas_rebuild():
    """A hot and two cold replicas: the hot one rebuilds while the others are
    copied; each follows the trajectory it has alone, bit for bit."""
    eam = eam_tables()
    systems = [W.eam_crystal(n_cells=n, temp_k=t, seed=50 + n, displace=0.02)
               for n, t in ((5, 1.0), (6, 1500.0), (7, 1.0))]
    with G.eam_context(eam, systems, precision=G.MIXED) as gpu:
        gpu.set_tuning(4, 512, 4, 512)
        gpu.run(60)
        both, th = gpu.atoms(), gpu.thermo_history(0, 60)
    at = 0
    for r, s in enumerate(systems):
        with G.eam_context(eam, [s], precision=G.MIXED) as one:
            one.set_tuning(4, 512, 4, 512)
            one.run(60)
            alone, t1 = one.atoms(), one.thermo_history(0, 60)
        for k in ("x", "p", "f", "rho"):
            assert np.array_equal(both[k][at:at + s.n], alone[k]), (r, k)
        assert np.array_equal(th[:, r, 6], t1[:, 0, 6])
        at += s.n
    assert th[1:, 1, 6].sum() > 0 and th[1:, 0, 6].sum() == 0


@pytest.mark.parametrize("precision", [G.FP64, G.MIXED])
@pytest.mark.parametrize("nrep,cells", [(1, 7), (1, 17), (3, 7)])
def test_pair_only_record_turns(nrep, cells, precision):
    """Without EAM the records alternate with the step counter: one run, runs
    of odd lengths and the separate entry points give the same trajectory
    through its rebuilds, and a static evaluation at its end the oracle's
    forces."""
    systems = [W.fcc_system((cells, cells + r, cells), 1.5496, [1.0], 0.7,
                            60 + r) for r in range(nrep)]
    end = []
    for parts in ((30,), (1, 2, 7, 20), None):
        with G.pair_context(lj(), systems, precision=precision,
                            nbl_margin=0.15) as gpu:
            gpu.set_tuning(4, 512, 4, 512)   # one order of summation
            if parts:
                for n in parts:
                    gpu.run(n)
            else:
                for _ in range(30):
                    gpu.calc_forces()
                    gpu.move_atoms()
                    gpu.check_nblist()
            th = gpu.thermo_history(0, 30)
            end.append((gpu.atoms(), th[..., 6]))
            rebuilt = np.nonzero(th[1:, 0, 6])[0] + 1
    for a, t in end[1:]:
        assert np.array_equal(t, end[0][1])
        for k in ("x", "p", "f", "epot"):
            assert np.array_equal(a[k], end[0][0][k]), k
    assert rebuilt.size
    a = end[0][0]
    systems[0].x, systems[0].p = (a[k][:systems[0].n] for k in ("x", "p"))
    orc = oracle_lj(systems[0], nbl_margin=0.15, timestep=0.002)
    orc.calc_forces()
    with G.pair_context(lj(), [systems[0]], precision=precision,
                        nbl_margin=0.15) as gpu:
        gpu.calc_forces()
        _check_static(gpu, orc, *TOL[precision], has_eam=False)


def test_list_of_shared_lanes(monkeypatch):
    """Several lanes per atom build the same list as one: cells of more than
    32 atoms (screened again when they are written), tiles that do not fit,
    open faces, in both entry formats; the pair sets are the oracle's and the
    per-atom lists are in the same order (densities bit for bit)."""
    eam = eam_tables()
    dense = W.eam_crystal(n_cells=7, temp_k=0.0, seed=3, displace=0.08)
    slab = W.fcc_system((8, 6, 5), 3.615, eam.masses, 0.0, 4,
                        pbc=(1, 0, 0), vacuum_z=12.0, displace=0.05)
    # a replica beyond the line: the batch takes one lane per atom
    large = W.eam_crystal(n_cells=44, temp_k=0.0, seed=5, displace=0.02)
    for s, margin in ((dense, 3.0), (dense, 0.4), (slab, 0.4)):
        orc = oracle_eam(s, eam, nbl_margin=margin, timestep=W.FS)
        orc.calc_forces()
        want = canon_pairs_oracle(orc.pairs())
        for list16 in ("1", "0"):
            for limit in ("1536", "64"):
                monkeypatch.setenv("IMDG_LIST16", list16)
                monkeypatch.setenv("IMDG_TILE_LIMIT", limit)
                got = []
                for systems in ([s], [s, large]):
                    with G.eam_context(eam, systems, precision=G.MIXED,
                                       nbl_margin=margin) as gpu:
                        gpu.set_tuning(1, 512, 1, 512)
                        gpu.calc_forces()
                        info = gpu.info()
                        got.append(gpu.atoms()["rho"][:s.n])
                        if len(systems) == 1:
                            assert canon_pairs_gpu(gpu.pairs()) == want
                        assert (info["tiles_fallback"] > 0) or limit != "64"
                assert np.array_equal(got[0], got[1])
