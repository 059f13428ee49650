"""Batches of replicas on both sides of the lines by which the rebuild chain
is chosen: the scan of the cell counts in the binning's last block or in its
own launch, by the number of replicas and of blocks; the lanes per atom of the
list build where all replicas rebuild at once.  The skin test of the entry
points."""
import numpy as np
import pytest

from imd_amd import imdg as G
from imd_amd import workloads as W

from helpers import (canon_pairs_gpu, canon_pairs_oracle, eam_tables, lj,
                     oracle_eam, rel_rms)
from test_gpu_tuning import TOL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrep", [20, 21])
def test_scan_by_number_of_replicas(nrep):
    """Small replicas of different sizes (27 to 80 cells): the pairs and
    forces of three of them are the oracle's, and a run of the batch rebuilds
    them as each does alone."""
    eam = eam_tables()
    systems = [W.fcc_system((5 + r % 3, 5 + r % 2, 5), 3.615, eam.masses,
                            W.kT(300.0 + 60.0 * r), 30 + r, displace=0.03)
               for r in range(nrep)]
    with G.eam_context(eam, systems, precision=G.FP64) as gpu:
        gpu.calc_forces()
        pairs, a = gpu.pairs(), gpu.atoms()
        at = 0
        for r, s in enumerate(systems):
            if r in (0, nrep // 2, nrep - 1):
                orc = oracle_eam(s, eam, nbl_margin=0.4, timestep=W.FS)
                orc.calc_forces()
                assert canon_pairs_gpu(pairs, r) == \
                    canon_pairs_oracle(orc.pairs())
                assert rel_rms(a["f"][at:at + s.n],
                               orc.atoms()["f"]) <= TOL[G.FP64][0]
            at += s.n
    with G.eam_context(eam, systems, precision=G.MIXED) as gpu:
        gpu.set_tuning(2, 512, 2, 512)
        gpu.run(60)
        both, th = gpu.atoms(), gpu.thermo_history(0, 60)
    at = sum(s.n for s in systems[:-1])
    with G.eam_context(eam, systems[-1:], precision=G.MIXED) as one:
        one.set_tuning(2, 512, 2, 512)
        one.run(60)
        alone, t1 = one.atoms(), one.thermo_history(0, 60)
    for k, v in alone.items():
        assert np.array_equal(both[k][at:], v), k
    assert np.array_equal(th[:, -1, 6], t1[:, 0, 6])
    assert t1[1:, 0, 6].sum() > 0


@pytest.mark.parametrize("cells,nrep", [(22, 1), (14, 4), (5, 70),
                                        (5, 1100)])
def test_skin_test_of_many_blocks(cells, nrep):
    """imdg_check_nblist of large replicas and of many: the loop of the three
    entry points rebuilds in the steps in which the fused run does, with the
    same bits, and the call's answer is the record's decision."""
    eam = eam_tables()
    systems = [W.eam_crystal(n_cells=cells, temp_k=200.0 + 1300.0 * r / nrep,
                             seed=70 + r) for r in range(1, nrep + 1)]
    got = []
    for fused in (True, False):
        with G.eam_context(eam, systems, precision=G.FP64) as gpu:
            assert gpu.info()["nslots"] > 256 * 128
            gpu.set_tuning(2, 512, 2, 512)
            answers = []
            if fused:
                gpu.run(40)
            else:
                for _ in range(40):
                    gpu.calc_forces()
                    gpu.move_atoms()
                    answers.append(gpu.check_nblist())
            got.append((gpu.atoms(), gpu.thermo_history(0, 40)))
    skin2 = (0.5 * 0.4) ** 2
    assert answers == (got[1][1][:, :, 5] > skin2).any(axis=1).tolist()
    assert any(answers)
    assert np.array_equal(got[0][1][..., 5:], got[1][1][..., 5:])
    for k in ("x", "p"):
        assert np.array_equal(got[0][0][k], got[1][0][k]), k


# 686 and 763 blocks, at most 8,192 cells: the scan folded and not
@pytest.mark.parametrize("cells,nrep", [(28, 1), (29, 1), (20, 2), (20, 3)])
def test_scan_by_number_of_blocks(cells, nrep, monkeypatch):
    """The sort is the same whichever launch scans the cells: one that takes
    no buckets and one that does give the bits of each other through
    rebuilds, and a static evaluation the oracle's pairs."""
    eam = eam_tables()
    systems = [W.eam_crystal(n_cells=cells, temp_k=1400.0, seed=40 + r)
               for r in range(nrep)]
    got = []
    for limit in (None, "0"):
        if limit:
            monkeypatch.setenv("IMDG_BUCKET_LIMIT", limit)
        with G.eam_context(eam, systems, precision=G.MIXED) as gpu:
            gpu.run(40)
            got.append((gpu.atoms(), gpu.thermo_history(0, 40)))
    for k, v in got[0][0].items():
        assert np.array_equal(v, got[1][0][k]), k
    assert np.array_equal(got[0][1], got[1][1])
    assert got[0][1][1:, 0, 6].sum() > 0
    with G.eam_context(eam, systems, precision=G.FP64) as gpu:
        gpu.make_nblist()
        pairs = gpu.pairs()
    orc = oracle_eam(systems[-1], eam, nbl_margin=0.4, timestep=W.FS)
    orc.calc_forces()
    assert canon_pairs_gpu(pairs, nrep - 1) == canon_pairs_oracle(orc.pairs())


@pytest.mark.parametrize("graph", ["0", "1"])
@pytest.mark.parametrize("case", ["eam-mixed", "lj-fp64"])
def test_first_list_of_a_full_chip(case, graph, monkeypatch):
    """A batch beyond the line: its first list and make_nblist take one lane
    per atom, the rebuilds of its steps four.  The replicas follow the
    trajectories they have alone (four lanes throughout), bit for bit, before
    and after a make_nblist between their steps."""
    monkeypatch.setenv("IMDG_GRAPH", graph)
    eam = eam_tables()
    if case == "eam-mixed":
        systems = [W.eam_crystal(n_cells=20, temp_k=1200.0, seed=5 + r)
                   for r in range(17)]

        def make(s):
            return G.eam_context(eam, s, precision=G.MIXED)
    else:
        systems = [W.fcc_system((9, 9, 9), 1.5496, [1.0], 0.7, 5 + r)
                   for r in range(179)]

        def make(s):
            return G.pair_context(lj(), s, precision=G.FP64, nbl_margin=0.3)

    def run(s):
        with make(s) as gpu:
            gpu.set_tuning(2, 512, 2, 512)
            gpu.run(30)
            gpu.make_nblist()
            gpu.run(30)
            return gpu.atoms(), gpu.thermo_history(0, 60)[:, :, 6]

    both, rebuilt = run(systems)
    for r in (0, len(systems) - 1):
        alone, t1 = run([systems[r]])
        at = sum(s.n for s in systems[:r])
        for k, v in alone.items():
            assert np.array_equal(both[k][at:at + systems[r].n], v), (r, k)
        assert np.array_equal(rebuilt[:, r], t1[:, 0])
        assert t1[1:, 0].sum() > 1
