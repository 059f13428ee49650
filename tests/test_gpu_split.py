"""Chunks of the neighbour loops split into units of some of their passes:
systems of a few chunks (four units a chunk with four lanes), at sizes where
four or two units a chunk are chosen and where the chunks fill the chip,
with the tables staged or read from L2, against the oracle at the bars of the launch shapes; one wavefront's chunk
that is not full; replicas, whose partial sums are per unit, over several
steps and lanes; the pair columns of two species, equal across the diagonal
(three are stored) or not (all four); the FP64 default shapes on both sides
of their line of size; the accuracy of the mixed sums with two lanes."""
import copy

import numpy as np
import pytest

from imd_amd import imdg as G
from imd_amd import workloads as W

from helpers import eam_tables, lj, oracle_eam, oracle_lj
from test_gpu_tuning import TOL, _check_static

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("staged", ["default", "1"])
@pytest.mark.parametrize("precision", [G.FP64, G.MIXED])
@pytest.mark.parametrize("cells", [(5, 5, 5), (6, 5, 7), (23, 22, 21),
                                   (28, 28, 28)])
def test_units_match_oracle(cells, precision, staged, monkeypatch):
    # tables from L2 (small systems) or staged in LDS
    if staged != "default":
        monkeypatch.setenv("IMDG_TABLES_IN_LDS", staged)
    eam = eam_tables()
    s = W.fcc_system(cells, 3.615, eam.masses, W.kT(600.0), 77, displace=0.03)
    orc = oracle_eam(s, eam, nbl_margin=0.4, timestep=W.FS)
    orc.calc_forces()
    with G.eam_context(eam, [s], precision=precision) as gpu:
        for lanes in (None, 4, 2, 1):
            if lanes:
                gpu.set_tuning(lanes, 1024, lanes, 512)
            gpu.calc_forces()
            _check_static(gpu, orc, *TOL[precision])
            if staged != "default":
                assert gpu.info()["tables_in_lds"] == 3


@pytest.mark.parametrize("precision", [G.FP64, G.MIXED])
@pytest.mark.parametrize("case", ["eam", "alloy", "lj", "spline", "vacancies"])
def test_wide_lanes_match_oracle(case, precision):
    """Systems small enough for 8 or 16 lanes per slot with four asked for:
    every loop variant, lists longer and shorter than one body (64 entries),
    and unequal ones, against the oracle."""
    interp = G.INTERP_3POINT
    if case == "lj":
        s = W.fcc_system((7, 6, 8), 1.5496, [1.0], 0.7, 12, displace=0.02)
        orc = oracle_lj(s, nbl_margin=0.3, timestep=0.002)
        make = lambda: G.pair_context(lj(), [s], precision=precision)
    else:
        nsp = 2 if case == "alloy" else 1
        eam = eam_tables(nspecies=nsp, rc=5.5 if nsp == 2 else 5.0)
        if case == "spline":
            interp = G.INTERP_SPLINE
        s = W.fcc_system((6, 7, 6), 3.615, eam.masses, W.kT(700.0), 13,
                         displace=0.04,
                         type_fractions=(0.6, 0.4) if nsp == 2 else None,
                         vacancy_fraction=0.4 if case == "vacancies" else 0.0)
        orc = oracle_eam(s, eam, interp=interp, nbl_margin=0.4,
                         timestep=W.FS)
        make = lambda: G.eam_context(eam, [s], precision=precision,
                                     interpolation=interp)
    orc.calc_forces()
    with make() as gpu:
        gpu.calc_forces()
        _check_static(gpu, orc, *TOL[precision], has_eam=case != "lj")
        gpu.set_tuning(4, 256, 4, 256)
        gpu.calc_forces()
        _check_static(gpu, orc, *TOL[precision], has_eam=case != "lj")


@pytest.mark.parametrize("npts", [5000, 5600, 700])
def test_fp64_values_in_lds(npts, monkeypatch):
    """The FP64 force loop on the staged table values gives the bits of the
    records read from L2, over tables whose values fit in LDS and (5,600
    points with the density loop's knots) nearly fill it."""
    eam = W.johnson_eam(npts=npts)
    s = W.fcc_system((7, 6, 6), 3.615, eam.masses, W.kT(900.0), 9,
                     displace=0.08)
    got = []
    for lds in ("0", "1"):
        monkeypatch.setenv("IMDG_TABLES_IN_LDS", lds)
        with G.eam_context(eam, [s], precision=G.FP64) as gpu:
            gpu.set_tuning(4, 512, 2, 512)
            gpu.run(5)
            got.append((gpu.atoms(), gpu.info()["tables_in_lds"]))
    assert got[0][1] == 0 and got[1][1] == 3
    for k, v in got[0][0].items():
        assert np.array_equal(v, got[1][0][k]), k


@pytest.mark.parametrize("lanes", [1, 2, 4])
def test_replica_units(lanes):
    """The thermo records of a batch are those of each replica alone: FP64,
    so the sums agree to rounding whatever their order (100 terms of 1e-16
    each per atom, amplified over 10 steps by less than 10)."""
    eam = eam_tables()
    systems = [W.fcc_system(c, 3.615, eam.masses, W.kT(500.0), 5 + k,
                            displace=0.02)
               for k, c in enumerate(((5, 5, 5), (6, 6, 6), (9, 5, 7)))]
    with G.eam_context(eam, systems, precision=G.FP64) as gpu:
        gpu.set_tuning(lanes, 512, lanes, 512)
        gpu.run(10)
        th = gpu.thermo_history(0, 10)
    for r, s in enumerate(systems):
        with G.eam_context(eam, [s], precision=G.FP64) as one:
            one.run(10)
            t1 = one.thermo_history(0, 10)
        scale = np.abs(t1[:, 0, 1:6]).max(axis=0) + 1e-300
        scale[2] = np.abs(t1[:, 0, 1]).max()  # the virial's terms cancel
        assert np.all(np.abs(th[:, r, 1:6] - t1[:, 0, 1:6]) <= 1e-12 * scale)


@pytest.mark.parametrize("last_knots_only", [True, False])
def test_unequal_cross_columns_keep_four(last_knots_only, monkeypatch):
    """phi_10 not phi_01, everywhere or in the last stored rows alone: no
    column is shared, and the forces are the same bits as from the records of
    all four columns (IMDG_RHO_BY_TYPE=0).  Equal columns are compared so in
    test_gpu_branches.py."""
    eam = copy.deepcopy(eam_tables(nspecies=2, rc=5.5))  # cached tables
    v = np.array(eam.pair.values[2])
    if last_knots_only:
        v[-40:] += 1e-4     # the outermost 0.23 A^2 of r^2
    else:
        v *= 1.05
    eam.pair.values[2] = v
    s = W.fcc_system((7, 7, 5), 3.615, eam.masses, W.kT(700.0), 48,
                     type_fractions=(0.7, 0.3), displace=0.04)
    res = []
    for by_type in ("1", "0"):
        monkeypatch.setenv("IMDG_RHO_BY_TYPE", by_type)
        ctx = G.eam_context(eam, [s], precision=G.MIXED)
        monkeypatch.delenv("IMDG_RHO_BY_TYPE")
        with ctx:
            ctx.calc_forces()
            res.append(ctx.atoms())
    for k in ("f", "epot", "rho", "df"):
        assert np.array_equal(res[0][k], res[1][k]), k


@pytest.mark.parametrize("cells", [(46, 46, 46), (47, 46, 47)])
def test_large_fp64_default_shapes(cells):
    """389,344 atoms (below 24 chunks per CU on 256 CUs) and 406,456 (above):
    the default shape's densities and forces against the shape of the other
    side.  Both sum the same ~60 terms per atom, each below 60 in magnitude,
    in another order: 60 x 60 x 2^-53 x 2 < 1e-12."""
    eam = eam_tables()
    s = W.fcc_system(cells, 3.615, eam.masses, W.kT(600.0), 49, displace=0.03)
    assert (s.x.shape[0] >= 24 * 256 * 64) == (cells[0] == 47)
    below, above = (4, 1024, 1, 512), (2, 512, 2, 512)
    res = []
    with G.eam_context(eam, [s], precision=G.FP64) as gpu:
        gpu.calc_forces()
        t = gpu.tuning()
        assert (t["density_lanes"], t["density_threads"], t["force_lanes"],
                t["force_threads"]) == (above if cells[0] == 47 else below)
        res.append(gpu.atoms())
        gpu.set_tuning(*(below if cells[0] == 47 else above))
        gpu.calc_forces()
        res.append(gpu.atoms())
    for k in ("f", "epot", "rho"):
        assert np.abs(res[0][k] - res[1][k]).max() <= 1e-12, k


@pytest.mark.parametrize("lanes", [None, 2, 4])
def test_mixed_sums_keep_four_lane_accuracy(lanes):
    """Two lanes per atom (the default beyond 65,000 atoms) sum twice as many
    terms each as four.  Term by term that gives relative RMS errors of
    8.2e-8 (rho) and 1.14e-7 (energy per atom) against FP64, four lanes
    7.2e-8 and 9.0e-8: no shape may be worse than four lanes term by term,
    plus 3 % for the sample."""
    eam = eam_tables()
    s = W.fcc_system((30, 30, 30), 3.615, eam.masses, W.kT(600.0), 50,
                     displace=0.02)
    with G.eam_context(eam, [s], precision=G.FP64) as gpu:
        gpu.calc_forces()
        ref = gpu.atoms()
    with G.eam_context(eam, [s], precision=G.MIXED) as gpu:
        if lanes:
            gpu.set_tuning(lanes, 1024, lanes, 1024)
        gpu.calc_forces()
        got = gpu.atoms()
    for k, bar in (("rho", 7.25e-8), ("epot", 9.0e-8)):
        d = got[k].astype(np.float64) - ref[k]
        err = np.sqrt(np.mean(d * d) / np.mean(ref[k] ** 2))
        assert err <= 1.03 * bar, (k, err)
