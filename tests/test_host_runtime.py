"""The host side of libimdg.so on a HIP runtime without a GPU (hip_stub.c):
which device its calls work on and what they allocate."""
import os
import subprocess
import sys
import textwrap

import pytest

from imd_amd import build as B

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PRELUDE = """
import ctypes as C, os, sys
sys.path[:0] = [%r, %r]
import numpy as np
from imd_amd import imdg as G
from imd_amd import workloads as W
from helpers import eam_tables, lj
stub = C.CDLL(os.environ["HIP_STUB"])
for f in ("live", "peak"):
    getattr(stub, "stub_" + f).restype = C.c_size_t
stub.stub_limit.argtypes = [C.c_size_t]
stub.stub_time.argtypes = [C.c_int, C.c_double]
for f in ("wrong_device", "mallocs", "launches"):
    getattr(stub, "stub_" + f).restype = C.c_long
stub.stub_pinned_from.restype = C.c_void_p
""" % (ROOT, os.path.join(ROOT, "tests"))


@pytest.fixture(scope="module")
def child(tmp_path_factory):
    """Runs a Python text in a process whose HIP runtime is the stub."""
    if not os.path.exists(B.LIB):
        B.build_lib()
    so = str(tmp_path_factory.mktemp("stub") / "libhip_stub.so")
    subprocess.check_call(
        ["gcc", "-std=gnu11", "-O1", "-shared", "-fPIC",
         "-I/opt/rocm/include", "-o", so,
         os.path.join(ROOT, "tests", "hip_stub.c")])
    preload = ":".join(p for p in (so, os.environ.get("LD_PRELOAD")) if p)

    def run(text, **env):
        r = subprocess.run(
            [sys.executable, "-c", PRELUDE + textwrap.dedent(text)],
            env={**os.environ, "LD_PRELOAD": preload, "HIP_STUB": so, **env},
            stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
            timeout=120)
        assert r.returncode == 0, r.stdout
        return r.stdout
    return run


def test_every_call_selects_its_device(child):
    """A context of device 1, called by a thread whose current device is 0:
    allocations and launches are on device 1."""
    child("""
        s = W.eam_crystal(n_cells=6, temp_k=300.0, seed=1)
        ctx = G.eam_context(eam_tables(), [s], device=1)
        ctx.set_stress(True)
        made = stub.stub_mallocs(0)
        assert made == 0 and stub.stub_mallocs(1) > 0
        calls = dict(
            atoms=ctx.atoms, calc_forces=ctx.calc_forces,
            move_atoms=ctx.move_atoms, check_nblist=ctx.check_nblist,
            make_nblist=ctx.make_nblist,
            deallocate_nblist=ctx.deallocate_nblist,
            run=lambda: ctx.run(3, sync=False), stress=ctx.stress,
            set_tuning=lambda: ctx.set_tuning(2, 512, 2, 512),
            autotune=lambda: ctx.autotune(1))
        for name, call in calls.items():
            stub.hipSetDevice(0)
            call()
            assert stub.stub_wrong_device() == 0, name
            assert stub.stub_mallocs(0) == 0, name
    """)


def test_autotune_times_the_shape_in_use(child):
    """The default shape of the smallest systems (blocks of one wavefront) is
    among those timed: kept, and still a default, where it is the fastest;
    replaced where another one is."""
    child("""
        small = W.eam_crystal(n_cells=6, temp_k=300.0, seed=1)
        large = W.eam_crystal(n_cells=20, temp_k=300.0, seed=2)
        for prec in (G.FP64, G.MIXED):
            with G.eam_context(eam_tables(), [small], precision=prec) as ctx:
                default = ctx.tuning()
                assert default["density_threads"] == 64
                assert default["force_threads"] == 64
                stub.stub_time(64, 0.25)
                got = ctx.autotune(2)
                stub.stub_time(64, 0.0)
                assert abs(got["density_ms"] - 0.25) < 1e-6
                assert abs(got["force_ms"] - 0.25) < 1e-6
                assert [got[k] for k in default][:4] == \\
                    [default[k] for k in default][:4]
                ctx.set_systems([large])
                assert ctx.tuning()["density_threads"] == 1024
                ctx.set_systems([small])
                stub.stub_time(256, 0.125)
                got = ctx.autotune(2)
                stub.stub_time(256, 0.0)
                assert got["density_threads"] == got["force_threads"] == 256
                ctx.set_systems([large])          # a chosen shape stays
                assert ctx.tuning()["density_threads"] == 256
        with G.pair_context(lj(), [W.lj_crystal(6)]) as ctx:
            stub.stub_time(64, 0.25)
            assert ctx.autotune(2)["force_threads"] == 64
    """)


@pytest.fixture(scope="module")
def ctl_offsets(tmp_path_factory):
    """Where the control block keeps what the tests look for or set in the
    kernels' place."""
    d = tmp_path_factory.mktemp("ctl")
    names = ("frozen", "cell_over", "export_bad", "exact_pairs", "steps_done",
             "done")
    (d / "o.cpp").write_text(
        '#include <cstddef>\n#include <cstdio>\n#include "%s"\n'
        "int main() {\n%s\n}\n"
        % (os.path.join(ROOT, "imd_amd", "csrc", "imdg_internal.h"),
           "\n".join('  printf("%%zu ", offsetof(Ctl, %s));' % n
                     for n in names)))
    subprocess.check_call(
        ["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
         "-o", str(d / "o"), str(d / "o.cpp")])
    out = subprocess.check_output([str(d / "o")], text=True).split()
    return dict(zip(names, map(int, out)))


def test_contended_counter_has_its_own_line(ctl_offsets):
    """The counter that the whole list build adds to shares no 128 B line
    with what its blocks read."""
    line = {k: v // 128 for k, v in ctl_offsets.items()}
    assert list(line.values()).count(line["exact_pairs"]) == 1


def test_empty_cells_take_little_memory(child, ctl_offsets):
    """2,048 atoms in 43 million cells take the 20 B per cell of the cell
    arrays and no buckets; in a million cells there are buckets (128 B each),
    until one full cell would make gigabytes of them."""
    child("""
        frozen, over = %s
        def cluster(ncell):
            s = W.lj_crystal(8)
            s.box = np.diag([2.8001 * ncell] * 3)
            return s
        with G.pair_context(lj(), [cluster(350)]) as ctx:
            assert ctx.grid() == (350, 350, 350)
            assert stub.stub_peak() < 20 * 350 ** 3 + (32 << 20)
        stub.stub_reset_peak()
        with G.pair_context(lj(), [cluster(100)]) as ctx:
            assert stub.stub_live() > 148 * 10 ** 6
            ctx.calc_forces()
            ctl = stub.stub_pinned_from()
            for n, least, most in ((40, 276, 300), (1200, 20, 60)):
                C.c_int.from_address(ctl + over).value = n
                C.c_int.from_address(ctl + frozen).value = 1
                ctx.calc_forces()
                assert C.c_int.from_address(ctl + over).value == 0
                assert least * 10 ** 6 < stub.stub_live() < most * 10 ** 6, n
            assert stub.stub_peak() < 500 * 10 ** 6
        # no room for the buckets: the sort does without
        stub.stub_limit(60 * 10 ** 6)
        with G.pair_context(lj(), [cluster(100)]) as ctx:
            ctx.calc_forces()
    """ % str((ctl_offsets["frozen"], ctl_offsets["cell_over"])))


def test_a_bad_export_is_reported_once(child, ctl_offsets):
    """A slot without an atom, met by one export, is that call's error and
    not the next one's."""
    child("""
        bad = %s
        s = W.eam_crystal(n_cells=6, temp_k=300.0, seed=1)
        ctx = G.eam_context(eam_tables(), [s])
        ctx.atoms()
        C.c_int.from_address(stub.stub_pinned_from() + bad).value = 1
        try:
            ctx.atoms()
        except G.ImdgError as e:
            assert "no atom" in str(e)
        else:
            raise AssertionError("not reported")
        ctx.atoms()
    """ % ctl_offsets["export_bad"])


def test_downloads_in_bounded_memory(child):
    """What a context keeps for its downloads is bounded (256 MiB), and a
    download needs no more than the memory that is left."""
    child("""
        s = W.eam_crystal(n_cells=92, temp_k=0.0, seed=1)   # 3.1 million
        ctx = G.eam_context(eam_tables(), [s])
        ctx.set_stress(True)
        ctx.run(1, sync=False)
        before = stub.stub_live()
        ctx.atoms()
        assert before < stub.stub_live() <= before + (256 << 20)
        ctx.stress()
        assert stub.stub_live() <= before + (256 << 20)
        ctx.deallocate_nblist()
        ctx.set_systems([s])
        ctx.run(1, sync=False)                   # the stress arrays
        before = stub.stub_live()
        stub.stub_limit(before + (3 << 20))
        ctx.atoms()
        ctx.stress()
        assert stub.stub_live() > before + (1 << 20)
        stub.stub_limit(before)
        try:
            ctx.atoms()
        except G.ImdgError as e:
            assert "(%d)" % G.ERR_NOMEM in str(e)
        else:
            raise AssertionError("no memory at all")
    """)


def test_scan_of_the_cells_in_its_own_launch(child):
    """The one launch of 1,024 threads in a step of small blocks is the scan
    of the cells: left out for a few small replicas, there for many and for
    large ones."""
    child("""
        for cells, nrep, per_step in ((5, 2, 0), (5, 20, 0), (5, 21, 1),
                                      (5, 64, 1), (28, 1, 0), (29, 1, 1),
                                      (20, 2, 0), (20, 3, 1)):
            s = W.eam_crystal(n_cells=cells, temp_k=300.0, seed=1)
            with G.eam_context(eam_tables(), [s] * nrep) as ctx:
                ctx.set_tuning(4, 512, 4, 512)
                ctx.run(1, sync=False)
                stub.stub_reset_launches()
                ctx.run(10, sync=False)
                assert stub.stub_launches(1024) == 10 * per_step
    """)


def test_check_ends_in_its_own_launch(child):
    """The skin test of imdg_check_nblist is two launches, the second one
    block of 1,024 threads: no fence and no count in the blocks of the
    first."""
    child("""
        for cells, nrep in ((6, 1), (21, 1), (5, 65)):
            s = W.eam_crystal(n_cells=cells, temp_k=0.0, seed=1)
            with G.eam_context(eam_tables(), [s] * nrep) as ctx:
                stub.stub_reset_launches()
                ctx.check_nblist()
                assert stub.stub_launches(128) == 1
                assert stub.stub_launches(1024) == 1, (cells, nrep)
    """)


def test_list_kernel_of_full_rebuilds(child):
    """Lanes per atom of the list build, told by its blocks (128 threads with
    one lane, as the binning's, 256 with four): by the blocks of the largest
    replica, and of all where all rebuild at once."""
    child("""
        eam = eam_tables()
        def crystal(n):
            return W.eam_crystal(n_cells=n, temp_k=0.0, seed=1)
        def dense(n):
            return W.fcc_system((n, n, n), 1.5496, [1.0], 0.0, 1)
        cases = [  # systems, pair only, precision; lanes: all rebuild, some do
            ([crystal(43)], 0, G.MIXED, 4, 4),
            ([crystal(44)], 0, G.MIXED, 1, 1),
            ([crystal(20)] * 16, 0, G.MIXED, 4, 4),   # 250 blocks each
            ([crystal(20)] * 17, 0, G.MIXED, 1, 4),
            ([crystal(20)] * 17, 0, G.FP64, 4, 4),    # 15 atoms a cell
            ([dense(9)] * 179, 1, G.FP64, 1, 4),      # 46, 23 blocks each
            ([dense(10)] * 129, 1, G.FP64, 4, 4),      # 32, 32 blocks each
        ]
        for systems, lj_only, prec, lanes_all, lanes_step in cases:
            ctx = G.pair_context(lj(), systems, precision=prec) if lj_only \\
                else G.eam_context(eam, systems, precision=prec)
            with ctx:
                ctx.set_tuning(2, 512, 2, 512)
                for call, lanes in ((ctx.make_nblist, lanes_all),
                                    (lambda: ctx.run(1, sync=False),
                                     lanes_step)):
                    stub.stub_reset_launches()
                    call()
                    got = 1 if stub.stub_launches(128) == 2 else 4
                    assert got == lanes, (len(systems), systems[0].n, prec)
    """)
