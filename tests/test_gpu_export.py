"""imdg_get_atoms / imdg_get_stress: the device puts the slots back into
input order.  Replicas of sizes around the 128-slot block, an empty one among
them; every array is identified with its atom through the mass and a
momentum that encode the input index, and a call that asks for some of the
arrays returns the same bytes as one that asks for all."""
import ctypes as C

import numpy as np
import pytest

from imd_amd import imdg as G
from imd_amd import workloads as W

from helpers import eam_tables

pytestmark = pytest.mark.gpu


def _systems():
    out = []
    for k, keep in enumerate((1, 127, 128, 0, 129, 864)):
        s = W.eam_crystal(n_cells=6, temp_k=300.0, seed=40 + k)
        rng = np.random.default_rng(k)
        at = rng.permutation(s.n)[:keep]
        s.x, s.p, s.type = s.x[at], s.p[at], s.type[at]
        s.mass, s.id = s.mass[at], np.arange(keep)
        out.append(s)
    return out


@pytest.mark.parametrize("precision", [G.FP64, G.MIXED])
def test_input_order_and_subsets(precision):
    systems = _systems()
    n = sum(s.n for s in systems)
    tag = np.arange(n, dtype=np.float64)
    at = 0
    for s in systems:
        s.p = np.column_stack([tag[at:at + s.n], -tag[at:at + s.n],
                               0.5 * tag[at:at + s.n]])
        at += s.n
    with G.eam_context(eam_tables(), systems, precision=precision) as ctx:
        ctx.make_nblist()          # sorts the slots; nothing moves
        ctx.calc_forces()
        full = ctx.atoms()
        assert np.array_equal(full["p"][:, 0], tag)
        assert np.array_equal(full["p"][:, 1], -tag)
        assert np.array_equal(full["x"], np.concatenate(
            [np.mod(s.x, np.diag(s.box)) for s in systems]))
        # the lone atom of the first replica feels nothing
        assert not full["f"][0].any() and full["rho"][0] == 0.0
        names = ("x", "p", "f", "epot", "rho", "df")
        for mask in (0, 1, 4, 8, 36, 63):
            arr = [np.full_like(full[k], 7.0) if mask >> q & 1 else None
                   for q, k in enumerate(names)]
            ptr = [a.ctypes.data_as(C.POINTER(C.c_double)) if a is not None
                   else None for a in arr]
            assert G.lib().imdg_get_atoms(ctx._h, *ptr) == G.OK
            for a, k in zip(arr, names):
                assert a is None or np.array_equal(a, full[k])


@pytest.mark.parametrize("precision", [G.FP64, G.MIXED])
def test_stress_in_input_order(precision):
    """Free particles: the tensor is p p^T / m of the atom itself."""
    s = W.eam_crystal(n_cells=6, temp_k=300.0, seed=3)
    s.x, s.p, s.type, s.mass = s.x[::7], s.p[::7], s.type[::7], s.mass[::7]
    s.id = np.arange(s.x.shape[0])
    flat = W.table_from_functions([lambda r: 0.0 * r], 1.0, 25.0, 500)
    ctx = G.Context(precision=precision, ntypes=1, timestep=W.FS,
                    nbl_margin=0.4)
    with ctx:
        ctx.set_tables(G.TableArrays.from_format2(flat))
        ctx.set_systems([s])
        ctx.set_stress(True)
        ctx.run(2)
        per, _ = ctx.stress()
    want = np.stack([s.p[:, a] * s.p[:, b] / s.mass for a, b in
                     ((0, 0), (1, 1), (2, 2), (1, 2), (2, 0), (0, 1))], 1)
    assert np.array_equal(per, want)


def test_windows_of_a_large_download():
    """5.8 million atoms: all arrays together go out in three windows, the
    stress tensor in two, an array alone in one; the bytes are the same, and
    free particles have p p^T / m."""
    s = W.fcc_system((113, 113, 113), 3.615, [W.MASS_CU], W.kT(300.0), 9)
    assert s.n * 12 * 8 > 2 * (256 << 20) and s.n * 6 * 8 > 256 << 20
    flat = W.table_from_functions([lambda r: 0.0 * r + 1.0], 1.0, 25.0, 500)
    ctx = G.Context(precision=G.MIXED, ntypes=1, timestep=W.FS,
                    nbl_margin=0.4)
    with ctx:
        ctx.set_tables(G.TableArrays.from_format2(flat))
        ctx.set_systems([s])
        ctx.set_stress(True)
        ctx.run(1)
        full = ctx.atoms()
        assert np.array_equal(full["p"], s.p)
        for q, k in enumerate(("x", "p", "f", "epot", "rho", "df")):
            one = np.full_like(full[k], 7.0)
            ptr = [None] * 6
            ptr[q] = one.ctypes.data_as(C.POINTER(C.c_double))
            assert G.lib().imdg_get_atoms(ctx._h, *ptr) == G.OK
            assert np.array_equal(one, full[k]), k
        per, _ = ctx.stress()
    want = np.stack([s.p[:, a] * s.p[:, b] / s.mass for a, b in
                     ((0, 0), (1, 1), (2, 2), (1, 2), (2, 0), (0, 1))], 1)
    assert np.array_equal(per, want)
