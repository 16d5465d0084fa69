"""The search's sort with its digit bases added from the scan tiles' sums, and
the cells' ranges, at particle counts around the tiles of 2048 entries (of 8
sort tiles each) and around more tiles than a workgroup has threads; the
refinement's list over several tiles of cells.  Integers and copied fields: equal."""
import numpy as np
import pytest

import abi
import cases
import oracle
import urbansph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2047, 16384, 16385, 4194304, 4194305])
def test_sort_is_stable_at_the_edges_of_its_tiles(n):
    """A small box among dummies, in random order."""
    B, _ = cases.box(nf=6, walls=3)
    P = np.zeros(n, dtype=B.dtype)
    P[:] = B[:1]
    P["i_type"] = 3
    r = np.random.RandomState(n % 1000)
    P[r.choice(n, len(B), replace=False)] = B
    prm = cases.box_params(urbansph.default_params())
    prm.update(ppe_solver=abi.PPE_REF_JACOBI)
    g = urbansph.Case(prm, n)
    g.upload(P)
    g.step(0, 1e-9)
    keys, perm, start, end = g.nnps()
    cells = len(start)
    up = np.empty(n, keys.dtype)
    up[perm] = keys
    np.testing.assert_array_equal(np.sort(perm), np.arange(n))
    np.testing.assert_array_equal(perm, np.argsort(up, kind="stable"))
    np.testing.assert_array_equal(keys == cells, P["i_type"][perm] == 3)
    lo, hi = np.searchsorted(keys, np.arange(cells)), np.searchsorted(keys, np.arange(1, cells + 1))
    np.testing.assert_array_equal(start, np.where(hi > lo, lo, -1))
    np.testing.assert_array_equal(end, np.where(hi > lo, hi, 0))


@pytest.mark.parametrize("shift", [0.2, 0.5])
def test_refinement_list_over_several_tiles_of_cells(shift):
    P, _ = cases.box(nf=6, walls=3)
    P["z"][P["z"] > 0.055] += shift
    P["y"][P["y"] > 0.055] += shift
    prm = cases.box_params(urbansph.default_params())
    prm.update(ppe_solver=abi.PPE_REF_JACOBI)
    cap = len(P) + 8 * 4000
    runs = []
    for cls in (urbansph.Case, oracle.Oracle):
        c = cls(prm, cap)
        c.upload(P)
        c.step(0, 1e-6)
        r = np.random.RandomState(3)
        target = np.where(c.ifield("P_TYPE") == 1, r.randint(0, 3, len(P)), 0.0)
        n = c.apr_refine(target.astype(np.float64), max_passes=3)
        n = n if isinstance(n, (int, np.integer)) else c.n
        runs.append((n, {f: c.field(f) for f in ("X", "Y", "Z", "M", "H", "VOL", "UX")}, c.ifield("I_TYPE"), c.nnps()))
    (ng, fg, ig, sg), (no, fo, io, so) = runs
    assert ng == no and ng > len(P)
    assert len(so[2]) > (2048 if shift < 0.3 else 3 * 2048)
    np.testing.assert_array_equal(ig, io)
    for f in fg:
        np.testing.assert_array_equal(fg[f], fo[f], err_msg=f)
    for a, b in zip(sg, so):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("n", [1728, 2048, 2049, 8191, 8192, 8193])
@pytest.mark.parametrize("shift", [0.0, 5.0])
def test_sort_of_few_particles(n, shift):
    """One workgroup up to 8192 particles; one digit of cells and three."""
    B, _ = cases.box(nf=6, walls=3)
    B["z"][B["z"] > 0.055] += shift
    B["y"][B["y"] > 0.055] += shift
    r = np.random.RandomState(n)
    P = np.zeros(n, dtype=B.dtype)
    P[:] = B[:1]
    P["i_type"] = 3
    P[r.choice(n, len(B), replace=False)] = B
    prm = cases.box_params(urbansph.default_params())
    prm.update(ppe_solver=abi.PPE_REF_JACOBI)
    g = urbansph.Case(prm, n)
    g.upload(P)
    g.step(0, 1e-9)
    keys, perm, start, end = g.nnps()
    cells = len(start)
    assert cells > (1 << 16) if shift else cells < 1 << 12
    up = np.empty(n, keys.dtype)
    up[perm] = keys
    np.testing.assert_array_equal(np.sort(perm), np.arange(n))
    np.testing.assert_array_equal(perm, np.argsort(up, kind="stable"))
    np.testing.assert_array_equal(keys == cells, P["i_type"][perm] == 3)
    np.testing.assert_array_equal(g.field("X"), P["x"][perm].astype(np.float64))
