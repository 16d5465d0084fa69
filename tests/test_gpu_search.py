"""The search's permutation of the whole state (several arrays a launch) and
the refinement's picks and children, at particle counts around a workgroup's
256, against numpy and the oracle: integer results and copied fields exactly."""
import numpy as np
import pytest

import abi
import cases
import oracle
import urbansph

pytestmark = pytest.mark.gpu

DOUBLES = ["X", "Y", "Z", "M", "H", "RHO", "CONCN", "ENTHALPY", "PRES0", "VOL", "FLOAT1", "HMZ"]
INTS = {"BUFFER_TYPE": "buffer_type", "P_TYPE": "p_type", "SOURCE": "source", "I_TYPE": "i_type"}


@pytest.mark.parametrize("n", [2, 64, 255, 256, 257, 513, 1700])
def test_search_permutes_every_field(n):
    P, _ = cases.box(nf=6, walls=3)
    r = np.random.RandomState(n)
    P = P[r.permutation(len(P))[:n]]
    for f in ("concn", "enthalpy", "vol", "float1", "hmz"):
        P[f] = r.uniform(0.5, 1.5, n)
    P["source"] = r.randint(0, 100, n)
    P["float1"][P["p_type"] == 1] = 0.0      # the wall model's diagnostics start a step at these values
    prm = cases.box_params(urbansph.default_params())
    prm.update(ppe_solver=abi.PPE_REF_JACOBI)
    g = urbansph.Case(prm, n + 7)
    g.upload(P)
    g.step(0, 1e-9)
    o = oracle.Oracle(prm, n + 7)
    o.upload(P)
    o.step(0, 1e-9)
    kg, pg, sg, eg = g.nnps()
    ko, po, so, eo = o.nnps()
    for a, b in ((kg, ko), (pg, po), (sg, so), (eg, eo)):
        np.testing.assert_array_equal(a, b)
    for f in DOUBLES:
        np.testing.assert_array_equal(g.field(f), o.field(f), err_msg=f)
        if f != "CONCN":   # the step adds to it at particles of source 1
            np.testing.assert_array_equal(g.field(f), P[f.lower()][pg].astype(np.float64), err_msg=f)
    for f, name in INTS.items():
        np.testing.assert_array_equal(g.ifield(f), P[name][pg], err_msg=f)


@pytest.mark.parametrize("nf,passes", [(5, 1), (6, 2), (7, 3)])
def test_refinement_passes_equal_oracle(nf, passes):
    """Cells with no, one and several particles that want to split, non-fluid
    ones with a high target (which block their cell) among them."""
    P, _ = cases.box(nf=nf, walls=3)
    prm = cases.box_params(urbansph.default_params())
    prm.update(ppe_solver=abi.PPE_REF_JACOBI)
    cap = len(P) + 8 * 4000
    runs = []
    for cls in (urbansph.Case, oracle.Oracle):
        c = cls(prm, cap)
        c.upload(P)
        c.step(0, 1e-6)
        r = np.random.RandomState(nf)
        target = np.where(c.ifield("P_TYPE") == 1, r.randint(0, 3, len(P)), 3.0 * (r.uniform(size=len(P)) < 0.02))
        n = c.apr_refine(target.astype(np.float64), max_passes=passes)
        n = n if isinstance(n, (int, np.integer)) else c.n
        runs.append((n, {f: c.field(f) for f in ("X", "Y", "Z", "M", "H", "VOL", "UX")}, c.ifield("I_TYPE"), c.nnps()))
    (ng, fg, ig, sg), (no, fo, io, so) = runs
    assert ng == no and ng > len(P)
    np.testing.assert_array_equal(ig, io)
    for f in fg:
        np.testing.assert_array_equal(fg[f], fo[f], err_msg=f)
    for a, b in zip(sg, so):
        np.testing.assert_array_equal(a, b)
