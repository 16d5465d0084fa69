"""The neighbour lists of the search (distances compared by their squares,
rows of cells out of reach skipped, particles of one window listed together)
against the oracle's pairs, exactly: one or several smoothing lengths, lengths
so small that the 1e-20 of the distance formulas counts, flat and offset
clouds, a particle outside the binning range, and every remainder of a wave's
four particles."""
import numpy as np
import pytest

import abi
import oracle
import urbansph
from test_gpu_parity import assert_nnps_equal
from test_oracle_nnps import _random_cloud

pytestmark = pytest.mark.gpu


def _cloud(n, kind):
    P = _random_cloud(max(n, 40), seed=n)
    r = np.random.default_rng(n + 1)
    P["h_ref"] = 0.012
    if kind in ("varied", "tiny_varied"):
        P["h"] = 0.012 * r.choice([0.5, 1.0, 1.7], len(P))
    if kind == "flat":
        P["y"] = 0.03
    if kind == "offset":
        P["x"] += 57.0
    if kind == "outside":       # the range leaves out the last particle, which joins an end cell
        P["x"][-1], P["y"][-1] = 0.21, 0.16
    if kind == "lattice":       # distances that equal the radii
        k = np.arange(len(P))
        d = np.float32(0.012)
        P["x"], P["y"], P["z"] = k % 11 * d, k // 11 % 9 * d, k // 99 * d
    if kind.startswith("tiny"):
        for f in ("x", "y", "z", "h", "h_ref"):
            P[f] *= np.float32(2e-4)
    return P[len(P) - n:]


@pytest.mark.parametrize("kind", ["uniform", "varied", "flat", "offset", "outside", "lattice", "tiny", "tiny_varied"])
@pytest.mark.parametrize("n", [33, 67, 2001])
def test_lists_equal_oracle(n, kind):
    P = _cloud(n, kind)
    print(f"[lists] n={n} {kind}", flush=True)
    prm = urbansph.default_params()
    prm.update(ppe_solver=abi.PPE_REF_JACOBI)
    o = oracle.Oracle(prm, n)
    o.upload(P)
    assert o.step(0, 1e-9) == 0
    g = urbansph.Case(prm, n)
    g.upload(P)
    g.step(0, 1e-9)
    g.sync()
    assert_nnps_equal(o, g)
