"""Matrix rows whose entry counts sit on and around the rounds of the row
products (8 entries in FP64, 16 in the mixed mode): one, a full round, one
entry more or less, and rows of every count up to the box's 100-odd, against
the FP64 oracle's converged solve.  The product adds a row's entries in
order, so FP64 keeps the parity bound of 1e-10; MIXED the float floor."""
import numpy as np
import pytest

import abi
import cases
import oracle
import urbansph
from test_gpu_mg import rel_l2
from test_gpu_parity import F32_FLOOR_MAX

pytestmark = pytest.mark.gpu


def _solve(cls, prm, P):
    c = cls(prm, len(P))
    c.upload(P)
    c.step(0, 1e-4)
    return c


# a rod of fluid particles `m` long and 1 or 2 wide in a wall box: rows of
# few entries; the cube gives the long ones
def _rod(m, width):
    P, _ = cases.box(nf=m, walls=2, sigma_u=0.02)
    mid = 0.01 * (2 + m // 2)
    y, z = P["y"].astype(float), P["z"].astype(float)
    keep = (np.abs(y - mid) < 0.01 * (width - 0.5)) & (np.abs(z - mid) < 0.01 * (width - 0.5))
    P["p_type"] = np.where((P["p_type"] == 1) & keep, 1, 0)
    for f in ("ux", "uy", "uz"):
        P[f] = np.where(P["p_type"] == 1, P[f], 0.0)
    return P


DECKS = {f"rod{m}x{w}": (lambda m=m, w=w: _rod(m, w)) for m, w in ((2, 1), (5, 1), (9, 1), (9, 2), (12, 2))}
DECKS["cube10"] = lambda: cases.box(nf=10, walls=2)[0]


@pytest.mark.parametrize("index16", [0, 1])
@pytest.mark.parametrize("deck", sorted(DECKS))
def test_row_products(deck, index16):
    P = DECKS[deck]()
    ref = cases.box_params(oracle.default_params(), tol=1e-12)
    o = _solve(oracle.Oracle, ref, P)
    fluid = o.ifield("P_TYPE") == 1
    for precision, tol, bound in ((abi.FP64, 1e-12, 1e-10), (abi.MIXED, 1e-10, F32_FLOOR_MAX)):
        prm = cases.box_params(urbansph.default_params(), tol=tol, precision=precision)
        prm.update(ppe_index16=index16)
        g = _solve(urbansph.Case, prm, P)
        for f in ("PRES", "UX"):
            e = rel_l2(g.field(f)[fluid], o.field(f)[fluid])
            assert e <= bound, (deck, precision, f, e)
