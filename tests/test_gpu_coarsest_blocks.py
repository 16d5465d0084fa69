"""The dense inverse of the multigrid's coarsest level is formed sixteen pivots a
launch in tiles of 64 columns and 32 rows: coarsest sizes that are whole blocks
of sixteen and ones that leave less than a half, a half and more of one, of a few
tiles and many.  A wrong inverse entry would show as more iterations or as a
solve that falls back to the diagonal scaling; the pressure is held to the float
floor against the FP64 solve."""
import numpy as np
import pytest

import abi
import cases
import urbansph
from test_gpu_mg import rel_l2
from test_gpu_parity import F32_FLOOR_MAX

pytestmark = pytest.mark.gpu

# fluid cubes of nf^3, the part above height `cut` wall; the size their coarsest level has
SIZES = {(23, 15): 144, (21, 17): 180, (21, 21): 216, (25, 17): 245, (25, 25): 343, (21, 5): 363, (18, 18): 729,
         (21, 13): 847, (23, 13): 1008}


def _step(nf, cut, tol, **opts):
    P, _ = cases.box(nf=nf, walls=3)
    high = (P["p_type"] == 1) & (np.rint(P["z"].astype(float) / 0.01) - 3 >= cut)
    P["p_type"] = np.where(high, 0, P["p_type"])
    for f in ("ux", "uy", "uz"):
        P[f] = np.where(high, 0.0, P[f])
    prm = cases.box_params(urbansph.default_params(), tol=tol)
    prm.update(**opts)
    c = urbansph.Case(prm, len(P))
    c.upload(P)
    c.step(0, 1e-4)
    return c


@pytest.mark.parametrize("nf,cut", list(SIZES))
def test_inverse(nf, cut):
    g = _step(nf, cut, 1e-9, precision=abi.MIXED, ppe_precond=abi.PRECOND_MULTIGRID)
    r = g.ppe_report()
    print(f"[coarsest] {r.mg_coarsest} unknowns, {r.iterations} iterations", flush=True)
    assert (r.converged, r.precond, r.mg_status, r.mg_coarsest) == (1, abi.PRECOND_MULTIGRID, abi.MG_OK, SIZES[nf, cut])
    j = _step(nf, cut, 1e-9, precision=abi.MIXED).ppe_report()
    assert 2 * r.iterations <= j.iterations
    ref = _step(nf, cut, 1e-12)
    fluid = ref.ifield("P_TYPE") == 1
    assert rel_l2(g.field("PRES")[fluid], ref.field("PRES")[fluid]) <= F32_FLOOR_MAX


def test_sizes_cover_the_remainders():
    left = {n % 16 for n in SIZES.values()}
    assert 0 in left and 8 in left and any(0 < r < 8 for r in left) and any(r > 8 for r in left)
    assert min(SIZES.values()) < 3 * 64 and max(SIZES.values()) > 1000
