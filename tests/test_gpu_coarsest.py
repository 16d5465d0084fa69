"""The dense inverse of the multigrid's coarsest level, formed eight pivots a
launch: coarsest sizes that are whole blocks of eight and ones that leave a
remainder, in cubes and slabs of different extents.  A wrong inverse entry
would show as more iterations (the Jacobi solve takes 25 or more) or as a
solve that falls back to the diagonal scaling; the converged pressure is held
to the float floor against the FP64 oracle."""
import numpy as np
import pytest

import abi
import cases
import oracle
import urbansph
from test_gpu_mg import rel_l2
from test_gpu_parity import F32_FLOOR_MAX

pytestmark = pytest.mark.gpu


def _slab(nf, cut):
    """The nf^3 box with the fluid above height `cut` turned to wall."""
    P, _ = cases.box(nf=nf, walls=3)
    k = np.rint(P["z"].astype(float) / 0.01) - 3
    high = (P["p_type"] == 1) & (k >= cut)
    P["p_type"] = np.where(high, 0, P["p_type"])
    for f in ("ux", "uy", "uz"):
        P[f] = np.where(high, 0.0, P[f])
    return P


SIZES = [(11, 11), (12, 10), (13, 9), (14, 9), (16, 16), (18, 7)]


def _run(nf, cut, precision, precond, tol):
    P = _slab(nf, cut)
    prm = cases.box_params(urbansph.default_params(), tol=tol, precision=precision)
    prm.update(ppe_precond=precond)
    c = urbansph.Case(prm, len(P))
    c.upload(P)
    c.step(0, 1e-4)
    return c, P


@pytest.mark.parametrize("nf,cut", SIZES)
def test_coarsest_inverse(nf, cut):
    g, P = _run(nf, cut, abi.MIXED, abi.PRECOND_MULTIGRID, 1e-9)
    r = g.ppe_report()
    assert (r.converged, r.precond, r.mg_status) == (1, abi.PRECOND_MULTIGRID, abi.MG_OK)
    j, _ = _run(nf, cut, abi.MIXED, abi.PRECOND_JACOBI, 1e-9)
    assert 2 * r.iterations <= j.ppe_report().iterations, (r.mg_coarsest, r.iterations)
    o = oracle.Oracle(cases.box_params(oracle.default_params(), tol=1e-12), len(P))
    o.upload(P)
    o.step(0, 1e-4)
    fluid = o.ifield("P_TYPE") == 1
    assert rel_l2(g.field("PRES")[fluid], o.field("PRES")[fluid]) <= F32_FLOOR_MAX


def test_coarsest_sizes_cover_remainders():
    left = {_run(nf, cut, abi.MIXED, abi.PRECOND_MULTIGRID, 1e-6)[0].ppe_report().mg_coarsest % 8 for nf, cut in SIZES}
    assert 0 in left and len(left) >= 3, left
