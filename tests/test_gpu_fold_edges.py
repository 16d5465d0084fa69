"""The solve's scalar steps inside its vector kernels, at the edge of the rule
(1024 partials, 262,144 rows): a case at the edge, folded alone, gives in a batch
with one of a row more, which nothing folds, the bits it gives alone; in both
precisions with both preconditioners.  And solves that end anywhere in an
iteration, after its half step among the rest: a small case at many tolerances."""
import numpy as np
import pytest

import abi
import cases
import urbansph

pytestmark = pytest.mark.gpu

EDGE = 1024 * 256
FIELDS = ("PRES", "UX", "UY", "UZ")
KINDS = [(abi.FP64, abi.PRECOND_JACOBI), (abi.FP64, abi.PRECOND_MULTIGRID), (abi.MIXED, abi.PRECOND_JACOBI),
         (abi.MIXED, abi.PRECOND_MULTIGRID)]


def _canyon(rows, precision, precond, tol=1e-6):
    P, nrm, geom = cases.sized_canyon(342000, u_scale=1.0, bh=0.08, dx=0.008)
    fluid = np.flatnonzero(P["p_type"] == 1)
    assert len(fluid) >= rows
    P["p_type"][fluid[:len(fluid) - rows]] = 0
    prm = cases.canyon_params(geom, urbansph.default_params(), tol=tol, precision=precision)
    prm.update(ppe_precond=precond)
    c = urbansph.Case(prm, len(P))
    c.upload(P, None, nrm)
    return c


def _box(precision, precond, tol):
    P, _ = cases.box(nf=11, walls=3)
    prm = cases.box_params(urbansph.default_params(), tol=tol, precision=precision)
    prm.update(ppe_precond=precond)
    c = urbansph.Case(prm, len(P))
    c.upload(P)
    return c


def _result(c):
    r = c.ppe_report()
    return [c.field(f) for f in FIELDS] + [np.array([r.iterations, r.converged, r.rel_residual, r.unknowns, r.precond])]


def _same(a, b):
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("precision,precond", KINDS)
def test_edge_of_the_rule(precision, precond):
    print(f"[fold] edge, precision {precision} preconditioner {precond}", flush=True)
    alone = []
    for rows in (EDGE, EDGE + 1):
        c = _canyon(rows, precision, precond)
        c.step(0, 5e-5)
        alone.append(_result(c))
        c.close()
    assert [a[-1][3] for a in alone] == [EDGE, EDGE + 1] and [a[-1][4] for a in alone] == [precond] * 2
    pair = [_canyon(EDGE, precision, precond), _canyon(EDGE + 1, precision, precond)]
    urbansph.Batch().step(pair, [0, 0], [5e-5, 5e-5])
    for c, a in zip(pair, alone):
        _same(_result(c), a)


@pytest.mark.parametrize("precision,precond", KINDS)
def test_any_end_of_a_solve(precision, precond):
    tols = [m * 10.0 ** -k for k in range(2, 9) for m in (1.0, 0.5, 0.2)]
    print(f"[fold] {len(tols)} tolerances, precision {precision} preconditioner {precond}", flush=True)
    alone = []
    for tol in tols:
        c = _box(precision, precond, tol)
        c.step(0, 1e-4)
        alone.append(_result(c))
        c.close()
    its = [a[-1][0] for a in alone]
    assert max(its) > min(its)
    batch = [_box(precision, precond, tol) for tol in tols] + [_canyon(EDGE + 1, precision, precond)]
    urbansph.Batch().step(batch, [0] * len(batch), [1e-4] * len(tols) + [5e-5])
    for c, a in zip(batch, alone):
        _same(_result(c), a)
