"""The solve's scalar steps inside its vector kernels (up to 1024 chunks of
rows) and in a kernel of their own (more): a case gives the same bits alone,
folded, and in a batch with a case too large for that, not folded; one chunk,
a few and several hundred."""
import numpy as np
import pytest

import abi
import cases
import urbansph

pytestmark = pytest.mark.gpu

FIELDS = ("PRES", "UX", "UY", "UZ")


def _case(target, precision, precond):
    if target < 5000:
        P, nrm = cases.box(nf=target, walls=3)
        prm = cases.box_params(urbansph.default_params(), tol=1e-9)
    else:
        P, nrm, geom = cases.sized_canyon(target, u_scale=1.0, bh=0.08, dx=0.008)
        prm = cases.canyon_params(geom, urbansph.default_params(), tol=1e-6)
    prm.update(precision=precision, ppe_precond=precond)
    c = urbansph.Case(prm, len(P))
    c.upload(P, None, nrm)
    return c


def _result(c):
    r = c.ppe_report()
    return {f: c.field(f) for f in FIELDS}, (r.iterations, r.converged, r.rel_residual, r.unknowns)


@pytest.mark.parametrize("precision,precond", [(abi.FP64, abi.PRECOND_JACOBI), (abi.MIXED, abi.PRECOND_MULTIGRID)])
def test_folded_scalars_equal_their_kernel(precision, precond):
    sizes = (5, 11, 100000, 360000)
    print(f"[fold] precision={precision}", flush=True)
    alone = []
    for n in sizes:
        c = _case(n, precision, precond)
        for s in range(2):
            c.step(s, 5e-5)
        alone.append(_result(c))
        c.close()
    rows = [a[1][3] for a in alone]
    assert rows[0] <= 256 < rows[1] and rows[1] < 65536 < rows[2] < 262144 < rows[3]
    batch = [_case(n, precision, precond) for n in sizes]
    b = urbansph.Batch()
    for s in range(2):
        b.step(batch, [s] * len(sizes), [5e-5] * len(sizes))
    for c, (fields, report) in zip(batch, alone):
        got, rep = _result(c)
        assert rep == report
        for f in FIELDS:
            np.testing.assert_array_equal(got[f], fields[f], err_msg=f)
