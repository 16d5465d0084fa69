"""The launch report: the boundary passes read the sizes they run at, which are
not tuned, the others a size the autotuner timed."""
import pytest

import abi
import cases
import urbansph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,neumann", [(abi.FP64, 64), (abi.MIXED, 256)])
def test_report_of_fixed_sizes(precision, neumann):
    P, nrm, geom = cases.sized_canyon(2e4)
    prm = cases.canyon_params(geom, urbansph.default_params(), tol=1e-5, precision=precision)
    c = urbansph.Case(prm, len(P))
    c.upload(P, None, nrm)
    for s in range(8):
        c.step(s, 5e-5)
    c.sync()
    (row,) = c.tuning().values()
    assert [row[f] for f in ("boundary3d", "freeslip", "ibm_force", "neumann")] == [256, 256, 256, neumann]
    assert all(v in (64, 128, 256, 512) for v in row.values())


def test_mixed_batch_with_a_case_without_boundary():
    """A case without boundary particles beside one with them: alone = batch."""
    P, nrm, geom = cases.sized_canyon(2e4)
    prm = cases.canyon_params(geom, urbansph.default_params(), tol=1e-5, precision=abi.MIXED)
    Q, _ = cases.box(nf=8, walls=3)
    Q["p_type"] = 1
    qrm = cases.box_params(urbansph.default_params(), precision=abi.MIXED)
    for p in (prm, qrm):   # (a case of fluid alone has a singular operator: the reference's sweep)
        p.update(ppe_solver=abi.PPE_REF_JACOBI)

    def make():
        a, b = urbansph.Case(prm, len(P)), urbansph.Case(qrm, len(Q))
        a.upload(P, None, nrm)
        b.upload(Q)
        return [a, b]

    alone, batch, b = make(), make(), urbansph.Batch()
    for s in range(2):
        for c in alone:
            c.step(s, 5e-5)
        b.step(batch, [s, s], [5e-5, 5e-5])
    for x, y in zip(alone, batch):
        for f in ("PRES", "UX", "UY", "UZ"):
            assert (x.field(f) == y.field(f)).all(), f
