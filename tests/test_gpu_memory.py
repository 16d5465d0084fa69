"""Device memory a context holds, blocks cached for its next search included: a
server admits requests by it, so a search keeps no scratch of its own, only the
records the case's passes read are there, and a set-up gives its blocks back.
Bounds in bytes a particle for the 120 k canyon, one per cent above what contexts
held when a search gathered its arrays one at a time (2999, 2213, 2956, 4033 and
4003 bytes, and 3034, 2245, 3430 and 4520 after further uploads)."""
import pytest

import abi
import cases
import urbansph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,precond,ale,first,again", [
    (abi.MIXED, abi.PRECOND_MULTIGRID, 0, 3030, 3065),
    (abi.MIXED, abi.PRECOND_JACOBI, 0, 2235, 2268),
    (abi.FP64, abi.PRECOND_JACOBI, 0, 2985, 3465),
    (abi.FP64, abi.PRECOND_MULTIGRID, 0, 4075, 4565),
    (abi.MIXED, abi.PRECOND_MULTIGRID, 1, 4045, 0)])
def test_held_bytes(precision, precond, ale, first, again):
    P, nrm, geom = cases.sized_canyon(1.2e5)
    prm = cases.canyon_params(geom, urbansph.default_params(), tol=1e-6, precision=precision)
    prm.update(ppe_precond=precond, ale_positions=ale)
    c = urbansph.Case(prm, len(P))
    c.upload(P, None, nrm)
    for s in range(4 if ale else 2):
        c.step(s, 5e-5)
    c.sync()
    held = c.device_bytes() / len(P)
    print(f"[memory] {held:.0f} bytes a particle", flush=True)
    assert held <= first
    if again:   # the same context, uploaded and searched again
        for _ in range(3):
            c.upload(P, None, nrm)
            c.step(0, 5e-5)
        c.sync()
        held = c.device_bytes() / len(P)
        print(f"[memory] after further uploads {held:.0f}", flush=True)
        assert held <= again
    c.close()
