"""The MIXED Neumann pass (a group of lanes per boundary particle over its
listed pairs) against the FP64 oracle's: boundary pressures and lid velocities
after a step, for the last boundary particles of a case too (sizes that leave
workgroups partly empty), and with moving particles, whose records are not
packed.

Bound: a Shepard average of values whose own error is the MIXED float floor
(5e-6), with weights of one sign within about 15 float roundings: 1e-5 of the
field; at the inlet the average's gradient times a few spacings is added, whose
terms cancel to a part of their absolute sum: 2e-5.
"""
import numpy as np
import pytest

import abi
import cases
import oracle
import urbansph
from test_gpu_mg import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dx,moving", [(0.012, 0), (0.0105, 0), (0.009, 0), (0.012, 1)])
def test_mixed_neumann_equals_oracle(dx, moving):
    P, nrm, geom = cases.small_canyon(dx=dx)
    n = len(P)
    print(f"[neumann] n={n} moving={moving}", flush=True)
    prm = cases.canyon_params(geom, urbansph.default_params(), tol=1e-10)
    prm.update(ale_positions=moving)
    o = oracle.Oracle(prm, n)
    o.upload(P, None, nrm)
    assert o.step(0, 5e-5) == 0
    prm.update(precision=abi.MIXED)
    g = urbansph.Case(prm, n)
    g.upload(P, None, nrm)
    g.step(0, 5e-5)
    inlet = np.isin(o.ifield("BUFFER_TYPE"), (1, -1)) & (o.ifield("P_TYPE") != 1)
    wall = (o.ifield("P_TYPE") != 1) & ~inlet
    assert wall.any()
    assert rel_l2(g.field("PRES")[wall], o.field("PRES")[wall]) <= 1e-5
    if inlet.any():
        assert rel_l2(g.field("PRES")[inlet], o.field("PRES")[inlet]) <= 2e-5
    lid = o.ifield("P_TYPE") == -1
    vec = lambda c: np.concatenate([c.field(f)[lid] for f in ("UX", "UY", "UZ")])   # noqa: E731
    assert rel_l2(vec(g), vec(o)) <= 1e-5
