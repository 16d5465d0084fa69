"""MIXED spreading of the marker forces (a group of lanes per particle) and
the marker flags of the lists, against the FP64 oracle.

Bound: the Shepard sum has terms of one sign, each within about 15 float
roundings (9e-7) and near the kernel's edge four times that of a term that is
small there: 1e-5 of the field.  The force is that average of the markers'
forces, so the oracle spreads the forces that the MIXED run's markers hold.
"""
import numpy as np
import pytest

import abi
import cases
import oracle
import urbansph
from test_gpu_mg import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dx", [0.012, 0.009])
@pytest.mark.parametrize("kernel", [abi.WENDLAND2, abi.QUINTIC])
def test_mixed_spreading_equals_oracle(dx, kernel):
    P, nrm, geom = cases.small_canyon(dx=dx)
    n = len(P)
    print(f"[ibm] n={n} kernel={kernel}", flush=True)
    prm = cases.canyon_params(geom, urbansph.default_params(), tol=1e-10)
    prm.update(kernel_type=kernel)
    o = oracle.Oracle(prm, n)
    o.upload(P, None, nrm)
    prm.update(precision=abi.MIXED)
    g = urbansph.Case(prm, n)
    g.upload(P, None, nrm)
    for s in range(2):
        assert o.step(s, 5e-5) == 0
        g.step(s, 5e-5)
    fluid = o.ifield("P_TYPE") == 1
    filt_o, filt_g = o.field("CONCENTRATION")[fluid], g.field("CONCENTRATION")[fluid]
    assert (filt_o > 0).any() and (filt_o == 0).any()
    np.testing.assert_array_equal(filt_g == 0, filt_o == 0)
    assert rel_l2(filt_g, filt_o) <= 1e-5
    marker = o.ifield("P_TYPE") == 1000
    for a in "XYZ":
        o.set_work("FB" + a, np.where(marker, g.field("FB" + a), 0.0))
    assert o.run_pass("ibm_spread") in (None, 0)
    vec = lambda f: np.concatenate([f("FB" + a)[fluid] for a in "XYZ"])   # noqa: E731
    assert rel_l2(vec(g.field), vec(o.work)) <= 1e-5
