"""The operator read past the caches and through them: two canyons whose
operators together exceed the caches' share give in a batch (nontemporal
loads) the bits that each gives alone (plain loads)."""
import numpy as np
import pytest

import abi
import cases
import urbansph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,target", [(abi.MIXED, 520000), (abi.FP64, 190000)])
def test_products_do_not_depend_on_the_loads(precision, target):
    # slots a particle x bytes a slot: 66 x 4 (MIXED, stencil slices), 78 x 10 (FP64);
    # alone below 240 MB, together above
    P, nrm, geom = cases.sized_canyon(target, u_scale=1.0, bh=0.08, dx=0.008)
    print(f"[streams] n={len(P)} precision={precision}", flush=True)
    prm = cases.canyon_params(geom, urbansph.default_params(), tol=1e-5)
    prm.update(precision=precision)

    def case():
        c = urbansph.Case(prm, len(P))
        c.upload(P, None, nrm)
        return c

    one = case()
    one.step(0, 5e-5)
    ref = {f: one.field(f) for f in ("PRES", "UX", "UY", "UZ")}
    slots, value = one.ppe_report().slots, 4 if precision == abi.MIXED else 10
    assert slots * value < 240e6 < 2 * slots * value
    del one
    pair = [case(), case()]
    b = urbansph.Batch()
    b.step(pair, [0, 0], [5e-5, 5e-5])
    for c in pair:
        for f, v in ref.items():
            np.testing.assert_array_equal(c.field(f), v, err_msg=f)
