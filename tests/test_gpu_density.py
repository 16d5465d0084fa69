"""The MIXED list passes keep the reciprocals of the last neighbour's density.
Whatever density a deck holds, the first neighbour's must be formed: fields of
a step agree with the FP64 mode's, which divides pair by pair.

Tolerance: a pair term is a product of about twenty float operations (relative
error 20 * 2^-24 = 1.2e-6), the sums are double; velocities and pressures enter
as differences, which lose two digits more: 1e-4 of the field's largest value."""
import numpy as np
import pytest

import abi
import cases
import urbansph

pytestmark = pytest.mark.gpu

FIELDS = ("FLT_S", "FTOTALX", "FTOTALY", "FTOTALZ", "FPX", "FPY", "FPZ", "PRES", "UX", "UY", "UZ")


def _fields(rho, **opts):
    P, _ = cases.box(nf=8, walls=3)
    P["rho"] = rho
    P["pres"] = np.linspace(0.0, 50.0, len(P))
    prm = cases.box_params(urbansph.default_params())
    prm.update(ppe_solver=abi.PPE_REF_JACOBI, **opts)
    c = urbansph.Case(prm, len(P))
    c.upload(P)
    c.step(0, 1e-4)
    got = {f: c.field(f) for f in FIELDS}
    c.close()
    return got


@pytest.mark.parametrize("rho", [-1.0, -2.0, 1.0])
@pytest.mark.parametrize("compact,tiles", [(1, 0), (0, 0), (1, 4 | 4 << 8 | 2 << 16)])
def test_mixed_passes_at_any_density(rho, compact, tiles):
    ref = _fields(rho, precision=abi.FP64)
    got = _fields(rho, precision=abi.MIXED, compact_records=compact, tile_cells=tiles)
    for f in FIELDS:
        scale = np.abs(ref[f]).max()
        assert np.isfinite(scale) and scale > 0.0, f
        assert np.abs(got[f] - ref[f]).max() <= 1e-4 * scale, f


@pytest.mark.parametrize("field,value,which", [("rho", 0.0, "wall"), ("rho", np.inf, "one"), ("m", np.inf, "one"),
                                               ("m", 0.0, "wall"), ("rho", np.nan, "one")])
def test_mixed_divides_by_what_the_deck_holds(field, value, which):
    """Masses and densities are not checked: where the pair formulas divide by
    a zero density or an infinite one, the MIXED passes give the zeros,
    infinities and NaN of the division, as the FP64 mode does."""
    P, _ = cases.box(nf=8, walls=3)
    fluid = np.flatnonzero(P["p_type"] == 1)
    P[field][np.flatnonzero(P["p_type"] == 0) if which == "wall" else fluid[3]] = value
    got = {}
    for precision in (abi.FP64, abi.MIXED):
        prm = cases.box_params(urbansph.default_params(), precision=precision)
        prm.update(ppe_solver=abi.PPE_REF_JACOBI)
        c = urbansph.Case(prm, len(P))
        c.upload(P)
        c.step(0, 1e-4)
        got[precision] = {f: c.field(f) for f in ("FLT_S", "INV_CM_XX", "INV_CM_XY", "INV_CM_ZZ")}
        c.close()
    for f, ref in got[abi.FP64].items():
        g = got[abi.MIXED][f]
        np.testing.assert_array_equal(np.isnan(g), np.isnan(ref), err_msg=f)
        odd = ~np.isfinite(ref)
        np.testing.assert_array_equal(g[odd], ref[odd], err_msg=f)
        assert np.abs(g[~odd] - ref[~odd]).max() <= 1e-4 * np.abs(ref[~odd]).max(), f
