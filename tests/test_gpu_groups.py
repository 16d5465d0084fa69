"""The MIXED passes that share a particle among a group of lanes (strain,
gradient correction, advection, pressure force, PPE assembly) against the
FP64 oracle, at particle counts that leave workgroups and groups partly
empty, for every kernel, viscosity and scalar option their pair formulas
branch on.

Bounds: the pressure and the velocity of a step whose solve is converged
(tolerance 1e-10) carry only the float pair sums' error, the MIXED float
floor of the parity tests (5e-6); a force sum's terms take at most 25
float roundings (1.5e-6) and its terms cancel to a fifth or more of their
absolute sum, so 1e-5 of the field.
"""
import numpy as np
import pytest

import abi
import cases
import oracle
import urbansph
from test_gpu_mg import rel_l2
from test_gpu_parity import F32_FLOOR_MAX

pytestmark = pytest.mark.gpu

DT = 1e-4


def _step(cls, prm, P, steps):
    c = cls(prm, len(P))
    c.upload(P)
    for s in range(steps):
        c.step(s, DT)
    return c


def _compare(P, steps=1, **opts):
    ref = cases.box_params(oracle.default_params(), tol=1e-12)
    ref.update(**opts)
    prm = cases.box_params(urbansph.default_params(), tol=1e-10, precision=abi.MIXED)
    prm.update(**opts)
    g, o = _step(urbansph.Case, prm, P, steps), _step(oracle.Oracle, ref, P, steps)
    fluid = o.ifield("P_TYPE") == 1
    vec = lambda c, f: np.concatenate([c.field(f + a)[fluid] for a in "XYZ"])   # noqa: E731
    for f, bound in (("U", F32_FLOOR_MAX), ("FTOTAL", 1e-5), ("FP", 1e-5)):
        e = rel_l2(vec(g, f), vec(o, f))
        assert e <= bound, (f, e)
    for f, bound in (("PRES", F32_FLOOR_MAX), ("FLT_S", 1e-5), ("INV_CM_XX", 1e-5), ("INV_CM_YZ", 1e-5)):
        e = rel_l2(g.field(f)[fluid], o.field(f)[fluid])
        assert e <= bound, (f, e)
    return g, o, fluid


# 7^3 .. 15^3 particles: below one 64-particle slice of fluid, and counts that
# are no multiple of the 8 .. 64 particles of a workgroup
@pytest.mark.parametrize("nf,walls", [(3, 2), (5, 3), (8, 3), (9, 3)])
def test_group_passes_at_odd_sizes(nf, walls):
    P, _ = cases.box(nf=nf, walls=walls)
    _compare(P, steps=2)


@pytest.mark.parametrize("kernel", range(6))
def test_group_passes_every_kernel(kernel):
    P, _ = cases.box(nf=7, walls=3)
    _compare(P, kernel_type=kernel)


def test_group_passes_monaghan_and_les():
    P, _ = cases.box(nf=8, walls=3, sigma_u=0.05)
    g, o, fluid = _compare(P, fv_solve=abi.FV_MONAGHAN, turbulence_model=abi.SSM)
    assert rel_l2(g.field("VIS_T")[fluid], o.field("VIS_T")[fluid]) <= 1e-5


def test_group_passes_scalars():
    P, _ = cases.box(nf=8, walls=3)
    P["temp"] = 300.0 + 5.0 * np.sin(40.0 * P["x"]) * np.cos(30.0 * P["z"])
    P["concn"] = 1.0 + 0.5 * np.cos(35.0 * P["y"])
    g, o, fluid = _compare(P, con_solve=1, concn_solve=1, boussinesq_solve=1, turbulence_model=abi.DDF, diff_coef=1e-4)
    for f in ("DTEMP", "DCONCN"):
        assert rel_l2(g.field(f)[fluid], o.field(f)[fluid]) <= 1e-5, f


def test_group_passes_varying_density_and_spacing():
    """Neighbours of different density and h: nothing kept from the previous
    pair of a lane may enter the next one."""
    P, _ = cases.box(nf=8, walls=3)
    k = np.arange(len(P))
    P["rho"] = 1000.0 + 50.0 * (k % 3)
    P["m"] = P["rho"] * np.float32(1e-6)
    P["h"] = np.float32(0.015) * np.where(k % 2 == 0, 1.0, 0.9)
    _compare(P)


def test_group_passes_coinciding_particles():
    """Two fluid particles at one place: their pair contributes nothing to
    the sums along the distance, and everything stays finite."""
    P, _ = cases.box(nf=8, walls=3)
    fl = np.flatnonzero(P["p_type"] == 1)
    a, b = fl[len(fl) // 2], fl[len(fl) // 2 + 1]
    for n in ("x", "y", "z"):
        P[n][b] = P[n][a]
    _compare(P)
