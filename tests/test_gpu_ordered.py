"""FP64 passes that share a particle among lanes and add its terms in list
order: the sums of one step before the pressure solve equal the oracle's
serial sums bit for bit (the same IEEE operations in the same order), at
particle counts that leave groups and workgroups partly empty and for every
option that adds a term; the boundary passes and the pressure force after it
within the FP64 tolerance, which the solve sets."""
import numpy as np
import pytest

import abi
import cases
import oracle
import urbansph
from test_gpu_parity import FP64_TOL, rel_l2, run_pair

pytestmark = pytest.mark.gpu

EXACT = ["INV_CM_XX", "INV_CM_XY", "INV_CM_YY", "INV_CM_YZ", "INV_CM_ZX", "INV_CM_ZZ", "FLT_S", "SR", "VIS_T",
         "FTOTALX", "FTOTALY", "FTOTALZ", "FTOTAL", "DTEMP", "DCONCN"]
OPTIONS = {
    "cleary": dict(),
    "monaghan_les": dict(fv_solve=abi.FV_MONAGHAN, turbulence_model=abi.SSM),
    "artificial": dict(artificial_viscosity=1, av_alpha=0.1, av_beta=0.2, av_c=10.0),
    "scalars": dict(con_solve=1, concn_solve=1, boussinesq_solve=1, diff_coef=1e-4, artificial_viscosity=1,
                    av_alpha=0.1, av_c=10.0),
    "no_pressure_force": dict(fp_solve=0),
}


@pytest.mark.parametrize("options", OPTIONS)
@pytest.mark.parametrize("nf,walls", [(3, 2), (5, 3), (9, 3)])
def test_ordered_sums_equal_serial(nf, walls, options):
    P, _ = cases.box(nf=nf, walls=walls)
    P["temp"] = 300.0 + 5.0 * np.sin(40.0 * P["x"]) * np.cos(30.0 * P["z"])
    P["concn"] = 1.0 + 0.5 * np.cos(35.0 * P["y"])
    P["eli"] = 0.25
    prm = cases.box_params(urbansph.default_params(), tol=1e-12)
    prm.update(**OPTIONS[options])
    o, g = run_pair(P, prm)
    for f in EXACT:
        np.testing.assert_array_equal(g.field(f), o.field(f), err_msg=f)
    for f in ("FPX", "FPY", "FPZ", "PRES", "UX", "TEMP"):
        assert rel_l2(g.field(f), o.field(f)) <= FP64_TOL, f


def test_ordered_boundary_and_marker_passes():
    P, nrm, geom = cases.small_canyon(dx=0.011)
    prm = cases.canyon_params(geom, urbansph.default_params(), tol=1e-12)
    o, g = run_pair(P, prm, normals=nrm, dt=5e-5)
    for f in ("UX", "UY", "UZ", "PRES", "TEMP", "FBX", "FBY", "FBZ", "CONCENTRATION"):
        assert rel_l2(g.field(f), o.field(f)) <= FP64_TOL, f
