"""rrsph_hip_profile_steps takes the steps that rrsph_hip_step takes: pairs of fused ones where the context fuses (constant
dt, no wave maker), whose pair pass integrates."""
import numpy as np
import pytest

from sph2d_amd import generators as G
from sph2d_amd import hip as H
from sph2d_amd import params as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [H.FP64, H.FP32])
@pytest.mark.parametrize("dim,density", [(2, P.DENSITY_CONTINUITY), (2, P.DENSITY_SUMMATION), (3, P.DENSITY_SUMMATION)])
def test_profiled_steps_are_the_fused_ones(dim, density, precision):
    lay = G.dam_break(delta=0.02, density_treatment=density) if dim == 2 else G.dam_break_3d(delta=0.05)
    out = []
    for profiled in (True, False):
        g = H.HipStep(lay.params, precision=precision)
        g.upload(lay.r, lay.v, lay.rho, lay.itype)
        g.step(1)  # the build
        if profiled:
            per_kernel, total = g.profile_steps(6)
            assert per_kernel["pair_kernel"] > 0 and per_kernel["integrate_kernel"] == 0 and total > 0
            per_kernel, _ = g.profile_steps(27)  # an odd number: the last one alone
            assert per_kernel["integrate_kernel"] > 0
        else:
            g.step(33)
        assert g.time()[2] == 34
        out.append(g.download())
        g.close()
    a, b = out
    # the schedules of builds may differ, and with them the order of sums
    tol = (1e-11, 1e-9, 1e-10) if precision == H.FP64 else (1e-6, 1e-3, 1e-5)
    assert np.max(np.abs(a["r"] - b["r"])) < tol[0]
    assert np.max(np.abs(a["v"] - b["v"])) < tol[1] * np.max(np.abs(b["v"]))
    assert np.max(np.abs(a["rho"] - b["rho"]) / b["rho"]) < tol[2]
