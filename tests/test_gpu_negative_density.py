"""A flow that is torn apart predicts negative densities.  With the options outside the cubic configuration list steps
give then what the cell walk and the oracle give: the sign stays in the viscosity and XSPH terms."""
import copy

import numpy as np
import pytest

import oracle
from sph2d_amd import generators as G
from sph2d_amd import hip as H
from sph2d_amd import params as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("approximation", [1, 2])
@pytest.mark.parametrize("skf", [3, 4])
def test_negative_predicted_densities(monkeypatch, skf, approximation):
    lay = G.dam_break(delta=0.03, tank=(1.5, 0.8), column=(0.6, 0.3), dt=1e-5)
    prm = copy.copy(lay.params)
    prm.density_skf = prm.intf_skf = prm.artificial_viscosity_skf = prm.average_velocity_skf = skf
    prm.intf_sph_approximation = approximation
    prm.consistency_check = False
    P.fill_in_computing_params(prm)
    P.post_fill_in_model_params(prm)
    nf = prm.nfluid
    c = lay.r[:nf].mean(axis=0)
    v = np.zeros_like(lay.r)
    v[:nf] = 3.0 * (lay.r[:nf] - c)
    rho = lay.rho.copy()
    rho[np.nonzero(np.linalg.norm(lay.r[:nf] - c, axis=1) < 0.08)[0][::2]] = -200.0
    out = []
    for lists in ("1", "0"):
        monkeypatch.setenv("RRSPH_HIP_LIST", lists)
        g = H.HipStep(prm, precision=H.FP64)
        g.upload(lay.r, v, rho, lay.itype)
        g.step(3)
        out.append(g.download())
        built = g.list_stats()
        assert (built["list_steps"] > 0) == (lists == "1"), built
        g.close()
    ora = oracle.Oracle(prm)
    ora.set_state(lay.r, v, rho, lay.itype, time=0.0, dt=prm.dt)
    assert ora.step(3) == 0
    s = ora.state()
    assert np.sum(s["rho"] + ora.fields()["drho"] * prm.dt / 2 < 0) >= 3
    for a in out:
        for k in ("r", "v", "rho"):
            assert np.max(np.abs(a[k] - s[k])) <= 1e-9 * np.max(np.abs(s[k])), k
