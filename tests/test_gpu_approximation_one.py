"""Pressure approximation 1 divides by both densities, (p_i + p_j) / (rho_i rho_j)
(RRSPH_COMMON/include/InternalForce.h:53-141): a flume whose densities differ between neighbours, on sorted steps."""
import copy

import numpy as np
import pytest

import oracle
from sph2d_amd import generators as G
from sph2d_amd import hip as H

pytestmark = pytest.mark.gpu


def test_approximation_one_uses_both_densities(monkeypatch):
    lay = G.piston_tank(delta=0.02, length=3.0, depth=0.3)
    prm = copy.copy(lay.params)
    prm.intf_sph_approximation = 1
    rho = lay.rho + np.random.default_rng(3).uniform(-0.5, 0.5, len(lay.rho))
    monkeypatch.setenv("RRSPH_HIP_LIST", "0")
    g = H.HipStep(prm, precision=H.FP64)
    g.upload(lay.r, lay.v, rho, lay.itype)
    g.step(10)
    s = g.download()
    g.close()
    ora = oracle.Oracle(prm)
    ora.set_state(lay.r, lay.v, rho, lay.itype, time=0.0, dt=prm.dt)
    assert ora.step(10) == 0
    o = ora.state()
    assert np.max(np.abs(s["r"] - o["r"])) < 1e-12
    assert np.max(np.abs(s["rho"] - o["rho"]) / o["rho"]) < 1e-12
