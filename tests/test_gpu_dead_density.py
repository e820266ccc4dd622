"""Summation density of particles that no longer exist (uploaded so, removed by FIX, or a wall that disappears), in list
steps and sorted ones: the oracle's, which is their own term, renormalised by itself; and nothing of them reaches the
sums of particles whose lists still name them."""
import copy

import numpy as np
import pytest

import oracle
from sph2d_amd import generators as G
from sph2d_amd import hip as H
from sph2d_amd import params as P

pytestmark = pytest.mark.gpu


def _case(dim, skf, dt_method, every, how):
    lay = G.dam_break(delta=0.03, tank=(1.5, 0.8), column=(0.6, 0.3), density_treatment=P.DENSITY_SUMMATION, dt=1e-4) \
        if dim == 2 else G.dam_break_3d(delta=0.05)
    prm = copy.copy(lay.params)
    if skf != 1:
        prm.density_skf = prm.intf_skf = prm.artificial_viscosity_skf = prm.average_velocity_skf = skf
    if every:
        prm.density_normalization, prm.density_normalization_every = 1, every
    if dt_method == 2:
        prm.dt_correction_method, prm.dt_dynamic_mode, prm.CFL_coef = 2, 1, 0.1
    nf = prm.nfluid
    r, v, rho, itype = lay.r.copy(), np.zeros_like(lay.r), lay.rho.copy(), lay.itype.copy()
    rng = np.random.default_rng(4)
    v[:nf] = rng.uniform(-0.2, 0.2, (nf, dim))
    itype[[3, 17, nf + 5]] = 0
    if how == "wall":  # the left wall disappears while the lists name it
        left = (itype < 0) & (r[:, 0] <= 1e-9) & (r[:, 1] > 0)
        o = np.concatenate([np.nonzero(~left)[0], np.nonzero(left)[0]])
        r, v, rho, itype = r[o], v[o], rho[o], itype[o]
        prm.nwm, prm.boundary_motion, prm.nwm_time_start = P.NWM_METHOD_WALL_DISAPPEAR, True, 12.5 * prm.dt
        prm.nwm_particles_start, prm.nwm_particles_end = prm.ntotal - int(left.sum()), prm.ntotal
    else:  # FIX: two particles above the column leave through the top
        prm.consistency_treatment = P.CONSISTENCY_FIX
        for k, i in enumerate((30, 31)):
            r[i, :2] = 0.7 + 0.3 * k, prm.y_maxgeom - 0.002 * (k + 1)
            v[i] = 0
            v[i, 1] = 2.0
    P.fill_in_computing_params(prm)
    P.post_fill_in_model_params(prm)
    return prm, r, v, rho, itype


# the fused steps take a constant dt without a wave maker, the others an integrator of their own
@pytest.mark.parametrize("lists", ["1", "0"])
@pytest.mark.parametrize("every", [0, 1, 3])
@pytest.mark.parametrize("dim,skf,dt_method,how", [(2, 1, 0, "wall"), (2, 1, 0, "fix"), (2, 3, 0, "wall"), (2, 3, 2, "fix"),
                                                   (2, 1, 2, "fix"), (3, 1, 0, "wall"), (3, 1, 0, "fix"), (3, 1, 2, "fix")])
def test_dead_particles_density(monkeypatch, dim, skf, dt_method, how, every, lists):
    monkeypatch.setenv("RRSPH_HIP_LIST", lists)
    prm, r, v, rho, itype = _case(dim, skf, dt_method, every, how)
    ora = oracle.Oracle(prm)
    ora.set_state(r, v, rho, itype, time=0.0, dt=prm.dt)
    g = H.HipStep(prm, precision=H.FP64)
    g.upload(r, v, rho, itype)
    died = 0
    for steps in (1, 9, 12, 18):
        g.step(steps)
        assert ora.step(steps) == 0
        a, b = g.download(), ora.state()
        assert np.array_equal(a["itype"], b["itype"])
        died = int(np.sum(b["itype"] == 0)) - 3
        # 40 steps of sums in other orders, 1e-13 a step at most of the largest value; dp = c^2 drho
        for f, scale in (("r", 1.0), ("v", 1.0), ("rho", prm.rho0), ("p", prm.eos_c_sqr * prm.rho0)):
            assert np.max(np.abs(a[f] - b[f])) <= 1e-11 * scale, (f, steps)
    assert died > 0
    if lists == "1":
        assert g.list_stats()["list_steps"] > 10
    g.close()
