"""Neighbour-list steps with the options outside the cubic configuration
(2D): every smoothing kernel, a kernel type per term, both pressure
approximations, artificial pressure, delta-SPH and summation density, against
the FP64 oracle and against the sorted step of every step.

FP64 tolerances are those of the cubic list steps (summation order); an FP32
pair pass starts from the same FP64 positions on both sides, so the two
differ by the rounding of FP32 sums over ~20-45 neighbours for 40 steps.
"""
import copy

import numpy as np
import pytest

import oracle
from sph2d_amd import generators as G
from sph2d_amd import hip as H
from sph2d_amd import params as P

pytestmark = pytest.mark.gpu

CASES = {
    "wendland_delta_ap": dict(skf=(3, 3, 3, 3, 3), density_treatment=2, artificial_pressure=True),
    "gauss_reach_3h": dict(skf=(2, 2, 2, 2, 2), density_treatment=1),
    "desbrun_sum": dict(skf=(4, 4, 4, 4, 4), density_treatment=0),
    "mixed_approx1": dict(skf=(1, 4, 3, 1, 3), density_treatment=2, intf_sph_approximation=1, artificial_pressure=True),
    "cubic_delta": dict(skf=(1, 1, 1, 1, 1), density_treatment=2),
}


def _params(base, skf, **options):
    prm = copy.copy(base)
    (prm.density_skf, prm.intf_skf, prm.artificial_viscosity_skf, prm.average_velocity_skf,
     prm.artificial_pressure_skf) = skf
    prm.density_delta_sph_coef, prm.artificial_pressure_coef, prm.artificial_pressure_index = 0.1, 0.2, 4.0
    for k, v in options.items():
        setattr(prm, k, v)
    P.fill_in_computing_params(prm)
    P.post_fill_in_model_params(prm)
    return prm


def _start(lay, n_fluid_cut=0):
    """The layout in motion, so that particles approach and separate and some pressures are negative."""
    rng = np.random.default_rng(5)
    r, v, rho = lay.r.copy(), np.zeros_like(lay.r), lay.rho.copy()
    nf = lay.params.nfluid
    r[:nf] += rng.uniform(-0.02, 0.02, (nf, 2)) * lay.params.delta
    v[:nf] = 0.3 * np.stack([np.sin(3 * r[:nf, 1]), np.cos(5 * r[:nf, 0])], 1)
    rho[:nf] += rng.uniform(-0.5, 0.5, nf)
    return r, v, rho


def _run(prm, r, v, rho, itype, steps, precision):
    g = H.HipStep(prm, precision=precision)
    g.upload(r, v, rho, itype)
    g.step(steps)
    out = g.download()
    out["time"], out["lists"] = g.time(), g.list_stats()
    g.close()
    return out


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("precision", [H.FP64, H.FP32])
def test_general_list_steps(monkeypatch, name, precision):
    lay = G.piston_tank(delta=0.02, length=3.0, depth=0.3)
    prm = _params(lay.params, **CASES[name])
    r, v, rho = _start(lay)
    print("general lists", name, precision, "n", prm.ntotal, flush=True)
    steps = 40
    a = _run(prm, r, v, rho, lay.itype, steps, precision)
    monkeypatch.setenv("RRSPH_HIP_LIST", "0")
    b = _run(prm, r, v, rho, lay.itype, steps, precision)
    assert a["lists"]["list_steps"] > 20 and a["lists"]["builds"] >= 1 and b["lists"]["interval"] == 0
    scale_v = np.max(np.abs(b["v"]))
    if precision == H.FP64:
        ora = oracle.Oracle(prm)
        ora.set_state(r, v, rho, lay.itype, time=0.0, dt=prm.dt)
        assert ora.step(steps) == 0
        o = ora.state()
        for ref in (b, o):
            assert np.array_equal(a["itype"], ref["itype"])
            assert np.max(np.abs(a["r"] - ref["r"])) < 1e-11
            assert np.max(np.abs(a["v"] - ref["v"])) < 1e-9 * scale_v
            assert np.max(np.abs(a["rho"] - ref["rho"]) / ref["rho"]) < 1e-11
    else:
        assert np.max(np.abs(a["r"] - b["r"])) < 1e-7
        assert np.max(np.abs(a["v"] - b["v"])) < 1e-3 * scale_v
        assert np.max(np.abs(a["rho"] - b["rho"]) / b["rho"]) < 1e-5


@pytest.mark.parametrize("n", [1, 2, 63, 65, 257])
def test_general_list_steps_of_few_particles(n):
    """Partial waves and blocks: the first n particles of a jittered block alone."""
    lay = G.dam_break(delta=0.02)
    prm = _params(lay.params, **CASES["wendland_delta_ap"])
    r, v, rho = _start(lay)
    prm.ntotal, prm.nfluid, prm.nvirt = n, n, 0
    prm.nwm_particles_start = prm.nwm_particles_end = n
    a = _run(prm, r[:n], v[:n], rho[:n], lay.itype[:n], 10, H.FP64)
    ora = oracle.Oracle(prm)
    ora.set_state(r[:n], v[:n], rho[:n], lay.itype[:n], time=0.0, dt=prm.dt)
    assert ora.step(10) == 0
    o = ora.state()
    assert np.max(np.abs(a["r"] - o["r"])) < 1e-12 and np.max(np.abs(a["rho"] - o["rho"]) / o["rho"]) < 1e-12


def test_general_neighbour_overflow_stops():
    """More neighbours than max_neighbours - 1 under the consistency check: the reference's error, and the state stays
    as it was before the step."""
    lay = G.dam_break(delta=0.02)
    prm = _params(lay.params, **CASES["wendland_delta_ap"])
    prm.max_neighbours = 12
    g = H.HipStep(prm, precision=H.FP64)
    g.upload(lay.r, lay.v, lay.rho, lay.itype)
    with pytest.raises(H.RrsphError) as e:
        g.step(3)
    assert e.value.status == 3
    s = g.download()
    g.close()
    assert np.array_equal(s["r"], lay.r) and np.array_equal(s["v"], lay.v)
