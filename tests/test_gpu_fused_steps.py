"""Pairs of list steps in which the pair pass integrates too (constant dt, no wave maker): runs of them, stops inside a
pair, stale lists, lists longer than max_neighbours and particles leaving the domain give what sorted steps give.

Tolerances: the two sides differ by summation order (FP64), and in FP32 by the rounding of FP32 sums for 40 steps."""
import copy

import numpy as np
import pytest

from sph2d_amd import generators as G
from sph2d_amd import hip as H
from sph2d_amd import params as P

pytestmark = pytest.mark.gpu

# lanes per particle 8, 2, 1 in 2D (the last in FP32 with continuity), and 3D
CASES = [(2, 0.02, P.DENSITY_CONTINUITY), (2, 0.0045, P.DENSITY_CONTINUITY), (2, 0.0018, P.DENSITY_CONTINUITY),
         (2, 0.02, P.DENSITY_SUMMATION), (2, 0.0045, P.DENSITY_SUMMATION), (3, 0.025, P.DENSITY_SUMMATION)]


def _layout(dim, delta, density):
    lay = G.dam_break(delta=delta, dt=5e-5 * delta / 0.01, density_treatment=density) if dim == 2 else \
        G.dam_break_3d(delta=delta, density_treatment=density)
    rng = np.random.default_rng(3)
    nf = lay.params.nfluid
    v = np.zeros_like(lay.r)
    v[:nf] = rng.uniform(-0.3, 0.3, (nf, dim))
    return lay, copy.copy(lay.params), v


def _start(prm, lay, v, precision):
    g = H.HipStep(prm, precision=precision)
    g.upload(lay.r, v, lay.rho, lay.itype)
    return g


def _same(a, b, precision):
    tol = (1e-11, 1e-9, 1e-10) if precision == H.FP64 else (1e-6, 1e-3, 1e-5)
    assert np.array_equal(a["itype"], b["itype"])
    assert np.max(np.abs(a["r"] - b["r"])) < tol[0]
    assert np.max(np.abs(a["v"] - b["v"])) < tol[1] * np.max(np.abs(b["v"]))
    assert np.max(np.abs(a["rho"] - b["rho"]) / b["rho"]) < tol[2]


@pytest.mark.parametrize("precision", [H.FP64, H.FP32])
@pytest.mark.parametrize("dim,delta,density", CASES)
def test_runs_and_stops_equal_sorted_steps(monkeypatch, dim, delta, density, precision):
    lay, prm, v = _layout(dim, delta, density)
    print("fused:", dim, "n", prm.ntotal, density, precision, flush=True)
    outs = []
    for lists in ("1", "0"):
        monkeypatch.setenv("RRSPH_HIP_LIST", lists)
        g = _start(prm, lay, v, precision)
        g.step(11)
        states = [g.download()]
        g.run_until(14.5 * prm.dt, 40)  # stops after 15 steps, within a batch of pairs
        states.append(g.download())
        assert g.time()[2] == 15
        g.run_until(17.5 * prm.dt, 40)  # ... and after 18
        assert g.time()[2] == 18
        states.append(g.download())
        g.step(22)
        states.append(g.download())
        assert g.time()[2] == 40
        if lists == "1":
            assert g.list_stats()["list_steps"] > 8
        outs.append(states)
        g.close()
    for a, b in zip(*outs):
        _same(a, b, precision)


@pytest.mark.parametrize("precision", [H.FP64, H.FP32])
@pytest.mark.parametrize("density", [P.DENSITY_CONTINUITY, P.DENSITY_SUMMATION])
def test_stale_and_long_lists_equal_sorted_steps(monkeypatch, density, precision):
    lay, prm, v = _layout(2, 0.02, density)
    monkeypatch.setenv("RRSPH_HIP_LIST", "0")
    g = _start(prm, lay, v, precision)
    g.step(40)
    b = g.download()
    g.close()
    monkeypatch.setenv("RRSPH_HIP_LIST", "1")
    monkeypatch.setenv("RRSPH_HIP_LIST_SKIN", "0.004")  # stale before the first interval ends
    g = _start(prm, lay, v, precision)
    g.step(40)
    a = g.download()
    assert g.list_stats()["stale_halts"] > 0
    g.close()
    _same(a, b, precision)
    monkeypatch.delenv("RRSPH_HIP_LIST_SKIN")
    prm.max_neighbours = 30  # more than any particle has, fewer than some list holds
    g = _start(prm, lay, v, precision)
    g.step(40)
    a = g.download()
    g.close()
    _same(a, b, precision)


@pytest.mark.parametrize("precision", [H.FP64, H.FP32])
def test_leaving_the_domain_stops_where_sorted_steps_stop(monkeypatch, precision):
    lay, prm, v = _layout(2, 0.02, P.DENSITY_CONTINUITY)
    v[:] = 0
    top = int(np.argmax(lay.r[: prm.nfluid, 1]))
    lay.r[top] = (1.5, prm.y_maxgeom - 12.5 * 3.0 * prm.dt)
    v[top] = (0.0, 3.0)  # alone, out after the 13th step
    states = []
    for lists in ("1", "0"):
        monkeypatch.setenv("RRSPH_HIP_LIST", lists)
        g = _start(prm, lay, v, precision)
        with pytest.raises(H.RrsphError):
            g.step(40)
        states.append((g.download(), g.time()[2]))
        g.close()
    assert states[0][1] == states[1][1]
    _same(states[0][0], states[1][0], precision)
