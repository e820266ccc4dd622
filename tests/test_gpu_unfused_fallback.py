"""Fused pairs of list steps (2D, continuity, constant dt, consistency check) cannot undo a step in which a particle has
too many neighbours, so they halt where some list, which holds the skin's particles too, is longer than
max_neighbours - 1; the context then goes on with unfused list steps.

Tolerances: the sides differ by summation order (FP64), and in FP32 by the rounding of FP32 sums for 40 steps (those
of test_gpu_fused_steps)."""
import copy

import numpy as np
import pytest
from scipy.spatial import cKDTree

from sph2d_amd import generators as G
from sph2d_amd import hip as H

pytestmark = pytest.mark.gpu

SKIN = 0.23  # of the cut-off, below 25,000 particles


def _most(r, radius):
    return int(cKDTree(r).query_ball_point(r, radius, return_length=True).max()) - 1


def _case(hsml_coef, max_neighbours):
    lay = G.dam_break(delta=0.02, dt=1e-4, hsml_coef=hsml_coef)
    prm = copy.copy(lay.params)
    if max_neighbours:
        prm.max_neighbours = max_neighbours
    rng = np.random.default_rng(3)
    v = np.zeros_like(lay.r)
    v[:prm.nfluid] = rng.uniform(-0.1, 0.1, (prm.nfluid, 2))
    # the reason to halt: lists longer than max_neighbours - 1, and no particle with that many neighbours
    cut = prm.cell_scale_k * prm.hsml
    assert prm.ntotal < 25000 and prm.consistency_check
    assert _most(lay.r, cut) <= prm.max_neighbours - 1 < _most(lay.r, cut * (1 + SKIN))
    return lay, prm, v


@pytest.mark.parametrize("precision", [H.FP64, H.FP32])
@pytest.mark.parametrize("hsml_coef,max_neighbours", [(1.2, 22), (2.0, 0)])
@pytest.mark.parametrize("entry", ["step", "run_until", "time_steps", "profile_steps"])
def test_lists_longer_than_max_neighbours_run_unfused(monkeypatch, entry, hsml_coef, max_neighbours, precision):
    lay, prm, v = _case(hsml_coef, max_neighbours)
    print("unfused fallback", entry, hsml_coef, prm.ntotal, precision, flush=True)
    outs = []
    for lists in ("1", "0"):
        monkeypatch.setenv("RRSPH_HIP_LIST", lists)
        g = H.HipStep(prm, precision=precision)
        g.upload(lay.r, v, lay.rho, lay.itype)
        if entry == "run_until":
            g.run_until(39.5 * prm.dt, 60)
        else:
            getattr(g, entry)(40)
        assert g.time()[2] == 40
        if lists == "1":
            assert g.list_stats()["list_steps"] > 20
        outs.append(g.download())
        g.close()
    a, b = outs
    tol = (1e-11, 1e-9, 1e-10) if precision == H.FP64 else (1e-6, 1e-3, 1e-5)
    assert np.array_equal(a["itype"], b["itype"])
    assert np.max(np.abs(a["r"] - b["r"])) < tol[0]
    assert np.max(np.abs(a["v"] - b["v"])) < tol[1] * np.max(np.abs(b["v"]))
    assert np.max(np.abs(a["rho"] - b["rho"]) / b["rho"]) < tol[2]
