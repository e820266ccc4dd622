"""The 2D list passes split a particle's list over 8, 2 or 1 lanes by particle count and precision: steps on either
side of each line equal the sorted steps (which walk the cells), in both precisions and with every density option, and
an overflowing list keeps the same neighbours whatever the split.

Tolerances: the two sides differ by summation order (FP64), and in FP32 by the rounding of FP32 sums for 20 steps."""
import copy

import numpy as np
import pytest

from sph2d_amd import generators as G
from sph2d_amd import hip as H
from sph2d_amd import params as P

pytestmark = pytest.mark.gpu


def _run(prm, lay, r, v, steps, precision):
    g = H.HipStep(prm, precision=precision)
    g.upload(r, v, lay.rho, lay.itype)
    g.step(steps)
    out = g.download()
    out["time"], out["lists"] = g.time(), g.list_stats()
    g.close()
    return out


# 24.6 thousand particles (8 lanes each), 25.5 (2), 152 (2; FP32 continuity 1)
@pytest.mark.parametrize("delta", [0.02140, 0.02100, 0.00833])
@pytest.mark.parametrize("precision", [H.FP64, H.FP32])
@pytest.mark.parametrize("density", [P.DENSITY_CONTINUITY, P.DENSITY_SUMMATION])
def test_lane_splits_equal_sorted_steps(monkeypatch, delta, precision, density):
    lay = G.piston_tank(delta=delta, length=20.0, depth=0.5)
    prm = copy.copy(lay.params)
    prm.density_treatment = density
    rng = np.random.default_rng(2)
    r, v = lay.r.copy(), np.zeros_like(lay.r)
    nf = prm.nfluid
    r[:nf] += rng.uniform(-0.01, 0.01, (nf, 2)) * prm.delta
    v[:nf] = 0.2 * np.stack([np.sin(3 * r[:nf, 1]), np.cos(5 * r[:nf, 0])], 1)
    print("lanes: n", prm.ntotal, "precision", precision, "density", density, flush=True)
    a = _run(prm, lay, r, v, 20, precision)
    monkeypatch.setenv("RRSPH_HIP_LIST", "0")
    b = _run(prm, lay, r, v, 20, precision)
    assert a["lists"]["list_steps"] > 5 and b["lists"]["interval"] == 0
    tol = (1e-11, 1e-9, 1e-11) if precision == H.FP64 else (1e-6, 1e-3, 1e-5)
    assert abs(a["time"][0] - b["time"][0]) <= tol[2] * b["time"][0]
    assert np.max(np.abs(a["r"] - b["r"])) < tol[0]
    assert np.max(np.abs(a["v"] - b["v"])) < tol[1] * np.max(np.abs(b["v"]))
    assert np.max(np.abs(a["rho"] - b["rho"]) / b["rho"]) < tol[2]


@pytest.mark.parametrize("delta", [0.03, 0.0205])
def test_capped_lists_keep_the_first_neighbours(monkeypatch, delta):
    """max_neighbours below the neighbour count, unchecked: on the build step (lists in walk order, as the sorted walk
    visits) every particle keeps the same first max_neighbours - 1."""
    lay = G.piston_tank(delta=delta, length=20.0, depth=0.5)
    prm = copy.copy(lay.params)
    prm.max_neighbours, prm.consistency_check = 11, False
    for precision in (H.FP64, H.FP32):
        a = _run(prm, lay, lay.r, lay.v, 1, precision)
        monkeypatch.setenv("RRSPH_HIP_LIST", "0")
        b = _run(prm, lay, lay.r, lay.v, 1, precision)
        monkeypatch.delenv("RRSPH_HIP_LIST")
        tol = 1e-9 if precision == H.FP64 else 1e-3
        assert a["lists"]["builds"] == 1
        assert np.max(np.abs(a["v"] - b["v"])) <= tol * np.max(np.abs(b["v"]))
