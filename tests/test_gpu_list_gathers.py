"""The FP64 list passes fetch the records of a wave's entries together: particles in a wave that is partly beyond the
particle count, lists of every length beside lists of none (isolated and non-existent particles), and both densities
give the steps of the cell walk.

Tolerances: the two sides differ by the order of FP64 sums of ~100 terms over 6 steps."""
import copy

import numpy as np
import pytest

from sph2d_amd import generators as G
from sph2d_amd import hip as H
from sph2d_amd import params as P

pytestmark = pytest.mark.gpu


def _run(prm, lay, r, v, itype, steps):
    g = H.HipStep(prm, precision=H.FP64)
    g.upload(r, v, lay.rho, itype)
    g.step(steps)
    out = g.download()
    out["lists"] = g.list_stats()
    g.close()
    return out


@pytest.mark.parametrize("dim,delta", [(2, 0.0215), (2, 0.04), (3, 0.03), (3, 0.0285)])
@pytest.mark.parametrize("density", [P.DENSITY_CONTINUITY, P.DENSITY_SUMMATION])
def test_gathered_records_equal_the_cell_walk(monkeypatch, dim, delta, density):
    lay = G.dam_break(delta=delta, jitter=0.0) if dim == 2 else G.dam_break_3d(delta=delta, jitter=0.0)
    prm = copy.copy(lay.params)
    prm.density_treatment = density
    prm.consistency_treatment = P.CONSISTENCY_FIX
    rng = np.random.default_rng(5)
    nf = prm.nfluid
    r, v, itype = lay.r.copy(), np.zeros_like(lay.r), lay.itype.copy()
    v[:nf] = rng.uniform(-0.3, 0.3, (nf, dim))
    itype[rng.choice(nf, nf // 6, replace=False)] = 0  # non-existent from the start, anywhere in a wave
    hole = rng.choice(nf, 5, replace=False)  # alone in the air: empty lists
    r[hole, 0] = np.linspace(0.6, 0.95, 5) * prm.x_maxgeom
    r[hole, dim - 1] = 0.8 * (prm.y_maxgeom if dim == 2 else prm.z_maxgeom)
    print("gathers: dim", dim, "n", prm.ntotal, prm.ntotal % 64, "density", density, flush=True)
    a = _run(prm, lay, r, v, itype, 6)
    monkeypatch.setenv("RRSPH_HIP_LIST", "0")
    b = _run(prm, lay, r, v, itype, 6)
    assert a["lists"]["builds"] > 0 and b["lists"]["interval"] == 0
    assert np.array_equal(a["itype"], b["itype"])
    alive = a["itype"] != 0
    assert np.all(np.isfinite(a["r"][alive])) and np.all(np.isfinite(a["rho"][alive]))
    assert np.max(np.abs(a["r"][alive] - b["r"][alive])) < 1e-12
    assert np.max(np.abs(a["v"][alive] - b["v"][alive])) < 1e-9 * np.max(np.abs(b["v"][alive]))
    assert np.max(np.abs(a["rho"][alive] - b["rho"][alive]) / b["rho"][alive]) < 1e-11
