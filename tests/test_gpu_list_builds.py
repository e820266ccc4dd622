"""A wave of the list build stages the union of its lanes' ranges of a column of cells and decides candidates in FP32
from a reference of the wave: tall domains (thousands of cells in a column, so a wave on the end of one column and the
start of the next spans all of it), long 3D channels and a domain of a few cells give the steps of the cell walk.

Tolerances: the two sides differ by summation order (FP64), and in FP32 by the rounding of FP32 sums for 8 steps."""
import numpy as np
import pytest

from sph2d_amd import generators as G
from sph2d_amd import hip as H

pytestmark = pytest.mark.gpu

LAYOUTS = {
    # 2D: 4000 cells a column, 41 columns; 7 x 17 cells; 3D: 530 cells in z, a handful of particles per column
    "tall": lambda: G.dam_break(delta=0.01, tank=(0.9, 95.0), column=(0.09, 60.0), jitter=0.0, dt=2e-6),
    "tiny": lambda: G.dam_break(delta=0.02, tank=(0.12, 0.3), column=(0.04, 0.1), jitter=0.0, dt=2e-5),
    "channel": lambda: G.dam_break_3d(delta=0.02, box=(0.3, 0.2, 27.0), column=(0.2, 0.1, 27.0), jitter=0.0),
}


def _run(prm, lay, r, v, precision):
    g = H.HipStep(prm, precision=precision)
    g.upload(r, v, lay.rho, lay.itype)
    g.step(8)
    out = g.download()
    out["lists"] = g.list_stats()
    g.close()
    return out


@pytest.mark.parametrize("precision", [H.FP64, H.FP32])
@pytest.mark.parametrize("name", list(LAYOUTS))
def test_lists_of_long_columns_equal_the_cell_walk(monkeypatch, name, precision):
    lay = LAYOUTS[name]()
    prm = lay.params
    rng = np.random.default_rng(11)
    nf = prm.nfluid
    r, v = lay.r.copy(), np.zeros_like(lay.r)
    r[:nf] += rng.uniform(-0.15, 0.15, (nf, prm.dim)) * prm.delta
    v[:nf] = rng.uniform(-0.2, 0.2, (nf, prm.dim))
    print("list builds:", name, "n", prm.ntotal, "precision", precision, flush=True)
    a = _run(prm, lay, r, v, precision)
    monkeypatch.setenv("RRSPH_HIP_LIST", "0")
    b = _run(prm, lay, r, v, precision)
    assert a["lists"]["builds"] > 0 and b["lists"]["interval"] == 0
    tol = (1e-12, 1e-10, 1e-11) if precision == H.FP64 else (1e-6, 1e-4, 1e-5)
    assert np.max(np.abs(a["r"] - b["r"])) < tol[0]
    assert np.max(np.abs(a["v"] - b["v"])) < tol[1] * np.max(np.abs(b["v"]))
    assert np.max(np.abs(a["rho"] - b["rho"]) / b["rho"]) < tol[2]
