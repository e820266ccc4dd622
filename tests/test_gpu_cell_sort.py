"""List builds sort by counting; the order is the radix sort's, so that every sum over a list has the same order and
whole runs are equal bit for bit, whatever order the atomics of the counting sort took."""
import numpy as np
import pytest

from sph2d_amd import generators as G
from sph2d_amd import hip as H

pytestmark = pytest.mark.gpu

LAYOUTS = {
    "one block": lambda: G.dam_break(delta=0.04, jitter=0.0, dt=5e-5),
    "few cells": lambda: G.dam_break(delta=0.02, tank=(0.12, 0.3), column=(0.04, 0.1), jitter=0.0, dt=2e-5),
    "2d": lambda: G.dam_break(delta=0.004, jitter=0.0, dt=1e-5),
    "tall": lambda: G.dam_break(delta=0.01, tank=(0.9, 95.0), column=(0.09, 60.0), jitter=0.0, dt=2e-6),
    "3d": lambda: G.dam_break_3d(delta=0.02, jitter=0.0),
}


def _run(prm, lay, r, v, t, precision):
    g = H.HipStep(prm, precision=precision)
    g.upload(r, v, lay.rho, t)
    g.step(30)
    out = g.download()
    lists = g.list_stats()
    g.close()
    return out, lists


@pytest.mark.parametrize("precision", [H.FP64, H.FP32])
@pytest.mark.parametrize("name", list(LAYOUTS))
def test_runs_equal_those_with_the_radix_sort(monkeypatch, name, precision):
    lay = LAYOUTS[name]()
    prm = lay.params
    rng = np.random.default_rng(3)
    nf = prm.nfluid
    # slots in no order at all, particles that no longer exist, and some that move enough for several builds
    order = rng.permutation(nf)
    r, v, t = lay.r.copy(), np.zeros_like(lay.r), lay.itype.copy()
    r[:nf] = r[:nf][order] + rng.uniform(-0.1, 0.1, (nf, prm.dim)) * prm.delta
    v[:nf] = rng.uniform(-1.0, 1.0, (nf, prm.dim))
    t[:nf:97] = 0
    monkeypatch.setenv("RRSPH_HIP_LIST_SKIN", "0.05")
    print("cell sort:", name, "n", prm.ntotal, "precision", precision, flush=True)
    a, qa = _run(prm, lay, r, v, t, precision)
    monkeypatch.setenv("RRSPH_HIP_BUILD_SORT", "radix")
    b, qb = _run(prm, lay, r, v, t, precision)
    print(qa, flush=True)
    assert qa["builds"] > 0 and qa == qb
    for f in ("r", "v", "rho", "p", "itype"):
        assert np.array_equal(a[f], b[f]), f
