"""The gradient of the cubic spline for close pairs in the FP32 list passes: the density rate of isolated pairs against
the closed form m F (v_i - v_j) . (r_i - r_j) with F = f / h^2 (3/2 q - 2), q <= 1 (SmoothingKernel.h:14-55,
Density.h:88-113).

Positions lie on FP32 values from the origin of one cell, so that r_i - r_j is exact in FP32 up to its last bit, and
the velocity difference points along it, so that nothing in the dot product cancels.  With u = 2^-24 and q <= 0.4:
|r|^2 within 2 u and |r| within 4 u, F within (u + 0.3 * 6 u) / 0.7 + u = 5 u, the dot product within 4 u (differences,
products, sum), the products with F and the mass factor (a rounded constant) 3 u, the sum over lanes exact: 12 u."""
import copy

import numpy as np
import pytest

from sph2d_amd import generators as G
from sph2d_amd import hip as H
from sph2d_amd import params as P

pytestmark = pytest.mark.gpu


def _pairs(dim):
    lay = G.dam_break() if dim == 2 else G.dam_break_3d(density_treatment=P.DENSITY_CONTINUITY)
    prm = copy.copy(lay.params)
    cell, h = prm.cell_scale_k * prm.hsml, prm.hsml
    lo = np.array([prm.x_mingeom, prm.y_mingeom, prm.z_mingeom][:dim])
    hi = np.array([prm.x_maxgeom, prm.y_maxgeom, prm.z_maxgeom][:dim])
    rng = np.random.default_rng(17)
    cells = np.stack(np.meshgrid(*[np.arange(2, int((b - a) / cell) - 2, 4) for a, b in zip(lo, hi)], indexing="ij"), -1)
    cells = cells.reshape(-1, dim)
    n = len(cells)
    q = np.exp(rng.uniform(np.log(0.02), np.log(0.4), n))
    e = rng.normal(size=(n, dim))
    e /= np.linalg.norm(e, axis=1)[:, None]
    origin = lo + cells * cell
    a = rng.uniform(0.35, 0.65, (n, dim)) * cell
    f32 = lambda x: np.asarray(x, np.float32).astype(np.float64)
    r = np.concatenate([origin + f32(a), origin + f32(a + e * (q * h)[:, None])])
    v = np.concatenate([np.zeros((n, dim)), f32(-0.2 * e)])
    prm.ntotal = prm.nfluid = 2 * n
    prm.nvirt = 0
    prm.nwm_particles_start = prm.nwm_particles_end = 2 * n
    return prm, r, v, n


@pytest.mark.parametrize("dim", [2, 3])
def test_density_rate_of_close_pairs(dim):
    prm, r, v, n = _pairs(dim)
    g = H.HipStep(prm, precision=H.FP32)
    g.set_export_fields(True)
    g.upload(r, v, np.full(2 * n, prm.rho0), np.full(2 * n, P.TYPE_WATER, np.int32))
    g.step(1)
    assert g.list_stats()["builds"] == 1
    got = g.fields()["drho"]
    g.close()
    h = prm.hsml
    f = 15 / (7 * prm.pi * h * h) if dim == 2 else 3 / (2 * prm.pi * h ** 3)
    e, dv = r[n:] - r[:n], v[n:] - v[:n]
    q = np.linalg.norm(e, axis=1) / h
    want = prm.mass * f / h ** 2 * (1.5 * q - 2) * np.sum(dv * e, axis=1)
    err = np.abs(got.reshape(2, n) / want - 1).max()
    print("close pairs", dim, "pairs", n, "q", q.min(), q.max(), "error / u", err * 2 ** 24, flush=True)
    assert q.min() < 0.03 and q.max() < 0.41
    assert err < 12 * 2.0 ** -24
