"""The fluid force on solids over the 3x3 cells' sub-column spans: cut off at the grid's edges, with
empty sub-columns, with none or one fluid particle, and with more than a round of the lanes."""
import numpy as np
import pytest

from helpers import case, fluid, params, solid
from sphnj_amd import Simulation

pytestmark = pytest.mark.gpu


# P64: sums of some hundred FP64 terms in another order, 1e-16 each.  M32: float terms, each with
# the rounding of a position in its cell (6e-8 of it) and of w' and 1/r: the float32 bar, 2e-5.
@pytest.mark.parametrize("precision,tol", [("p64", 1e-12), ("m32", 2e-5)])
@pytest.mark.parametrize("per_cell", [0.3, 3, 11, 40])
@pytest.mark.parametrize("persistent", [False, True])
def test_fluid_force_on_solids_matches_the_oracle(gpu, oracle_mod, precision, tol, per_cell, persistent):
    p = params(gravity=0.0, dt=1e-7, shift_per_step=0)
    rc = 3.0 * p.smoothing_length
    rng = np.random.default_rng(int(10 * per_cell) + 1)
    lo, hi = p.cell_xmin + 1e-6, p.cell_xmax - 1e-6
    # solids in the corners, on the edges, in the middle and in a corner without fluid
    a = np.array([lo, lo + 0.4 * rc, 0.43, 0.5, hi - 0.4 * rc, hi])
    sx, sy = (v.ravel() for v in np.meshgrid(a, a, indexing="ij"))
    n = int(per_cell * ((hi - lo) / rc) ** 2)
    x, y = rng.uniform(lo, hi, n), rng.uniform(lo, hi, n)
    # no fluid in one corner and in a band of columns, none closer to a solid than a tenth of rc
    keep = ~((x > 0.9) & (y > 0.9)) & ~((x > 0.45) & (x < 0.45 + 0.6 * rc))
    r2 = (x[:, None] - sx) ** 2 + (y[:, None] - sy) ** 2
    keep &= r2.min(1) > (0.1 * rc) ** 2
    x, y = x[keep], y[keep]
    m = len(x)
    c = case(p, fluid(x, y, u=rng.normal(0, 3, m), v=rng.normal(0, 3, m), p=rng.uniform(0, 900, m)),
             solid(sx, sy, u=rng.normal(0, 3, len(sx)), v=rng.normal(0, 3, len(sx))))
    sim, ora = Simulation(c, precision, persistent_solid=persistent), oracle_mod.Oracle(c)
    for st in ("cells", "couple", "solid"):
        sim.stage(st)
        ora.stage(st)
    got, want = sim.download()["solid"]["couple_dudt"], ora.download()["solid"]["couple_dudt"]
    assert np.count_nonzero(want) > 0
    assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want)
    assert np.array_equal(got == 0, want == 0)


# The fluid's increments of velocity and density: P64 to the 1e-9 bar, M32 to 1e-4 (sums of float
# terms of both signs, each to a few 1e-7, that cancel to some tenth of the largest).
@pytest.mark.parametrize("precision,tol", [("p64", 1e-9), ("m32", 1e-4)])
@pytest.mark.parametrize("solids_per_cell", [0.2, 2, 9, 30])
def test_solid_terms_of_the_fluid_match_the_oracle(gpu, oracle_mod, precision, tol, solids_per_cell):
    p = params(gravity=0.0, dt=1e-5, shift_per_step=0)
    rc = 3.0 * p.smoothing_length
    rng = np.random.default_rng(int(10 * solids_per_cell) + 2)
    lo, hi = p.domain_xmin + 1e-6, p.domain_xmax - 1e-6
    n = int(solids_per_cell * ((hi - lo) / rc) ** 2)
    sx, sy = rng.uniform(lo, hi, n), rng.uniform(lo, hi, n)
    keep = ~((sx > 0.7) & (sy > 0.7)) & ~((sx > 0.35) & (sx < 0.35 + 1.5 * rc))  # cells without any
    sx, sy = sx[keep], sy[keep]
    x, y = rng.uniform(lo, hi, 600), rng.uniform(lo, hi, 600)
    far = ((x[:, None] - sx) ** 2 + (y[:, None] - sy) ** 2).min(1) > (0.05 * rc) ** 2
    x, y = x[far], y[far]
    m = len(x)
    u, v = rng.normal(0, 3, m), rng.normal(0, 3, m)
    c = case(p, fluid(x, y, u=u, v=v, p=rng.uniform(0, 900, m)),
             solid(sx, sy, u=rng.normal(0, 3, len(sx)), v=rng.normal(0, 3, len(sx))))
    sim, ora = Simulation(c, precision), oracle_mod.Oracle(c)
    for st in ("cells", "couple", "wall", "fluid"):
        sim.stage(st)
        ora.stage(st)
    a, b = sim.download()["fluid"], ora.download()["fluid"]
    for f, f0 in (("u", u), ("v", v), ("rho", 1000.0)):
        want = b[f] - f0
        assert np.linalg.norm((a[f] - f0) - want) <= tol * np.linalg.norm(want), f
