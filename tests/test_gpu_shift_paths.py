"""The flags that say whether a cell column's lanes have moved further than half the runs' skin:
paths below half of it, between half and all of it, past it, and none at all beside them."""
import numpy as np
import pytest

from helpers import case, fluid, lattice, params, wall
from sphnj_amd import Simulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["p64", "m32"])
@pytest.mark.parametrize("share", [0.002, 0.0095, 0.0105, 0.0195, 0.03])
@pytest.mark.parametrize("passes", [2, 3, 6])
def test_runs_and_windows_agree_at_the_skin(gpu, precision, share, passes):
    """One cell column of a block at rest moves by `share` of the cut-off in a step (the runs' skin
    is 0.02 of it): its tiles and those beside it take the tested path, the others walk their runs
    unseen.  Runs (mode 1), full windows (0) and recorded but never walked runs (2) give the same
    bits in every field."""
    p = params(shift_per_step=passes)
    rc = 3.0 * p.smoothing_length
    x, y = lattice(40, 40, 0.02, 0.1, 0.1)
    rng = np.random.default_rng(5)
    x = x + 0.001 * rng.standard_normal(len(x))
    y = y + 0.001 * rng.standard_normal(len(y))
    band = (x > 0.45) & (x < 0.52)
    v = np.where(band, share * rc / p.dt, 0.0)
    c = case(p, fluid(x, y, v=v, p=50.0 * (1.0 - y)), None, wall(*lattice(44, 3, 0.02, 0.06, 0.03)))
    got = {}
    for mode in (0, 1, 2):
        sim = Simulation(c, precision, shift_runs=mode)
        sim.step(3)
        got[mode] = sim.download()["fluid"]
    for mode in (1, 2):
        for k, a in got[0].items():
            assert np.array_equal(a, got[mode][k]), (mode, k)


@pytest.mark.parametrize("precision", ["p64", "m32"])
@pytest.mark.parametrize("spacing", [0.03, 0.02, 0.013, 0.008, 0.005])
def test_listed_walls_give_the_bits_of_all_walls(gpu, precision, spacing):
    """A block of fluid in a corner of walls from sparse to too many for a lane's list (47 walls) and
    for a tile's (255): the passes that take the listed walls, all walls (mode 0) and a recording
    that lists none (mode 2) give the same bits in every field."""
    p = params(shift_per_step=4)
    x, y = lattice(30, 30, 0.02, 0.1, 0.1)
    rng = np.random.default_rng(9)
    x, y = x + 0.002 * rng.standard_normal(len(x)), y + 0.002 * rng.standard_normal(len(y))
    n, m = int(0.7 / spacing), max(2, int(0.06 / spacing))
    bx, by = lattice(n, m, spacing, 0.04, 0.09 - m * spacing)
    lx, ly = lattice(m, n, spacing, 0.09 - m * spacing, 0.1)
    c = case(p, fluid(x, y, u=-0.3, v=-0.2, p=50.0 * (1.0 - y)), None,
             wall(np.concatenate([bx, lx]), np.concatenate([by, ly])))
    got = {}
    for mode in (0, 1, 2):
        sim = Simulation(c, precision, shift_runs=mode)
        sim.step(3)
        got[mode] = sim.download()["fluid"]
    for mode in (1, 2):
        for k, a in got[0].items():
            assert np.array_equal(a, got[mode][k]), (mode, k)
