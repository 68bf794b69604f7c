"""Shift passes that walk recorded runs, on cells barely wider than the cut-off: particles two cell
rows apart (which are no candidates of each other) come within the cut-off during the step."""
import numpy as np
import pytest

from conftest import rel_l2
from helpers import case, fluid, params
from sphnj_amd import Simulation
from sphnj_amd.sim import grid

pytestmark = pytest.mark.gpu

FIELDS = ("x", "y", "u", "v", "rho", "p")


def approaching(passes, axis_factor=1.0005):
    """Twelve groups, four cells apart and from the grid's left edge on: 1 to 4 particles of a sub-column, the last just below the top
    of cell row cy, and 1 to 3 of the same sub-column just above the bottom of row cy + 2.  They are
    1.0021 cut-offs apart at the hash and 0.9941 after the fluid's update; each path is 0.004 cut-offs,
    less than half the runs' skin.  The lower particle's runs end with itself, after 1 to 4 entries."""
    p = params(gravity=0.0, shift_per_step=passes)
    rc = 3.0 * p.smoothing_length
    p.domain_xmin = p.cell_xmin
    p.cell_xmax = p.cell_xmin + 18 * axis_factor * rc
    p.cell_ymax = p.cell_ymin + 18 * axis_factor * rc
    nx, ny, cdx, cdy = grid(p)
    assert nx == 18 and ny == 18 and 1.0 < cdy / rc < 1.01
    x, y, v, low = [], [], [], []
    speed = 0.004 * rc / p.dt
    for k in range(12):
        below, above = 1 + k % 4, 1 + k // 4
        cx, cy = 4 * (k % 4), 4 + 4 * (k // 4)
        x0 = p.cell_xmin + (cx + 0.25) * cdx
        top, bottom = p.cell_ymin + (cy + 1) * cdy, p.cell_ymin + (cy + 2) * cdy
        for q in range(below - 1):  # at rest, in the run of the lower particle
            x.append(x0 + 0.01 * rc * q)
            y.append(top - (0.75 - 0.2 * q) * cdy)
            v.append(0.0)
        low.append(len(x))
        x.append(x0)
        y.append(top - 0.0008 * rc)
        v.append(speed)
        for q in range(above):
            x.append(x0 + 0.02 * rc * q)
            y.append(bottom + 0.0008 * rc)
            v.append(-speed)
    n = len(x)
    c = case(p, fluid(x, y, v=v, rho=1.0, phase=np.ones(n, np.int32)))  # gas: every particle shifts
    return c, np.array(low), rc


@pytest.mark.parametrize("precision", ["p64", "m32"])
@pytest.mark.parametrize("passes", [2, 10])
@pytest.mark.parametrize("pair_block", [256, 128])
def test_runs_leave_out_what_is_past_the_3x3_cells(gpu, oracle_mod, precision, passes, pair_block):
    """Runs recorded by the pair kernel (equal block sizes) or by the first shift pass give the bits of
    full windows (mode 0), and of runs recorded and not walked (mode 2); P64 is the oracle's to 1e-9."""
    c, low, rc = approaching(passes)
    got = {}
    for mode in (0, 1, 2):
        sim = Simulation(c, precision, shift_runs=mode)
        sim.set_block(0, pair_block)
        sim.set_block(1, 256)
        sim.step(1)
        assert sim.status() == 0
        got[mode] = sim.download()["fluid"]
    # the premise: each lower particle and the next one up are within the cut-off now
    d = np.hypot(got[0]["x"][low + 1] - got[0]["x"][low], got[0]["y"][low + 1] - got[0]["y"][low])
    assert (d < rc).all()
    for mode in (1, 2):
        for k, a in got[0].items():
            assert np.array_equal(a, got[mode][k]), (mode, k)
    if precision == "p64":
        ora = oracle_mod.Oracle(c)
        ora.step(1)
        want = ora.download()["fluid"]
        for k in FIELDS:
            assert rel_l2(got[1][k], want[k]) <= 1e-9, k
