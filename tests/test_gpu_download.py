"""Downloads of every size class: one inline copy (up to 3 MiB of staging) and pieces taken by
several threads (1 MiB each), with piece edges inside and between fields, against the uploaded arrays."""
import numpy as np
import pytest

from helpers import case, fluid, lattice, params, solid, wall
from sphnj_amd import Simulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["p64", "m32"])
@pytest.mark.parametrize("n", [1, 257, 30011, 65537, 262144, 300007])
def test_download_returns_the_upload_in_input_order(gpu, precision, n):
    """Before any step a context holds what was uploaded, sorted: the download undoes the sort.
    Doubles come back bit for bit; what M32 holds in float comes back as the float's value."""
    rng = np.random.default_rng(n)
    side = int(np.ceil(np.sqrt(n)))
    dx = 0.9 / side
    x, y = lattice(side, side, dx, 0.05, 0.05)
    pick = rng.permutation(side * side)[:n]
    f = fluid(x[pick], y[pick], u=rng.standard_normal(n), v=rng.standard_normal(n),
              rho=1000.0 + rng.standard_normal(n), p=1e3 * rng.standard_normal(n),
              phase=rng.integers(0, 2, n).astype(np.int32))
    m = min(n, 5003)
    X, Y = lattice(101, 101, 0.005, 0.2, 0.2)
    ps = rng.permutation(len(X))[:m]
    s = solid(X[ps] + 1e-4, Y[ps] - 1e-4, X[ps], Y[ps], u=np.zeros(m), v=np.zeros(m))
    w = wall(*lattice(40, 3, 0.02, 0.1, -0.06), bc=1)
    d = min(max(dx, 2e-3), 0.05)
    p = params(particle_diameter=d, smoothing_length=1.3 * d)
    sim = Simulation(case(p, f, s, w), precision)
    held = np.float32 if precision == "m32" else np.float64
    for _ in range(2):  # staging is made by the first call and kept for the second
        got = sim.download()
        for k in ("x", "y", "u", "v", "rho"):
            assert np.array_equal(got["fluid"][k], f[k]), k
        assert np.array_equal(got["fluid"]["p"], f["p"].astype(held).astype(np.float64))
        assert np.array_equal(got["fluid"]["phase"], f["phase"])
        assert (got["fluid"]["boundary_type"] == 1).all() and (got["fluid"]["near"] == 0).all()
        assert got["fluid"]["du_dx"].shape == (n, 4) and not got["fluid"]["du_dx"].any()
        for k in ("x", "y", "X", "Y"):
            assert np.array_equal(got["solid"][k], s[k]), k
        assert np.array_equal(got["solid"]["deformation"], np.tile([1.0, 0.0, 0.0, 1.0], (m, 1)))
        for k in ("x", "y", "bc"):
            assert np.array_equal(got["wall"][k], w[k]), k
    part = sim.download(species=("solid",))
    assert list(part) == ["solid"] and np.array_equal(part["solid"]["x"], s["x"])
