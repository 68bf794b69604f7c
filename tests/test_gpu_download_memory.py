"""Downloads larger than the bounded device staging: gathered in rounds, with the memory they keep."""
import ctypes

import numpy as np
import pytest

from helpers import case, fluid, lattice, params, solid, wall
from sphnj_amd import Simulation

pytestmark = pytest.mark.gpu


def free_memory():
    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("precision", ["p64", "m32"])
def test_download_takes_bounded_device_memory(gpu, precision):
    """2.2 M fluid particles, 30 k solids and 20 k walls (about 210 MB in P64, 160 in M32) come back in
    input order through at most 64 MiB of staging (2 MiB of slack: the allocator's granularity), on the
    first call and, with nothing more taken, on the second."""
    rng = np.random.default_rng(3)
    n, dx = 1484, 6.0e-4
    x, y = lattice(n, n, dx, 0.05, 0.05)
    o = rng.permutation(n * n)
    m = n * n
    f = fluid(x[o], y[o], u=rng.standard_normal(m), v=rng.standard_normal(m), rho=1000.0 + rng.standard_normal(m),
              p=1e3 * rng.standard_normal(m), phase=rng.integers(0, 2, m).astype(np.int32))
    X, Y = lattice(300, 100, 2e-3, 0.2, 0.2)
    o = rng.permutation(len(X))
    s = solid(X[o] + 1e-5, Y[o], X[o], Y[o])
    w = wall(*lattice(2000, 10, dx, 0.02, 0.02), bc=1)
    p = params(particle_diameter=2e-3, smoothing_length=2.6e-3)
    sim = Simulation(case(p, f, s, w), precision)
    held = np.float32 if precision == "m32" else np.float64
    before = free_memory()
    for _ in range(2):
        got = sim.download()
        assert before - free_memory() <= (64 << 20) + (2 << 20)
        for k in ("x", "y", "u", "v", "rho"):
            assert np.array_equal(got["fluid"][k], f[k]), k
        assert np.array_equal(got["fluid"]["p"], f["p"].astype(held).astype(np.float64))
        assert np.array_equal(got["fluid"]["phase"], f["phase"])
        assert got["fluid"]["du_dx"].shape == (m, 4) and not got["fluid"]["du_dx"].any()
        for k in ("x", "y", "X", "Y"):
            assert np.array_equal(got["solid"][k], s[k]), k
        for k in ("x", "y", "bc"):
            assert np.array_equal(got["wall"][k], w[k]), k


def test_wall_lists_take_no_memory_without_walls(gpu):
    """The P64 shift passes' wall lists (48 bytes a fluid particle) belong to contexts with walls only:
    a context without takes that much less than the same with one wall (4 MiB of slack)."""
    n = 1024
    x, y = lattice(n, n, 8.5e-4, 0.05, 0.05)
    p = params(particle_diameter=8.5e-4, smoothing_length=1.105e-3)
    taken = []
    Simulation(case(p, fluid(x, y), None, wall([0.02], [0.02])), "p64").close()  # (loads the kernels)
    for w in (None, wall([0.02], [0.02])):
        before = free_memory()
        sim = Simulation(case(p, fluid(x, y), None, w), "p64")
        taken.append(before - free_memory())
        sim.close()
    assert taken[1] - taken[0] >= 48 * n * n - (4 << 20)
