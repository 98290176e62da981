"""lu (the symmetric Gauss-Seidel sweep from zero) on skewed rows against the
oracle's serial sweep: the same bits, at the edges of its range -- sides around
the wave and group sizes, either side the longer one, one line, the widest
workgroup and the sizes past it."""
import numpy as np
import pytest

from hydro_amd import capi
from hydro_amd.hydro import stencil_solve
from oracle import pyoracle

pytestmark = pytest.mark.gpu


def rows(nx, ny, seed):
    rng = np.random.default_rng(seed)
    n = nx * ny
    s, w, e, nn = (-rng.uniform(0.5, 1.0, n) for _ in range(4))
    i, j = np.arange(n) % nx, np.arange(n) // nx
    s[j == 0] = 0
    w[i == 0] = 0
    e[i == nx - 1] = 0
    nn[j == ny - 1] = 0
    return s, w, -(s + w + e + nn) + 0.05, e, nn, rng.normal(size=n)


SIZES = [(1, 1), (1, 9), (9, 1), (3, 7), (8, 8), (16, 16), (63, 64), (64, 63), (64, 64), (65, 66),
         (128, 20), (40, 333), (129, 500), (513, 540), (600, 513), (1024, 1030), (1026, 1025)]


@pytest.mark.parametrize("nx,ny", SIZES)
def test_lu_bitwise(gpu, nx, ny):
    print(f"case: lu {nx}x{ny}", flush=True)
    r = rows(nx, ny, nx + 2 * ny)
    x, _ = stencil_solve(nx, ny, *r, "lu", tol=0.0, max_iters=1, omega=1.0)
    xo, _ = pyoracle.stencil_solve(nx, ny, *r, capi.SOLVERS["lu"], tol=0.0, max_iters=1, omega=1.0)
    assert np.array_equal(x, xo)
