"""gauss_seidel (lexicographic SOR) with many sweeps in flight against the
oracle's serial sweeps: the same bits and the same sweep count at the edges
of its range -- sides around the thread and ring limits, either side the
longer one, stops by the tolerance at the first, a middle and the last sweep,
and grids that keep the one-sweep kernel."""
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


SIZES = [(1, 1), (3, 7), (1, 8), (8, 8), (9, 8), (2, 50), (16, 16), (31, 33), (64, 64), (65, 64),
         (57, 64), (128, 20), (40, 333), (1024, 12), (9, 1030), (513, 600), (1030, 1027), (64, 256),
         (256, 65), (217, 333), (30, 700)]


@pytest.mark.parametrize("nx,ny", SIZES)
@pytest.mark.parametrize("tol,limit", [(0.0, 0), (0.0, 7), (1e9, 5), (1e-2, 60)])
def test_sor_bitwise(gpu, nx, ny, tol, limit):
    if nx * ny > 100000 and limit > 7:
        limit = 9
    print(f"case: SOR {nx}x{ny} tol {tol} limit {limit}", flush=True)
    r = rows(nx, ny, 3)
    args = dict(tol=tol, max_iters=limit, omega=1.7)
    x, st = stencil_solve(nx, ny, *r, "gauss_seidel", **args)
    xo, so = pyoracle.stencil_solve(nx, ny, *r, capi.SOLVERS["gauss_seidel"], **args)
    assert st.iterations == so.iterations
    assert np.array_equal(x, xo)


# a limit that only says "stop by the tolerance": its last step is past 32 bits
# on the grids that run over several workgroups (here 4, 11 and 21 of them)
@pytest.mark.parametrize("nx,ny", [(64, 256), (333, 217), (512, 512), (64, 64)])
@pytest.mark.parametrize("limit", [10**9, 2**31 - 1])
def test_sor_without_a_limit(gpu, nx, ny, limit):
    print(f"case: SOR {nx}x{ny} limit {limit}", flush=True)
    r = rows(nx, ny, 5)
    args = dict(tol=3e-2, omega=1.7)
    x, st = stencil_solve(nx, ny, *r, "gauss_seidel", max_iters=limit, **args)
    xo, so = pyoracle.stencil_solve(nx, ny, *r, capi.SOLVERS["gauss_seidel"], max_iters=1000,
                                    **args)
    assert 2 < so.iterations < 1000 and st.iterations == so.iterations
    assert np.array_equal(x, xo)
