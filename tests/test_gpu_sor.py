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


# stops within and just past the sweeps that one workgroup runs ahead of the
# pipeline: one and several waves, part of a wave, lines much longer than wide
@pytest.mark.parametrize("nx,ny", [(1, 8), (8, 8), (9, 8), (31, 33), (64, 64), (65, 64), (40, 333),
                                   (9, 1030), (128, 128), (217, 333), (513, 600), (1024, 12)])
@pytest.mark.parametrize("sweep", [0, 1, 2, 3, 4])
def test_sor_stops_in_its_first_sweeps(gpu, nx, ny, sweep):
    print(f"case: SOR {nx}x{ny} stops in sweep {sweep}", flush=True)
    r = rows(nx, ny, nx)
    sid = capi.SOLVERS["gauss_seidel"]
    args = dict(omega=1.2)
    tol = pyoracle.stencil_solve(nx, ny, *r, sid, tol=0.0, max_iters=sweep, **args)[1].final_diff
    x, st = stencil_solve(nx, ny, *r, sid, tol=tol, max_iters=1000, **args)
    xo, so = pyoracle.stencil_solve(nx, ny, *r, sid, tol=tol, max_iters=1000, **args)
    assert st.iterations == so.iterations <= sweep and st.final_diff == so.final_diff
    assert np.array_equal(x, xo)


# values that are not finite spread as in the serial sweeps, and constants of -0
# (the signs of zeros included); stops at once, after two and after nine sweeps
@pytest.mark.parametrize("nx,ny", [(9, 8), (64, 65), (217, 333), (3, 7)])
@pytest.mark.parametrize("value", [np.nan, np.inf, -0.0])
@pytest.mark.parametrize("limit", [0, 1, 8])
def test_sor_special_values(gpu, nx, ny, value, limit):
    print(f"case: SOR {nx}x{ny} {value} limit {limit}", flush=True)
    s, w, c, e, n, k = rows(nx, ny, 11)
    if value == 0:
        k = np.full(nx * ny, value)
    else:
        k[nx * ny // 2] = value
    args = dict(tol=0.0, max_iters=limit, omega=1.3)
    x, st = stencil_solve(nx, ny, s, w, c, e, n, k, "gauss_seidel", **args)
    xo, so = pyoracle.stencil_solve(nx, ny, s, w, c, e, n, k, capi.SOLVERS["gauss_seidel"], **args)
    assert st.iterations == so.iterations
    assert np.array_equal(x, xo, equal_nan=True)
    assert np.array_equal(np.signbit(x[~np.isnan(x)]), np.signbit(xo[~np.isnan(xo)]))
