"""lu (the symmetric Gauss-Seidel sweep from zero) on skewed rows against the
oracle's serial sweep: the same bits, at the edges of its range -- sides around
the wave and group sizes, either side the longer one, one line, the widest
workgroup and the sizes past it."""
import numpy as np
import pytest

from hydro_amd import capi, workloads
from hydro_amd.hydro import Hydro, stencil_solve
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


# two right-hand sides and the update of a base, as the velocity of a step has
# them: one, several and 16 waves, either side the longer one.  The bits where the
# mesh is exact (sides that are powers of two); elsewhere the bar of the FP64 path,
# as cell lengths are rounded before the sweep (a value of another row or
# right-hand side in the sweep is off by far more)
@pytest.mark.parametrize("nx,ny", [(64, 128), (128, 64), (512, 512), (1024, 1024), (1024, 2048),
                                   (2048, 1024), (60, 130), (65, 130), (130, 65), (520, 530),
                                   (530, 520)])
def test_lu_velocity(gpu, nx, ny):
    print(f"case: lu velocity {nx}x{ny}", flush=True)
    text = workloads.dam(nx, ny, solver_p="jacobi", solver_v="lu",
                         extra="set int lu_relaxed_num_iters_limit 2\n"
                               "set int num_iterations_limit 2\nset vect initial_velocity (1, 0.5)")
    o = pyoracle.Oracle(capi.parse_config(text))
    with Hydro(text) as h:
        sg, so = h.step(), o.step()
        assert sg.simple_iterations == so.simple_iterations
        for f in (capi.HG_FIELD_VELOCITY_X, capi.HG_FIELD_VELOCITY_Y):
            u, uo = h.get(f), o.get(f)
            assert np.isfinite(u).all() and np.ptp(u) > 0
            if nx & (nx - 1) or ny & (ny - 1):
                assert np.linalg.norm(u - uo) <= 1e-10 * np.linalg.norm(uo)
            else:
                assert np.array_equal(u, uo)
    o.close()
