"""Solves whose workgroups wait for each other inside one launch, made to give up
from the host: with a bound of 0 polls the first wait ends the kernel, and the solve is run again by kernels that do not wait.  The result is
that of those kernels bit for bit, from the start values the solve had (a warm
start among them), the next solves do not try, and with the default bound the
object goes back to one launch, on words that hold what the failed solve left."""
import numpy as np
import pytest

from hydro_amd import capi, workloads
from hydro_amd.hydro import Hydro, Hydro3, Poisson
from oracle import pyoracle

pytestmark = pytest.mark.gpu

PRESSURE = capi.HG_FIELD_PRESSURE
FIELDS = (capi.HG_FIELD_VELOCITY_X, capi.HG_FIELD_VELOCITY_Y, PRESSURE)


def poisson(nx, ny):
    rng = np.random.default_rng(nx)
    kx, ky = rng.uniform(0.5, 2.0, (ny, nx + 1)), rng.uniform(0.5, 2.0, (ny + 1, nx))
    kx[:, 0] = kx[:, -1] = 0.0
    ky[0] = ky[-1] = 0.0
    return Poisson(nx, ny, kx.reshape(-1), ky.reshape(-1)), rng.normal(size=nx * ny)


# four workgroups, 16 of one cell per thread, 64 of four
@pytest.mark.parametrize("nx,ny", [(64, 64), (128, 128), (512, 512)])
@pytest.mark.parametrize("precision", [0, 1])
def test_cg_gives_up(gpu, nx, ny, precision):
    print(f"case: cg {nx}x{ny} precision {precision}", flush=True)
    ps, rhs = poisson(nx, ny)
    args = dict(solver="cg", tol=1e-6, precision=precision)
    p0, s0 = ps.solve(rhs, **args)
    assert s0.converged and ps.wait_give_ups() == 0
    ps.set_wait_polls(0)
    p1, s1 = ps.solve(rhs, **args)  # gives up, then a launch per iteration
    assert s1.converged and ps.wait_give_ups() == 1
    p2, s2 = ps.solve(rhs, **args)  # does not try
    assert ps.wait_give_ups() == 1
    assert np.array_equal(p1, p2) and s1.iterations == s2.iterations
    ps.set_wait_polls(-1)
    p3, s3 = ps.solve(rhs, **args)
    assert ps.wait_give_ups() == 1
    assert np.array_equal(p3, p0) and s3.iterations == s0.iterations


@pytest.mark.parametrize("precision", [0, 1])
def test_cg_gives_up_without_an_iteration_cap(gpu, precision):
    """The cap of 2^31 - 1 iterations, where twice the cap and the cap plus a
    batch are past 32 bits: the solve that gave up meets its tolerance, and so do
    solves on the same words afterwards, with the bits of the first."""
    print(f"case: cg 129x128 precision {precision}, no cap", flush=True)
    ps, rhs = poisson(129, 128)
    args = dict(solver="cg", tol=1e-6, precision=precision, max_iters=2**31 - 1)
    p0, s0 = ps.solve(rhs, **args)
    for _ in range(3):
        ps.set_wait_polls(0)
        p1, s1 = ps.solve(rhs, **args)
        assert s1.converged and s1.iterations > 32
        ps.set_wait_polls(-1)
        p2, s2 = ps.solve(rhs, **args)
        assert np.array_equal(p2, p0) and s2.iterations == s0.iterations
    assert ps.wait_give_ups() == 3


def test_give_ups_are_remembered(gpu):
    print("case: cg 64x64, give-ups in a row", flush=True)
    ps, rhs = poisson(64, 64)
    args = dict(solver="cg", tol=1e-3, precision=0)
    ps.set_wait_polls(0)
    counts = []
    for _ in range(1 + 16 + 1 + 32 + 1):
        ps.solve(rhs, **args)
        counts.append(ps.wait_give_ups())
    assert counts == [1] * 17 + [2] * 33 + [3]


def test_cg_gives_up_from_a_warm_start(gpu):
    """Steps whose first solve, warm-started, gives up against steps of a context
    that does not try: the same bits, so the solve restored its start."""
    print("case: rt 64x128 cg fp64", flush=True)
    text = workloads.rt(64, 128, solver_p="cg")
    with Hydro(text) as a, Hydro(text) as b:
        for h in (a, b):
            workloads.set_rt_state(h)
            h.set_wait_polls(0)
        for n in range(5):
            a.set_wait_polls(0)
            a.step()
            b.step()
            assert a.wait_give_ups() >= n + 1
        assert b.wait_give_ups() < a.wait_give_ups()
        for f in FIELDS:
            assert np.array_equal(a.get(f), b.get(f))
        a.set_wait_polls(-1)
        n = a.wait_give_ups()
        assert a.step().pressure_converged and a.wait_give_ups() == n


def test_sor_gives_up(gpu):
    """gauss_seidel over several workgroups in a step, against the oracle."""
    print("case: dam 256x128 gauss_seidel", flush=True)
    text = workloads.dam(256, 128, extra="set int lu_relaxed_num_iters_limit 150")
    o = pyoracle.Oracle(capi.parse_config(text))
    with Hydro(text) as h:
        for polls, ups in ((-1, 0), (0, 1), (-1, 1)):
            h.set_wait_polls(polls)
            sg, so = h.step(), o.step()
            assert sg.simple_iterations == so.simple_iterations
            assert sg.pressure_solve_iters_total == so.pressure_solve_iters_total
            assert h.wait_give_ups() == ups
            for f in FIELDS:
                np.testing.assert_array_equal(h.get(f), o.get(f))
    o.close()


@pytest.mark.parametrize("nx,ny,nz", [(16, 16, 16), (40, 28, 17), (50, 40, 40)])
def test_jacobi3d_gives_up(gpu, nx, ny, nz):
    print(f"case: 3D jacobi {nx}x{ny}x{nz}", flush=True)
    text = workloads.cavity3d(nx, ny, nz)
    o = pyoracle.Oracle3(capi.parse_config3(text))
    with Hydro3(text) as h:
        for polls, ups in ((-1, 0), (0, 1), (-1, 1)):
            h.set_wait_polls(polls)
            sg, so = h.step(), o.step()
            assert sg.simple_iterations == so.simple_iterations <= 17
            assert h.wait_give_ups() == ups
            for f in (capi.HG_FIELD_VELOCITY_X, capi.HG_FIELD_VELOCITY_Z, PRESSURE):
                np.testing.assert_array_equal(h.get(f), o.get(f))
    o.close()
