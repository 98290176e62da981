"""Pressure Poisson solves on the GPU (variable coefficients, density ratio
1000), judged by the true FP64 residual computed here in numpy."""
import numpy as np
import pytest

from hydro_amd import workloads
from hydro_amd.hydro import Poisson
from oracle import pyoracle

pytestmark = pytest.mark.gpu


def apply(kx, ky, p, nx, ny):
    kx = kx.reshape(ny, nx + 1)
    ky = ky.reshape(ny + 1, nx)
    P = p.reshape(ny, nx)
    d = kx[:, :-1] + kx[:, 1:] + ky[:-1, :] + ky[1:, :]
    y = d * P
    y[:, 1:] -= kx[:, 1:-1] * P[:, :-1]
    y[:, :-1] -= kx[:, 1:-1] * P[:, 1:]
    y[1:, :] -= ky[1:-1, :] * P[:-1, :]
    y[:-1, :] -= ky[1:-1, :] * P[1:, :]
    return y.reshape(-1)


@pytest.fixture(scope="module")
def problem():
    n = 128
    kx, ky, rhs = workloads.poisson_problem(n, seed=3)
    return n, kx, ky, rhs


@pytest.mark.parametrize("solver,precision", [("cg", 0), ("cg", 1), ("fcg_learned", 1),
                                              ("fcg_mg", 1), ("fcg_mg", 0)])
def test_poisson_true_residual(gpu, problem, solver, precision):
    n, kx, ky, rhs = problem
    print(f"case: poisson {n}x{n} {solver} precision {precision}", flush=True)
    ps = Poisson(n, n, kx, ky)
    p, st = ps.solve(rhs, solver=solver, tol=1e-8, precision=precision)
    b = rhs - rhs.mean()
    res = np.linalg.norm(b - apply(kx, ky, p, n, n)) / np.linalg.norm(b)
    assert st.converged and res <= 1.05e-8, (res, st.rel_residual, st.iterations)
    assert abs(res - st.rel_residual) <= 1e-3 * res + 1e-14


def test_poisson_matches_oracle_cg(gpu, problem):
    n, kx, ky, rhs = problem
    ps = Poisson(n, n, kx, ky)
    pg, sg = ps.solve(rhs, solver="cg", tol=1e-12, precision=0)
    po, so = pyoracle.poisson_solve(n, n, kx, ky, rhs, tol=1e-12)
    # both are solutions of the singular Neumann system: compare mean-free parts
    pg = pg - pg.mean()
    po = po - po.mean()
    assert np.linalg.norm(pg - po) <= 1e-8 * np.linalg.norm(po)


def test_multigrid_cuts_iterations(gpu, problem):
    n, kx, ky, rhs = problem
    ps = Poisson(n, n, kx, ky)
    _, s_cg = ps.solve(rhs, solver="cg", tol=1e-8, precision=0)
    _, s_mg = ps.solve(rhs, solver="fcg_learned", tol=1e-8, precision=1)
    print(f"jacobi-pcg {s_cg.iterations} it {s_cg.ms:.2f} ms; fcg+mg {s_mg.iterations} it "
          f"{s_mg.ms:.2f} ms", flush=True)
    assert s_mg.iterations * 10 < s_cg.iterations


def test_fp64_vcycle_same_iterations(gpu, problem):
    """fcg_mg with the V-cycle on FP64 levels (precision 0) against the FP32
    one (precision 1): the same kernels, so FP32 costs the preconditioner no
    strength (iteration counts within one), only halves its bytes."""
    n, kx, ky, rhs = problem
    ps = Poisson(n, n, kx, ky)
    _, s32 = ps.solve(rhs, solver="fcg_mg", tol=1e-8, precision=1)
    _, s64 = ps.solve(rhs, solver="fcg_mg", tol=1e-8, precision=0)
    print(f"fcg_mg FP32 V-cycle {s32.iterations} it {s32.ms:.3f} ms; FP64 V-cycle "
          f"{s64.iterations} it {s64.ms:.3f} ms", flush=True)
    assert s32.converged and s64.converged
    assert abs(s32.iterations - s64.iterations) <= 1


# sides that are odd at the first, a middle or every halving, lines that
# shrink to one cell, grids around the one-workgroup cycle's limits
@pytest.mark.parametrize("nx,ny", [(8, 8), (9, 9), (2, 50), (3, 700), (45, 45), (46, 45), (64, 33),
                                   (65, 32), (97, 150), (129, 130), (333, 217), (510, 509)])
def test_multigrid_any_side(gpu, nx, ny):
    """fcg_mg on grids of any sides: the true residual meets the tolerance,
    in tens of iterations where the Jacobi-PCG takes hundreds."""
    n = max(nx, ny)
    kx, ky, _ = workloads.poisson_problem(n, seed=5)
    kx = kx.reshape(n, n + 1)[:ny, :nx + 1].copy()
    ky = ky.reshape(n + 1, n)[:ny + 1, :nx].copy()
    kx[:, -1] = 0.0
    ky[-1, :] = 0.0
    rhs = np.random.default_rng(1).normal(size=nx * ny)
    print(f"case: fcg_mg {nx}x{ny}", flush=True)
    p, st = Poisson(nx, ny, kx.reshape(-1), ky.reshape(-1)).solve(rhs, solver="fcg_mg", tol=1e-8,
                                                                 precision=1)
    b = rhs - rhs.mean()
    res = np.linalg.norm(b - apply(kx, ky, p, nx, ny)) / np.linalg.norm(b)
    assert st.converged and res <= 1.05e-8
    assert st.iterations <= 100


# grids around the one-launch solve's cells per thread and workgroup counts,
# rows longer and shorter than a workgroup's range, the first sizes past it
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nx,ny", [(2, 3), (64, 16), (2, 1030), (1500, 2), (129, 127), (128, 128),
                                   (129, 128), (257, 128), (1000, 67), (1999, 9), (2100, 9),
                                   (512, 512), (513, 512)])
def test_jacobi_pcg_any_size(gpu, nx, ny, precision):
    """cg against the oracle's Jacobi-PCG: the true residual meets the
    tolerance, and in FP64 the iteration counts agree (the same recurrence;
    sums in another order, so within two and one per cent)."""
    rng = np.random.default_rng(nx + ny)
    kx, ky = rng.uniform(0.5, 2.0, (ny, nx + 1)), rng.uniform(0.5, 2.0, (ny + 1, nx))
    kx[:, 0] = kx[:, -1] = 0.0
    ky[0] = ky[-1] = 0.0
    kx, ky, rhs = kx.reshape(-1), ky.reshape(-1), rng.normal(size=nx * ny)
    print(f"case: cg {nx}x{ny} precision {precision}", flush=True)
    ps = Poisson(nx, ny, kx, ky)
    b = rhs - rhs.mean()
    for _ in range(2):  # a second solve on the same exchange words
        p, st = ps.solve(rhs, solver="cg", tol=1e-6, precision=precision)
        res = np.linalg.norm(b - apply(kx, ky, p, nx, ny)) / np.linalg.norm(b)
        assert st.converged and res <= 1.05e-6, (res, st.iterations)
        if precision == 0:
            _, so = pyoracle.poisson_solve(nx, ny, kx, ky, rhs, tol=1e-6)
            assert abs(st.iterations - so.iterations) <= 2 + 0.01 * so.iterations
    q, sq = ps.solve(rhs, solver="cg", tol=0.0, max_iters=3, precision=0)
    assert nx * ny < 7 or (sq.iterations == 3 and not sq.converged)
