"""The plan arithmetic of the pipelined SOR (hydro_amd/csrc/sor_plan.h) on the
host, under UndefinedBehaviorSanitizer: limits up to 2^31 - 1 sweeps ("stop by
the tolerance alone"), against the same formulas in Python's integers."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
KEYS = ("ok_one q_one rounds doubles_one chain q g span le doubles_many a b end first workspace").split()


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ not found")
    exe = tmp_path_factory.mktemp("sor") / "sor_plan_driver"
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=undefined",
                        "-fno-sanitize-recover=all", "-o", str(exe),
                        os.path.join(ROOT, "tests", "sor_plan_driver.cpp")],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]

    def run(cases):
        text = "".join("%d %d %d %d\n" % (c if len(c) == 4 else c + (0,)) for c in cases)
        r = subprocess.run([str(exe)], input=text, capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stderr[-3000:]
        return [dict(zip(KEYS, map(int, line.split()))) for line in r.stdout.splitlines()]

    return run


GRIDS = [(64, 128), (128, 64), (128, 128), (64, 256), (256, 128), (333, 217), (512, 512),
         (1024, 1024), (2048, 1024), (9, 1030), (3, 700), (1, 100000), (1024, 9000)]


def test_last_step_of_any_limit(plan):
    limits = [0, 7, 100, 10**6, 10**8, 10**9, 2**31 - 1]
    cases = [(nx, ny, lim) for nx, ny in GRIDS for lim in limits]
    chains = 0
    for (nx, ny, lim), p in zip(cases, plan(cases)):
        if not p["chain"]:
            continue
        chains += 1
        stages = 2 * p["q"]
        ptot = p["g"] * stages
        st = lim % ptot
        end = st // stages * p["span"] + 2 * (st % stages) + lim // ptot * p["b"] + p["a"] + p["b"]
        assert p["end"] == end, (nx, ny, lim)
        # a line is kept apart from its reader, and 32 bits hold every step the
        # kernel can reach (2^30) with what it adds to one
        assert p["g"] * p["span"] <= p["b"] and ptot < p["b"]
        assert 2**30 + 2 * (p["le"] + p["b"] + p["span"] * p["g"]) < 2**31
    assert chains > 30


def test_workspace_is_bounded(plan):
    """512 MB and a double per cell, or two sweeps' ring where that is more;
    a solve of few sweeps asks for less; a chain's holds a ring for the retry."""
    grids = GRIDS + [(64, 65536), (32, 120000), (512, 1024), (1024, 20000), (2, 4000000)]
    cases = [(nx, ny, lim) for nx, ny in grids for lim in (-3, 0, 5, 1000, 2**31 - 1)]
    for (nx, ny, lim), p in zip(cases, plan(cases)):
        n = nx * ny
        ring = 32 + (7 + 2 * p["rounds"]) * n
        assert p["workspace"] <= max(2**26 + n, ring), (nx, ny, lim)
        if min(nx, ny) <= 1024 and lim >= 0 and ring < 2**29:
            assert p["workspace"] >= ring
        if lim == 0:
            assert p["workspace"] <= ring
        if lim == 5:  # three pairs of sweeps
            assert p["workspace"] <= 32 + (7 + 6 * p["rounds"]) * n


def test_workspace_holds_the_first_sweeps(plan):
    """A solve in the workspace it asks for keeps the first sweeps' values too; one
    in less drops those before it drops sweeps in flight."""
    grids = GRIDS + [(512, 1024), (64, 65536), (700, 290), (16, 16)]
    cases = [(nx, ny, lim) for nx, ny in grids for lim in (0, 100, 2**31 - 1)]
    full = plan(cases)
    again = plan([c + (p["workspace"],) for c, p in zip(cases, full)])
    for c, p, q in zip(cases, full, again):
        assert not p["workspace"] or q["first"], c
    # the 16 MiB array of the allocation-free call, less its header
    for (nx, ny), q, g in [((700, 290), 1, 0), ((333, 217), 5, 7), ((340, 435), 2, 0)]:
        p = plan([(nx, ny, 100, 2096992)])[0]
        assert p["g"] == g if g else (p["ok_one"] and p["q_one"] == q and not p["chain"]), (nx, p)
