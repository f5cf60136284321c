"""Sweep routes at the sizes where a tile can go wrong: pencils of one
segment and of several, one cell either side of a segment's limit, and the
widths around a tile's pencil count, against the oracle bit for bit (the
arithmetic is the oracle's, so no difference is allowed)."""
import numpy as np
import pytest

import oracle
from enzo_ppm import abi, device, problems
from helpers import cpu_library, field_report

# owned cells per segment are at most 57 (4 x 64 tiles): 51 active cells fill
# one segment with their ghosts, 52 need two, 108 / 109 two and three
EDGES = [(51, 4, 5), (52, 5, 4), (4, 108, 3), (3, 4, 109), (2, 2, 3), (9, 12, 7)]


def check(lib, active, solver, ncolours, dual, diffusion=0, stretch=0.0, cycle=1):
    g, glob, run = problems.random_smooth(list(active), seed=sum(active), ncolours=ncolours,
                                          dual_energy=dual, gravity=ncolours == 1,
                                          flags=(1, 1, diffusion), stretch=stretch)
    glob["RiemannSolver"] = solver
    g.fill_periodic()
    g.dt = oracle.compute_time_step("port", g, glob, run["cfl"])
    ref = g.copy()
    st = device.solve_ppm_de(g, glob, cycle=cycle, lib=lib)
    sto, _ = oracle.solve_ppm_de("port", ref, glob, cycle=cycle)
    assert st == sto == abi.SUCCESS
    for a, b in zip(g.fields, ref.fields):
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64)), field_report(g, ref)


SOLVERS = pytest.mark.parametrize("solver", [1, 4], ids=["hll", "hllc"])
SIZES = pytest.mark.parametrize("active", EDGES, ids=lambda a: "x".join(map(str, a)))


@SOLVERS
@SIZES
def test_solver_tiles_cpu(active, solver):
    check(cpu_library(), active, solver, ncolours=sum(active) % 3, dual=active[0] % 2 == 0)


@pytest.mark.gpu
@SOLVERS
@SIZES
def test_solver_tiles_gpu(active, solver):
    for ncolours, dual, stretch in ((0, False, 0.0), (2, True, 0.0), (1, True, 0.1)):
        check(None, active, solver, ncolours, dual, stretch=stretch)
