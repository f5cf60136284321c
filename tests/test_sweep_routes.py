"""Sweep routes at the sizes where a tile can go wrong: pencils of one
segment and of several, one cell either side of a segment's limit, and the
widths around a tile's pencil count, against the oracle bit for bit (the
arithmetic is the oracle's, so no difference is allowed)."""
import numpy as np
import pytest

import oracle
from enzo_ppm import abi, device, problems
from helpers import DeviceArrays, cpu_library, field_report, noalloc_solve

# owned cells per segment are at most 57 (4 x 64 tiles): 51 active cells fill
# one segment with their ghosts, 52 need two, 108 / 109 two and three
EDGES = [(51, 4, 5), (52, 5, 4), (4, 108, 3), (3, 4, 109), (2, 2, 3), (9, 12, 7)]


def check(lib, active, solver, ncolours, dual, stretch=0.0, cycle=1):
    g, glob, run = problems.random_smooth(list(active), seed=sum(active), ncolours=ncolours,
                                          dual_energy=dual, gravity=ncolours == 1,
                                          stretch=stretch)
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


# Diffusion in one launch: slices that wait for each other along every axis,
# rows in one and several groups, single-row slices (2-D), and the slices
# next to the edges that read no neighbour (3 and 2 active cells across).
DIFF_SIZES = [(52, 3, 9), (4, 60, 3), (6, 2, 51), (13, 11, 12), (40, 17), (21, 53)]
DIFFUSION = pytest.mark.parametrize("active", DIFF_SIZES, ids=lambda a: "x".join(map(str, a)))
ALL_SOLVERS = pytest.mark.parametrize("solver", [5, 1, 4], ids=["twoshock", "hll", "hllc"])


def check_diffusion(lib, active, solver, ncolours, dual, stretch=0.0):
    for cycle in range(len(active)):
        g, glob, run = problems.random_smooth(list(active), rank=len(active), seed=sum(active),
                                              ncolours=ncolours, dual_energy=dual,
                                              gravity=ncolours == 1, flags=(1, 1, 1), amp=0.2,
                                              vamp=0.4, stretch=stretch)
        glob["RiemannSolver"] = solver
        g.fill_periodic()
        g.dt = 0.5 * oracle.compute_time_step("port", g, glob, run["cfl"])
        ref = g.copy()
        sto, nfb = oracle.solve_ppm_de("port", ref, glob, cycle=cycle)
        assert sto == abi.SUCCESS and nfb == 0  # no case here needs the per-cell fallback
        assert device.solve_ppm_de(g, glob, cycle=cycle, lib=lib) == abi.SUCCESS
        for a, b in zip(g.fields, ref.fields):
            assert np.array_equal(a.view(np.uint64), b.view(np.uint64)), field_report(g, ref)


@ALL_SOLVERS
@DIFFUSION
def test_diffusion_slices_cpu(active, solver):
    check_diffusion(cpu_library(), active, solver, ncolours=sum(active) % 3, dual=active[0] % 2 == 0)


@pytest.mark.gpu
@ALL_SOLVERS
@DIFFUSION
def test_diffusion_slices_gpu(active, solver):
    for ncolours, dual, stretch in ((0, False, 0.0), (2, True, 0.0), (1, True, 0.1)):
        check_diffusion(None, active, solver, ncolours, dual, stretch)


def large_diffusion_case():
    """A grid that fits the entry point that allocates nothing, but not with
    the exchange array beside it (256 MiB): the exchange then stays in the
    state's own arrays."""
    g, glob, run = problems.random_smooth([129, 129, 129], seed=3, dual_energy=True,
                                          flags=(1, 1, 1), amp=0.2, vamp=0.4)
    g.fill_periodic()
    g.dt = 0.5 * oracle.compute_time_step("port", g, glob, run["cfl"])
    return g, glob


@pytest.mark.gpu
def test_diffusion_exchange_in_state():
    g, glob = large_diffusion_case()
    fields = DeviceArrays(g.fields)
    try:
        st, nfb = noalloc_solve(abi.load_library(), g, glob, 1, fields.addrs())
        assert (st, nfb) == (abi.SUCCESS, 0)
        got = [np.empty_like(f) for f in g.fields]
        for k, f in enumerate(got):
            fields.read(k, f)
    finally:
        fields.free()
    assert device.solve_ppm_de(g, glob, cycle=1) == abi.SUCCESS
    for a, b in zip(got, g.fields):
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64))
