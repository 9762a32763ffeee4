"""
Which way a mesh's solves swept (``hg_sweep_counts``): up to four columns in one launch a round
(``csrc/flow.hip``), more level by level, and a launch that gave up waiting noted by the first call
that sees it, so that no later solve waits for another.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from ordito_amd import _lib
from tests import conftest

pytestmark = pytest.mark.gpu


def _solver(cuda, mesh, method, precision, patience):
    from ordito_amd import heat

    trimesh = heat.Trimesh(*mesh)
    solver = trimesh.heat_solver(method=method, precision=precision)
    assert solver.factor()
    if method == "igl":
        done = ctypes.c_int32()
        _lib.call("hg_factor", solver._native().ptr, _lib.HG_SYSTEM_PINNED, 0, ctypes.byref(done))
        assert done.value
    if patience is not None:
        _lib.call("hg_set_sweep_patience", solver._native().ptr, patience)
    return trimesh, solver


def _counts(solver):
    out = (ctypes.c_int64 * 3)()
    _lib.call("hg_sweep_counts", solver._native().ptr, out)
    return list(out)


def _sets(cuda, n, columns):
    return [cuda.tensor([(7 * q) % n], dtype=cuda.int32, device="cuda") for q in range(columns)]


def _mesh(name):
    from ordito_amd import creation

    return creation.planar_grid(171, 83, 1.0, 0.2, 4) if name == "grid" else conftest.mesh(name)


@pytest.mark.parametrize("name", ["grid", "saddle_graded"])
@pytest.mark.parametrize("graphs", [True, False])
@pytest.mark.parametrize("method,systems", [("meshlab", 2), ("igl", 3)])
def test_fp64_queries(cuda, name, graphs, method, systems):
    trimesh, solver = _solver(cuda, _mesh(name), method, "fp64", None)
    solver.set_graphs(graphs)
    for columns in (1, 4):
        before = _counts(solver)
        for _ in range(3):
            solver.geodesic(_sets(cuda, trimesh.n_vertices, columns))
        calls = 1 if graphs else 3  # a graph's rounds count where it is captured
        flows, levels, given_up = (a - b for a, b in zip(_counts(solver), before))
        assert (flows, levels, given_up) == (systems * calls, 0, 0)
    before = _counts(solver)
    solver.geodesic(_sets(cuda, trimesh.n_vertices, 5))
    assert [a - b for a, b in zip(_counts(solver), before)] == [0, systems, 0]


@pytest.mark.parametrize("graphs", [True, False])
def test_a_launch_that_gave_up_is_the_last(cuda, graphs):
    trimesh, solver = _solver(cuda, _mesh("grid"), "meshlab", "fp64", 0)
    solver.set_graphs(graphs)
    sets = _sets(cuda, trimesh.n_vertices, 2)
    first = solver.geodesic(sets).cpu().numpy()
    # The speculating pass that gave up, and one level by level.
    assert _counts(solver) == [2, 2, 1]
    for _ in range(3):
        again = solver.geodesic(sets).cpu().numpy()
        assert np.max(np.abs(again - first)) <= 1e-10 * np.ptp(first)
    flows, levels, given_up = _counts(solver)
    assert (flows, given_up) == (2, 1) and levels > 2
    # Setting the patience returns the mesh to one-launch sweeps.
    _lib.call("hg_set_sweep_patience", solver._native().ptr, 1 << 21)
    solver.geodesic(sets)
    assert _counts(solver) == [4, levels, 1]


@pytest.mark.parametrize("patience", [None, 0])
def test_rounds_that_wait_for_their_verdicts(cuda, patience):
    trimesh, solver = _solver(cuda, _mesh("grid"), "meshlab", "mixed", patience)
    solver.geodesic(_sets(cuda, trimesh.n_vertices, 3))
    flows, levels, given_up = _counts(solver)
    if patience is None:
        rounds = solver.last_stats["heat_refinements"] + solver.last_stats["poisson_refinements"]
        assert (flows, levels, given_up) == (rounds, 0, 0)
    else:
        assert (flows, given_up) == (1, 1) and levels > 0
    rhs = cuda.zeros((1, trimesh.n_vertices), dtype=cuda.float64, device="cuda")
    rhs[0, 3] = 1.0
    before = _counts(solver)
    solver.diffuse(rhs, cuda.empty_like(rhs))
    flows, levels, given_up = (a - b for a, b in zip(_counts(solver), before))
    assert given_up == 0 and (flows > 0) == (patience is None) and (levels > 0) == (patience == 0)


@pytest.mark.parametrize("columns", [1, 4])
def test_many_fp32_entries_sweep_level_by_level(cuda, columns):
    """A torus of 160,000 rows stores 38.3 million entries, past the 2^25 of FP32 blocks that sweep in
    one launch."""
    from ordito_amd import creation

    mesh = creation.torus(400, 400, 1.0, 0.3, 0.1, 4)
    fields = {}
    for precision in ("mixed", "fp64"):
        trimesh, solver = _solver(cuda, mesh, "meshlab", precision, None)
        assert solver.plan_stats()["solve_block_entries"] > 1 << 25
        fields[precision] = solver.geodesic(_sets(cuda, trimesh.n_vertices, columns)).cpu().numpy()
        flows, levels, given_up = _counts(solver)
        assert given_up == 0
        assert (flows == 0 and levels > 0) if precision == "mixed" else (flows == 2 and levels == 0)
    for got, want in zip(fields["mixed"], fields["fp64"]):
        assert np.max(np.abs(got - want)) <= 1e-6 * np.ptp(want)
