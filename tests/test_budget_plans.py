"""
A memory budget set when a factor is held on a plan whose small separators are merged
(``csrc/api.hip``, ``require_budget``): what is then factored allocates no more than the budget. A
long strip cut into leaves of four rows stores more than half again as much merged as unmerged, so a
budget of the unmerged peak does not hold the merged factorization; the grid's merged factorization
allocates less than its unmerged peak, and its plan stays.

Bar: 1e-10 of the range between the fields of the two plans, as between any two direct solves of one
system.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from ordito_amd import _lib

pytestmark = pytest.mark.gpu


def _solver(shape, leaf, budget=0):
    from ordito_amd import creation, heat

    mesh = heat.Trimesh(*creation.planar_grid(*shape, 1.0, 0.2, 6))
    solver = mesh.heat_solver(method="meshlab")
    _lib.call("hg_set_plan_options", solver._native().ptr, leaf, 0, 0)
    if budget:
        solver.set_memory_budget(budget)
    return mesh, solver


def _factor(solver, system, precision=_lib.HG_PRECISION_FP64):
    done = ctypes.c_int32()
    _lib.call("hg_factor", solver._native().ptr, system, precision, ctypes.byref(done))
    return bool(done.value)


@pytest.mark.parametrize("shape,leaf,stays", [((600, 5), 4, False), ((150, 140), 128, True)])
@pytest.mark.parametrize("mixed", [False, True])
def test_what_is_factored_keeps_within_the_budget(cuda, shape, leaf, stays, mixed):
    unmerged_mesh, unmerged = _solver(shape, leaf, 1 << 40)
    assert unmerged.factor()
    plain = unmerged.plan_stats()
    peak = 8 * plain["arena_entries"] + 16 * plain["solve_block_entries"]

    mesh, solver = _solver(shape, leaf)
    assert _factor(solver, _lib.HG_SYSTEM_HEAT, int(mixed))
    merged = solver.plan_stats()
    assert merged["supernodes"] < plain["supernodes"]
    nnz = solver.operators[0].values.numel()

    solver.set_memory_budget(peak - 1)
    assert not _factor(solver, _lib.HG_SYSTEM_POISSON)
    assert solver.plan_stats() == merged and _factor(solver, _lib.HG_SYSTEM_HEAT)

    solver.set_memory_budget(peak)
    assert _factor(solver, _lib.HG_SYSTEM_POISSON)
    stats = solver.plan_stats()
    allocated = 8 * (stats["arena_entries"] + stats["solve_block_entries"] + nnz)
    assert allocated <= peak
    assert stats["supernodes"] == (merged if stays else plain)["supernodes"]
    # The heat factor held before the budget is held still, with its FP32 blocks.
    systems = ctypes.c_int32()
    _lib.call("hg_factored", solver._native().ptr, ctypes.byref(systems))
    assert systems.value == _lib.HG_SYSTEM_HEAT | _lib.HG_SYSTEM_POISSON
    blocks = 8 * stats["solve_block_entries"] + 8 * nnz
    held = 2 * blocks + (4 * stats["solve_block_entries"] if mixed else 0)
    assert solver.nbytes >= held

    sets = [cuda.tensor([3, mesh.n_vertices - 1], dtype=cuda.int32, device="cuda"),
            cuda.tensor([7], dtype=cuda.int32, device="cuda")]
    for a, b in zip(solver.geodesic(sets).cpu().numpy(), unmerged.geodesic(sets).cpu().numpy()):
        assert np.max(np.abs(a - b)) <= 1e-10 * np.ptp(b)
    # Poisson solves of the caller's fields, through the pins of the plan in place.
    rhs = cuda.zeros((2, mesh.n_vertices), dtype=cuda.float64, device="cuda")
    rhs[0, 5], rhs[0, 9], rhs[1, 2], rhs[1, -2] = 1.0, -1.0, 2.0, -2.0
    out, other = cuda.empty_like(rhs), cuda.empty_like(rhs)
    solver.solve_poisson(rhs, out)
    unmerged.solve_poisson(rhs, other)
    for a, b in zip(out.cpu().numpy(), other.cpu().numpy()):
        assert np.max(np.abs(a - b)) <= 1e-10 * np.ptp(b)


def test_a_poisson_solve_that_replaces_the_plan(cuda):
    """The plan replaced within the call that needs the Poisson factor."""
    _, unmerged = _solver((600, 5), 4, 1 << 40)
    assert unmerged.factor()
    stats = unmerged.plan_stats()
    mesh, solver = _solver((600, 5), 4)
    assert _factor(solver, _lib.HG_SYSTEM_HEAT)
    solver.set_memory_budget(8 * stats["arena_entries"] + 16 * stats["solve_block_entries"])
    rhs = cuda.zeros((1, mesh.n_vertices), dtype=cuda.float64, device="cuda")
    rhs[0, 5], rhs[0, 9] = 1.0, -1.0
    out, other = cuda.empty_like(rhs), cuda.empty_like(rhs)
    solver.solve_poisson(rhs, out)
    unmerged.solve_poisson(rhs, other)
    assert solver.plan_stats()["supernodes"] == stats["supernodes"]
    a, b = out.cpu().numpy(), other.cpu().numpy()
    assert np.max(np.abs(a - b)) <= 1e-10 * np.ptp(b)
