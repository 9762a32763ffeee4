"""
Separators merged upwards into one front (``csrc/analysis.cpp``): the same fields as from the plan that
keeps each its own front (which a memory budget asks for), on one body and several, a mesh with vertices
of very many neighbours, a rim's second heat system and a graph that is one leaf; and the budget itself,
held against the unmerged plan's peak whichever plan the mesh has.

Bar: 1e-10 of the range, as between any two direct solves of one system.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from ordito_amd import _lib
from tests import meshes

pytestmark = pytest.mark.gpu


def _meshes():
    from ordito_amd import creation

    v, f = creation.torus(60, 44, 1.0, 0.3, 0.1, 3)
    w, g = creation.planar_grid(43, 39, 1.0, 0.2, 6)
    bodies = (np.concatenate([v, np.asarray(w, np.float32) + np.float32(4.0)]),
              np.concatenate([f, np.asarray(g, np.int32) + np.int32(len(v))]).astype(np.int32))
    return {
        "bodies": bodies,
        "hub": meshes.hub_disk(),
        "grid": creation.planar_grid(150, 140, 1.0, 0.2, 6),
        "leaf": creation.planar_grid(9, 8, 1.0, 0.2, 6),
    }


def _solver(name, method, budget):
    from ordito_amd import heat

    mesh = heat.Trimesh(*_meshes()[name])
    solver = mesh.heat_solver(method=method)
    if budget:
        solver.set_memory_budget(budget)
    return mesh, solver


@pytest.mark.parametrize("name,method", [("bodies", "meshlab"), ("hub", "igl"), ("grid", "igl"),
                                         ("grid", "potpourri3d"), ("leaf", "meshlab")])
@pytest.mark.parametrize("columns", [1, 4, 5, 64])
def test_fields_match_the_unmerged_plan(cuda, name, method, columns):
    rng = np.random.default_rng(columns)
    fields, fronts = [], []
    sources = None
    for budget in (0, 1 << 40):
        mesh, solver = _solver(name, method, budget)
        assert solver.factor()
        if sources is None:
            sources = [rng.integers(0, mesh.n_vertices, 2).astype(np.int32) for _ in range(columns)]
        fronts.append(solver.plan_stats()["supernodes"])
        fields.append(solver.geodesic([cuda.tensor(s, dtype=cuda.int32, device="cuda")
                                       for s in sources]).cpu().numpy())
    assert fronts[0] == fronts[1] if name == "leaf" else fronts[0] < fronts[1]
    for a, b in zip(*fields):
        assert np.max(np.abs(a - b)) <= 1e-10 * max(np.ptp(b), 1e-300)


def test_a_budget_is_held_against_the_unmerged_peak(cuda):
    _, solver = _solver("grid", "meshlab", 1 << 40)
    assert solver.factor()
    stats = solver.plan_stats()
    peak = 8 * stats["arena_entries"] + 16 * stats["solve_block_entries"]
    mesh, fresh = _solver("grid", "meshlab", peak - 1)
    assert not fresh.factor()
    fresh.set_memory_budget(peak)
    assert fresh.factor()
    # A heat factor held on the merged plan stays; the Poisson system is held against the same peak.
    mesh, late = _solver("grid", "meshlab", 0)
    done = ctypes.c_int32()
    _lib.call("hg_factor", late._native().ptr, _lib.HG_SYSTEM_HEAT, 0, ctypes.byref(done))
    assert done.value and late.plan_stats()["supernodes"] < stats["supernodes"]
    late.set_memory_budget(peak - 1)
    assert not late.factor()
    late.set_memory_budget(peak)
    assert late.factor()
    assert late.plan_stats()["supernodes"] < stats["supernodes"]
