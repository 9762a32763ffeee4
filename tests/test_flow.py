"""
The sweeps of a few right-hand sides in one launch (``csrc/flow.hip``): against the same solves
level by level, which a mesh falls back to when such a launch gives up waiting.

Bar: both are float64 sums of the same products in different orders, refined to the same residual
tests; the fields agree to 1e-10 of their range (the graded saddle's conditioning, the worst here,
leaves its factored answer within 1e-9 of the oracle's), and two passes give the same bits.
"""

from __future__ import annotations

import numpy as np
import pytest

from tests import conftest


def _meshes():
    from ordito_amd import creation

    return {
        "tetrahedron": lambda: (
            np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]], np.float32),
            np.array([0, 2, 1, 0, 1, 3, 1, 2, 3, 2, 0, 3], np.int32),
        ),  # one front of one tile
        "one_front": lambda: creation.torus(16, 8, 1.0, 0.3, 0.1, 3),  # 128 rows: a leaf alone
        "two_bodies": lambda: conftest.mesh("two_bodies"),
        "saddle_graded": lambda: conftest.mesh("saddle_graded"),
        "hub_disk": lambda: conftest.mesh("hub_disk"),
        "grid": lambda: creation.planar_grid(171, 83, 1.0, 0.2, 4),
        "torus": lambda: creation.torus(400, 200, 1.0, 0.3, 0.1, 5),  # fronts past 1,024 rows
    }


NAMES = ("tetrahedron", "one_front", "two_bodies", "saddle_graded", "hub_disk", "grid", "torus")


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("name", NAMES)
def test_one_launch_sweeps_equal_level_sweeps(cuda, name, precision):
    from ordito_amd import _lib, heat

    v, f = _meshes()[name]()
    n = len(v)
    rng = np.random.default_rng(1)
    solver = None
    for columns in (1, 2, 3, 4):
        sets = [cuda.tensor(rng.choice(n, 1 + q % 2, replace=False), dtype=cuda.int32, device="cuda")
                for q in range(columns)]
        fields = {}
        for patience in (1 << 21, 0):
            mesh = heat.Trimesh(v, f)
            solver = mesh.heat_solver(method="meshlab", precision=precision)
            assert solver.factor()
            _lib.call("hg_set_sweep_patience", solver._native().ptr, patience)
            first, second = (solver.geodesic(sets).cpu().numpy() for _ in range(2))
            assert np.array_equal(first, second)
            fields[patience] = first
        one, level = fields[1 << 21], fields[0]
        tolerance = 1e-10 if precision == "fp64" else 1e-6  # mixed is refined to 1e-6
        for q in range(columns):
            assert np.max(np.abs(one[q] - level[q])) <= tolerance * np.ptp(level[q])


@pytest.mark.gpu
def test_later_rounds_and_other_layouts(cuda):
    """A diffusion through the factors refined in several rounds (a target one round misses), from
    and to fields stored by columns, one launch a sweep and level by level."""
    from ordito_amd import _lib, heat

    v, f = conftest.mesh("saddle_graded")
    n = len(v)
    rhs = cuda.zeros((3, n), dtype=cuda.float64, device="cuda")
    for q, s in enumerate((0, 300, n - 1)):
        rhs[q, s] = 1.0
    out = {}
    for patience in (1 << 21, 0):
        mesh = heat.Trimesh(v, f)
        solver = mesh.heat_solver(method="meshlab", precision="mixed")
        assert solver.factor()
        _lib.call("hg_set_sweep_patience", solver._native().ptr, patience)
        solver.set_refinement(heat=1e-11, poisson=1e-10)
        field = cuda.empty_like(rhs)
        solver.diffuse(rhs, field)
        assert solver.last_stats["heat_refinements"] > 1
        out[patience] = field.cpu().numpy()
    # Componentwise backward errors of 1e-11 twice over the field's own conditioning.
    one, level = out[1 << 21], out[0]
    assert np.max(np.abs(one - level) / np.abs(level).max()) <= 1e-8


def test_tasks_cover_every_output_in_dependency_order():
    """hg_plan_validate's checks of the one-launch lists, at several front shapes."""
    import scipy.sparse as sp

    from ordito_amd import analysis

    for name in NAMES:
        v, f = _meshes()[name]()
        t = np.asarray(f).reshape(-1, 3)
        i = np.r_[t[:, 0], t[:, 1], t[:, 2], t[:, 1], t[:, 2], t[:, 0], np.arange(len(v))]
        j = np.r_[t[:, 1], t[:, 2], t[:, 0], t[:, 0], t[:, 1], t[:, 2], np.arange(len(v))]
        a = sp.csr_matrix((np.ones(len(i)), (i, j)))
        a.sum_duplicates()
        a.sort_indices()
        for leaf, top in ((0, 0), (16, 64), (300, 2000)):
            analysis.analyse(a.indptr.astype(np.int32), a.indices.astype(np.int32), v,
                             leaf_rows=leaf, top_rows=top, validate=True)
