"""
The heat step's forward sweep over the fronts its sources reach only (``csrc/solve.hip``,
``mark_fronts_kernel``): a source set solved in a batch whose sources lie in a few fronts, against
the same set in a batch with a column that has a source in every front, which marks them all. Both
widths' sweeps, several components with sources in some of them, packed meshes asked about in part,
``igl``'s two heat solves, an empty set and repeated sources.

Bar: 1e-10 of the range, as between any two batches of one set (the products left out are of zeros).
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _two_tori():
    from ordito_amd import creation

    v, f = creation.torus(220, 110, 1.0, 0.3, 0.1, 3)
    w, g = creation.torus(150, 140, 1.0, 0.3, 0.1, 4)
    return (np.concatenate([v, w + np.float32(4.0)]),
            np.concatenate([f, g + np.int32(len(v))]).astype(np.int32))


def _meshes():
    from ordito_amd import creation

    return {
        "torus": creation.torus(400, 200, 1.0, 0.3, 0.1, 5),
        "two_tori": _two_tori(),
        "grid": creation.planar_grid(260, 170, 1.0, 0.2, 6),
    }


def _tensor(cuda, values):
    return cuda.tensor(np.asarray(values, np.int32), dtype=cuda.int32, device="cuda")


@pytest.mark.parametrize("name,method", [("torus", "meshlab"), ("two_tori", "meshlab"),
                                         ("grid", "igl"), ("grid", "potpourri3d")])
@pytest.mark.parametrize("columns", [1, 3, 7, 40, 64, 70])
def test_few_sources_equal_sources_everywhere(cuda, name, method, columns):
    from ordito_amd import heat

    v, f = _meshes()[name]
    n = len(v)
    mesh = heat.Trimesh(v, f)
    solver = mesh.heat_solver(method=method)
    assert solver.factor()
    assert solver.plan_stats()["supernodes"] >= 256  # else every front is swept anyway
    rng = np.random.default_rng(columns)
    # All sources near one vertex (in one body of two), with repeats and an empty set.
    sets = [_tensor(cuda, [17, 17, int(rng.integers(n // 3))]), _tensor(cuda, [])]
    sets = (sets + [_tensor(cuda, rng.integers(0, 200, 2)) for _ in range(columns)])[:columns]
    everywhere = _tensor(cuda, np.arange(0, n, 11))
    few = solver.geodesic(sets).cpu().numpy()
    # The same chunk's columns beside one with a source in every front; a chunk holds 64.
    for start in range(0, columns, 63):
        part = sets[start : start + 63]
        all_fronts = solver.geodesic(part + [everywhere]).cpu().numpy()
        for q in range(len(part)):
            worst = np.max(np.abs(few[start + q] - all_fronts[q]))
            assert worst <= 1e-10 * max(np.ptp(all_fronts[q]), 1e-300), (start + q, worst)


def test_packed_meshes_asked_about_in_part(cuda):
    from ordito_amd import creation
    from ordito_amd.batch import MeshBatch

    rng = np.random.default_rng(0)
    meshes = list(creation.mesh_collection(12, 1000, 20000, rng).values())
    batch = MeshBatch(meshes)
    queries = [(m, rng.choice(len(meshes[m][0]), 3, replace=False).astype(np.int32))
               for m in (2, 5, 5, 11)]
    some = [field.cpu().numpy() for field in batch.geodesic(queries)]
    every = queries + [(m, np.arange(0, len(meshes[m][0]), 7, dtype=np.int32)) for m in range(12)]
    fields = [field.cpu().numpy() for field in batch.geodesic(every)]
    for a, b in zip(some, fields):
        assert np.max(np.abs(a - b)) <= 1e-10 * np.ptp(b)
