"""
The divergence of fields stored by rows (``csrc/assembly.hip``, ``divergence_rows_kernel`` and its
form for pairs of columns) from per-corner records in the corner's own plane: the widths on both sides
of each kernel's range (pairs of columns from five on, 64 a chunk; odd ones), vertices of
very many corners and of none, grid rows of fewer corners than a batch and rim rows, faces of no area,
two bodies (one without a source, whose heat is flat zero), and heat far below 1 (a mesh many
diffusion lengths across, whose directions are scaled before they are normalized).

Bar: 1e-9 of the range against the oracle, as for every direct query.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import heat_oracle as oracle
from tests import meshes

pytestmark = pytest.mark.gpu


def _meshes():
    from ordito_amd import creation

    def joined():
        v, f = creation.torus(40, 24, 1.0, 0.3, 0.1, 3)
        w, g = creation.icosphere(2)
        return (np.concatenate([v, np.asarray(w, np.float32) + np.float32(4.0)]),
                np.concatenate([f, np.asarray(g, np.int32) + np.int32(len(v))]).astype(np.int32))

    def flat_faces():
        v, f = creation.torus(40, 24, 1.0, 0.3, 0.1, 3)
        extra = np.asarray([5, 6, 6, 9, 9, 9], np.int32)  # no area: no gradient
        return v, np.concatenate([f[:600], extra, f[600:]]).astype(np.int32)

    return {
        "hub": meshes.hub_disk(),
        "grid": creation.planar_grid(37, 23, 1.0, 0.2, 6),
        "joined": joined(),
        "flat_faces": flat_faces(),
        "far": creation.planar_grid(400, 5, 1.0, 0.1, 6),
    }


@pytest.mark.parametrize("name", ["hub", "grid", "joined", "flat_faces", "far"])
@pytest.mark.parametrize("columns", [1, 2, 4, 5, 7, 8, 31, 32, 33, 64, 65])
def test_columns_match_the_oracle(cuda, name, columns):
    from ordito_amd import heat

    v, f = _meshes()[name]
    n = len(v)
    rng = np.random.default_rng(columns)
    first = n // 2 if name == "joined" else n  # the second body of two is never a source's
    sources = [rng.integers(0, first, 1).astype(np.int32) for _ in range(columns)]
    mesh = heat.Trimesh(v, f)
    solver = mesh.heat_solver(method="meshlab")
    assert solver.factor()
    got = solver.geodesic([cuda.tensor(s, dtype=cuda.int32, device="cuda") for s in sources])
    got = got.cpu().numpy().reshape(columns, n)
    for c in sorted({0, columns // 2, columns - 1}):
        want = oracle.geodesic(v, f, sources[c]).distance
        assert oracle.relative_error(got[c], want)[0] <= 1e-9, (name, columns, c)
