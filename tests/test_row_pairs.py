"""
Passes over fields stored by rows (``csrc/solve.hip``): the residual (``residual_pairs_kernel``, two
columns a lane and the operator's entries staged in LDS) and the finish (``rows_partial_kernel``,
``rows_decide_kernel`` with one component's mean and with several's, ``rows_out_kernel`` 16, 32 and 64
columns wide). Widths on both sides of its range and odd ones (whose last
lane repeats a column), rows of very many entries and tiles with more entries than a block holds, pinned
rows (``igl``'s second heat solve on a mesh with a rim), and float32 factors, whose refinement corrects
by every round's residual.

Bar: 1e-9 of the range against the oracle, as for every direct query; 1e-4 for mixed precision, whose
refinement stops at a served accuracy.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import heat_oracle as oracle
from tests import meshes

pytestmark = pytest.mark.gpu


def _bodies():
    from ordito_amd import creation

    v, f = creation.torus(40, 24, 1.0, 0.3, 0.1, 3)
    w, g = creation.planar_grid(23, 19, 1.0, 0.2, 6)
    return (np.concatenate([v, np.asarray(w, np.float32) + np.float32(4.0)]),
            np.concatenate([f, np.asarray(g, np.int32) + np.int32(len(v))]).astype(np.int32))


def _meshes():
    from ordito_amd import creation

    return {
        "hub": meshes.hub_disk(),
        "grid": creation.planar_grid(61, 43, 1.0, 0.2, 6),
        "torus": creation.torus(90, 45, 1.0, 0.3, 0.1, 3),
        "bodies": _bodies(),
    }


@pytest.mark.parametrize("name,method,precision", [
    ("hub", "meshlab", "fp64"), ("bodies", "meshlab", "fp64"), ("grid", "igl", "fp64"), ("hub", "igl", "fp64"),
    ("torus", "meshlab", "mixed"), ("grid", "potpourri3d", "mixed"), ("hub", "igl", "mixed")])
@pytest.mark.parametrize("columns", [1, 2, 3, 4, 5, 16, 17, 32, 33, 63, 64, 67])
def test_columns_match_the_oracle(cuda, name, method, precision, columns):
    from ordito_amd import heat

    v, f = _meshes()[name]
    n = len(v)
    rng = np.random.default_rng(columns)
    sources = [rng.integers(0, n, 2).astype(np.int32) for _ in range(columns)]
    mesh = heat.Trimesh(v, f)
    solver = mesh.heat_solver(method=method, precision=precision)
    assert solver.factor()
    bar = 1e-9 if precision == "fp64" else 1e-4
    got = solver.geodesic([cuda.tensor(s, dtype=cuda.int32, device="cuda") for s in sources])
    got = got.cpu().numpy().reshape(columns, n)
    for c in sorted({0, columns // 2, columns - 1}):
        want = oracle.geodesic(v, f, sources[c], method=method).distance
        assert oracle.relative_error(got[c], want)[0] <= bar, (name, columns, c)
