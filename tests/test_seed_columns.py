"""
Every kind of source set in every kind of place of a batch (``csrc/assembly.hip``, ``seed_kernel``,
``seed_rows_kernel``): an empty set, every vertex but one, and repeated ones, first, last and between, on
meshes whose bitmap is a few words and on one of more rows than a block gathers them for; 1 to 4,096 sources
in one launch, more in two. (With every vertex a source the field's mean over the sources is its mean, and
its orientation a matter of rounding.)

Bar: 1e-9 of the range against the oracle, as for every direct query; a set without sources has no distance.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import heat_oracle as oracle

pytestmark = pytest.mark.gpu


def _mesh(name):
    from ordito_amd import creation

    return {"tiny": lambda: creation.planar_grid(5, 4, 1.0, 0.2, 6),
            "grid": lambda: creation.planar_grid(61, 47, 1.0, 0.2, 6),
            "past": lambda: creation.planar_grid(103, 80, 1.0, 0.2, 6)}[name]()  # 258 words


@pytest.mark.parametrize("name", ["tiny", "grid", "past"])
@pytest.mark.parametrize("columns,each", [(5, 3), (6, 900), (64, 2), (64, 70), (65, 64)])
def test_sets_in_every_place(cuda, name, columns, each):
    from ordito_amd import heat

    v, f = _mesh(name)
    n = len(v)
    mesh = heat.Trimesh(v, f)
    solver = mesh.heat_solver(method="meshlab")
    assert solver.factor()
    rng = np.random.default_rng(columns + each)
    few = rng.integers(0, n, each).astype(np.int32)
    kinds = [np.asarray([], np.int32), np.arange(n - 1, dtype=np.int32), np.repeat(few[:2], 3), few]
    wants = [np.zeros(n)] + [oracle.geodesic(v, f, k).distance for k in kinds[1:]]
    for turn in range(len(kinds)):
        at = [(q + turn) % len(kinds) for q in range(columns)]
        if each >= 64:  # the whole mesh once, so that both sides of 4,096 sources are met
            at = [3 if k == 1 and q != (turn + 1) % columns else k for q, k in enumerate(at)]
        got = solver.geodesic([cuda.tensor(kinds[k], dtype=cuda.int32, device="cuda") for k in at])
        got = got.cpu().numpy().reshape(columns, n)
        for q, k in enumerate(at):
            assert oracle.relative_error(got[q], wants[k])[0] <= 1e-9, (turn, q, k)
