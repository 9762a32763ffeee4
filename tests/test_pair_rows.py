"""
The rows a block of the residual and of the divergence takes from three and five columns on
(``csrc/kernels.h``, ``pair_rows``): one turn of them up to 8,192 rows, several past that. Both sides of
that line, with a row of many neighbours past it, at widths that fill a turn differently.

Bar: 1e-9 of the range against the oracle, as for every direct query.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import heat_oracle as oracle
from tests.test_long_rows import cone

pytestmark = pytest.mark.gpu


def _mesh(name):
    from ordito_amd import creation

    if name == "hub":
        return cone(70, 130)  # 9,101 rows
    return creation.torus(128, 64 if name == "last" else 65, 1.0, 0.3, 0.1, 3)  # 8,192 and 8,320


@pytest.mark.parametrize("name", ["last", "first", "hub"])
@pytest.mark.parametrize("columns", [3, 5, 16, 33, 64])
def test_columns_match_the_oracle(cuda, name, columns):
    from ordito_amd import heat

    v, f = _mesh(name)
    mesh = heat.Trimesh(v, f)
    solver = mesh.heat_solver(method="meshlab")
    assert solver.factor()
    rng = np.random.default_rng(columns)
    sources = [rng.integers(0, len(v), 2).astype(np.int32) for _ in range(columns)]
    got = solver.geodesic([cuda.tensor(s, dtype=cuda.int32, device="cuda") for s in sources])
    got = got.cpu().numpy().reshape(columns, len(v))
    for c in (0, columns - 1):
        want = oracle.geodesic(v, np.asarray(f).reshape(-1), sources[c]).distance
        assert oracle.relative_error(got[c], want)[0] <= 1e-9, c
