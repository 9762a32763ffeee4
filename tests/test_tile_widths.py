"""
The tile products' column blocks (``csrc/solve.hip``): batches at the edges of the 16-, 32- and
64-column instances, each column against its set solved on its own, on meshes whose fronts end
inside a 16-row operand block.

Bar: 1e-10 of the range, as the one-launch sweeps' (a column's sums are the same products in another
order, refined to the same tests).
"""

from __future__ import annotations

import numpy as np
import pytest

from tests import conftest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("columns", [5, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 69])
@pytest.mark.parametrize("name", ["two_bodies", "hub_disk", "torus_61x47"])
def test_each_column_equals_its_set_alone(cuda, name, columns, precision):
    from ordito_amd import creation, heat

    v, f = creation.torus(61, 47, 1.0, 0.3, 0.1, 9) if name == "torus_61x47" else conftest.mesh(name)
    mesh = heat.Trimesh(v, f)
    solver = mesh.heat_solver(method="meshlab", precision=precision)
    assert solver.factor()
    rng = np.random.default_rng(columns)
    sets = [cuda.tensor(rng.choice(len(v), 1 + q % 3, replace=False), dtype=cuda.int32, device="cuda")
            for q in range(columns)]
    fields = solver.geodesic(sets).cpu().numpy()
    tolerance = 1e-10 if precision == "fp64" else 1e-6
    for q in sorted({0, 1, columns // 2, columns - 2, columns - 1}):
        alone = solver.geodesic([sets[q]])[0].cpu().numpy()
        assert np.max(np.abs(fields[q] - alone)) <= tolerance * np.ptp(alone), q
