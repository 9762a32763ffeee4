"""
The one-column conjugate gradient in one block (``csrc/cg.hip``, ``choose_resident``): the last size of each
number of threads and the first of the next.

Bars, as for every iterate: the heat solve stops at the round the oracle's settled iteration stops at,
with a componentwise backward error of 1e-6 in float64; a Poisson iterate's true residual is within twice
the stopping tolerance 1e-8 of its right-hand side; a repeated solve gives the same bits.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import heat_oracle as ho

pytestmark = pytest.mark.gpu


def _mesh(n: int):
    """A torus of a multiple of 64 vertices, or one and an unreferenced vertex."""
    from ordito_amd import creation

    v, f = creation.torus(n // 64 * 4, 16, 1.0, 0.3, 0.1, 3) if n >= 64 else creation.torus(6, 7, 1.0, 0.3, 0.1, 3)
    v = np.concatenate([v, np.zeros((n - len(v), 3), np.float32)]).astype(np.float32)
    return v, np.asarray(f).reshape(-1)


@pytest.mark.parametrize("n", [42, 256, 257, 512, 513, 1024])
def test_iterates_meet_their_stopping_rules(cuda, n):
    from ordito_amd import creation, heat

    v, f = _mesh(n)
    assert len(v) == n
    h = creation.mean_face_edge_length(v, f)
    source = np.zeros(n)
    source[[0, n // 3]] = 1.0
    waves = np.sin(5.0 * v[:, 0].astype(np.float64)) + v[:, 2]
    waves[np.setdiff1d(np.arange(n), f)] = 0.0
    for poisson in (False, True):
        fields = []
        for _ in range(2):
            mesh = heat.Trimesh(v, f)
            solver = mesh.heat_solver(t=h * h, method="meshlab")
            A = solver.operators[3 if poisson else 0].to_scipy()
            b = A @ waves if poisson else source
            rhs = cuda.from_numpy(b).cuda()
            out = cuda.empty_like(rhs)
            (solver.solve_poisson if poisson else solver.diffuse)(rhs, out)
            rounds = solver.last_stats["poisson_rounds" if poisson else "heat_rounds"]
            assert rounds > 0 and not solver.ill_conditioned
            fields.append(out.cpu().numpy())
        assert np.array_equal(fields[0], fields[1])
        x = fields[0]
        if poisson:
            assert np.linalg.norm(b - A @ x) <= 2e-8 * np.linalg.norm(b)
        else:
            assert rounds == ho.settled_cg(A, source, settle_rounds=solver.settle_rounds)[1]
            assert np.all(np.abs(b - A @ x) <= 1e-6 * (abs(A) @ np.abs(x) + b))
