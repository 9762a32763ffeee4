"""
The one-column conjugate gradient whose state stays on the chip (``csrc/cg.hip``,
``cg_resident_kernel``), at the edges of its instances: one block and the last rows of it, the
smallest grid of blocks, the sizes where a block's threads or rows a thread change, the largest
system it holds and one past it, rows longer than the entries kept in registers, several
components, unreferenced vertices and a scrambled numbering.

Bars: the heat solve stops at the round the oracle's settled iteration stops at (up to 70,000
rows); its iterate passes the solver's own acceptance test, the componentwise backward error of
1e-6 in float64 (ordito ``linalg.py:179``), unless the mesh is the ill-shaped one whose settled
iterate falls back to the factorization by that test; a
Poisson iterate's true residual is within twice the stopping tolerance 1e-8 of its right-hand side
(the recurrence's residual stops at 1e-8; the two differ by rounding); a repeated solve gives the
same bits.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import heat_oracle as ho
from tests import conftest

pytestmark = pytest.mark.gpu


def _scrambled(a: int, b: int):
    from ordito_amd import creation

    v, f = creation.torus(a, b, 1.0, 0.3, 0.1, 2)
    order = np.random.default_rng(3).permutation(len(v))
    place = np.argsort(order)
    return v[order], place[np.asarray(f)].astype(np.int32)


def _unreferenced():
    from ordito_amd import creation

    v, f = creation.jittered_icosphere(4, 0.01, 3)
    extra = np.full((1500, 3), 0.25, np.float32)
    return np.concatenate([extra[:700], v, extra[700:]]), (np.asarray(f) + 700).astype(np.int32)


def _torus(a: int, b: int):
    from ordito_amd import creation

    return creation.torus(a, b, 1.0, 0.3, 0.1, 1)


CASES = {
    "single": lambda: conftest.mesh("icosphere3"),
    "single_last_row": lambda: _torus(32, 32),  # 1,024 rows
    "smallest_grid": lambda: _torus(41, 25),  # 1,025
    "icosphere4": lambda: conftest.mesh("icosphere4"),  # 2,562
    "two_bodies": lambda: conftest.mesh("two_bodies"),
    "unreferenced": _unreferenced,  # 4,062
    "hub": lambda: conftest.mesh("hub_disk"),  # 8,001, one row of 401 entries
    "scrambled": lambda: _scrambled(180, 90),  # 16,200
    "row_a_thread_last": lambda: _torus(256, 256),  # 65,536
    "two_rows_first": lambda: _torus(345, 190),  # 65,550
    "two_rows_last": lambda: _torus(512, 512),  # 262,144
    "four_rows_first": lambda: _torus(640, 410),  # 262,400
    "four_rows_last": lambda: _torus(1024, 512),  # 524,288
    "past_the_chip": lambda: _torus(1025, 512),  # 524,800: the state in memory
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_resident_solves_meet_their_stopping_rules(cuda, name):
    from ordito_amd import creation, heat

    v, f = CASES[name]()
    faces = np.asarray(f).reshape(-1)
    h = creation.mean_face_edge_length(v, faces)
    mesh = heat.Trimesh(v, faces)
    solver = mesh.heat_solver(t=h * h, method="meshlab")
    n = len(v)
    rng = np.random.default_rng(0)
    referenced = np.unique(faces)
    source = np.zeros(n)
    # A source every few hundred vertices: a field that a few sources leave hundreds of decades
    # below its peak settles on a large mesh before it passes the test, and falls back.
    source[rng.choice(referenced, 3 + n // 300, replace=False)] = 1.0
    rhs = cuda.from_numpy(source).cuda()
    fields = []
    for _ in range(2):
        out = cuda.empty_like(rhs)
        solver.diffuse(rhs, out)
        rounds = solver.last_stats["heat_rounds"]
        assert rounds > 0
        assert name == "hub" or not solver.ill_conditioned
        solver.release()  # forget the solve count: the second call iterates too
        fields.append(out.cpu().numpy())
    assert np.array_equal(fields[0], fields[1])
    A = solver.operators[0].to_scipy()
    x = fields[0]
    if n <= 70000:
        assert rounds == ho.settled_cg(A, source, settle_rounds=solver.settle_rounds)[1]
    residual = np.abs(source - A @ x)
    assert np.all(residual <= 1e-6 * (abs(A) @ np.abs(x) + source))

    mesh = heat.Trimesh(v, faces)  # with nothing factored: the Poisson solve iterates
    solver = mesh.heat_solver(t=h * h, method="meshlab")
    L = solver.operators[3].to_scipy()
    wave = np.sin(5.0 * v[:, 0].astype(np.float64)) + v[:, 2]
    wave[np.setdiff1d(np.arange(n), referenced)] = 0.0
    b = L @ wave
    rhs = cuda.from_numpy(b).cuda()
    fields = []
    for _ in range(2):
        out = cuda.empty_like(rhs)
        solver.solve_poisson(rhs, out)
        assert solver.last_stats["poisson_rounds"] > 0 and solver._factored() == 0
        solver.release()
        fields.append(out.cpu().numpy())
    assert np.array_equal(fields[0], fields[1])
    assert np.linalg.norm(b - L @ fields[0]) <= 2e-8 * np.linalg.norm(b)
