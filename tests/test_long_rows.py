"""
Meshes with vertices of very many neighbours: the conjugate gradient deals a long row's entries over
its wave (``csrc/cg.hip``, ``kLong``), the residual of three columns and more over its block
(``csrc/solve.hip``), and the divergence's records are formed a thread a corner. Rows about the lengths
where those start, of a wave's width and past it, several in a wave and a block, more than a block
stages, at each of the instances' sizes.

Bars, as for every iterate: a heat iterate that is accepted passes the solver's own test, a componentwise
backward error of 1e-6 in float64; a Poisson iterate's true residual is within twice the stopping
tolerance 1e-8 of its right-hand side; a repeated solve gives the same bits. Refined factored solves meet their targets, computed here (twice them, for the rounding of
sums of thousands of terms).
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def cone(spokes: int, rings: int):
    """An apex joined to the first of `rings` rings of `spokes` vertices."""
    a = np.arange(spokes) * (2 * np.pi / spokes)
    v = [np.zeros((1, 3))]
    for r in range(1, rings + 1):
        rr = r / rings
        v.append(np.stack([rr * np.cos(a), rr * np.sin(a), np.full(spokes, 0.3 * rr)], 1))
    i, j = np.arange(spokes), (np.arange(spokes) + 1) % spokes
    f = [np.stack([np.zeros(spokes, int), 1 + i, 1 + j], 1)]
    for r in range(1, rings):
        o, p = 1 + (r - 1) * spokes, 1 + r * spokes
        f += [np.stack([o + i, p + i, p + j], 1), np.stack([o + i, p + j, o + j], 1)]
    return np.concatenate(v).astype(np.float32), np.concatenate(f).astype(np.int32)


def _cones(count: int, spokes: int):
    """Fans beside each other, each a component: a hub every `spokes` + 1 rows."""
    v, f = cone(spokes, 1)
    at = np.stack([3.0 * (np.arange(count) % 9), 3.0 * (np.arange(count) // 9), np.zeros(count)], 1)
    vertices = (v[None] + at[:, None].astype(np.float32)).reshape(-1, 3)
    faces = (f[None] + (len(v) * np.arange(count))[:, None, None]).reshape(-1, 3)
    return vertices.astype(np.float32), faces.astype(np.int32)


CASES = {
    "24": lambda: cone(24, 43),  # the longest row 25 entries: its thread's
    "25": lambda: cone(25, 41),  # 26: dealt
    "40": lambda: _cones(60, 40),  # several in a wave, 2,460 rows
    "72": lambda: cone(72, 15),  # 64 entries past those in registers
    "73": lambda: cone(73, 15),
    "600": lambda: cone(600, 20),
    "2000_two_rows": lambda: cone(2000, 40),  # 80,001 rows, two a thread
    "3000_four_rows": lambda: cone(3000, 90),  # 270,001, four
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_iterates_meet_their_stopping_rules(cuda, name):
    from ordito_amd import creation, heat

    v, f = CASES[name]()
    faces = f.reshape(-1)
    n = len(v)
    h = creation.mean_face_edge_length(v, faces)
    source = np.zeros(n)
    source[np.random.default_rng(0).choice(n, 3 + n // 100, replace=False)] = 1.0
    fields, accepted = [], False
    for _ in range(2):
        mesh = heat.Trimesh(v, faces)
        solver = mesh.heat_solver(t=h * h, method="meshlab")
        rhs = cuda.from_numpy(source).cuda()
        out = cuda.empty_like(rhs)
        solver.diffuse(rhs, out)
        assert solver.last_stats["heat_rounds"] > 0
        accepted = not solver.ill_conditioned
        fields.append(out.cpu().numpy())
    assert np.array_equal(fields[0], fields[1])
    assert accepted or int(name.split("_")[0]) > 73  # the finest fans' slivers fall back
    A = solver.operators[0].to_scipy()
    assert np.all(np.abs(source - A @ fields[0]) <= 1e-6 * (abs(A) @ np.abs(fields[0]) + source))

    fields = []
    for _ in range(2):
        mesh = heat.Trimesh(v, faces)
        solver = mesh.heat_solver(t=h * h, method="meshlab")
        L = solver.operators[3].to_scipy()
        b = L @ (np.sin(5.0 * v[:, 0].astype(np.float64)) + v[:, 2])
        rhs = cuda.from_numpy(b).cuda()
        out = cuda.empty_like(rhs)
        solver.solve_poisson(rhs, out)
        assert solver.last_stats["poisson_rounds"] > 0 and solver._factored() == 0
        fields.append(out.cpu().numpy())
    assert np.array_equal(fields[0], fields[1])
    assert np.linalg.norm(b - L @ fields[0]) <= 2e-8 * np.linalg.norm(b)


FACTORED = {
    "63": lambda: cone(63, 9),  # a row of 64 entries
    "64": lambda: cone(64, 9),  # 65: dealt
    "70": lambda: _cones(40, 70),  # several in a block
    "1500": lambda: cone(1500, 3),  # more than a block stages
}


@pytest.mark.parametrize("columns", [3, 4, 5, 20, 63, 64])
@pytest.mark.parametrize("name", sorted(FACTORED))
def test_refined_solves_meet_their_targets(cuda, name, columns):
    """From FP32 blocks, so that every round but the last multiplies a residual."""
    from ordito_amd import heat

    v, f = FACTORED[name]()
    n = len(v)
    mesh = heat.Trimesh(v, f)
    solver = mesh.heat_solver(method="meshlab", precision="mixed")
    assert solver.factor()
    solver.set_refinement(heat=1e-11, poisson=1e-11)
    A, L = solver.operators[0].to_scipy(), solver.operators[3].to_scipy()
    rng = np.random.default_rng(columns)
    b = np.zeros((columns, n))
    b[np.arange(columns), rng.integers(0, n, columns)] = 1.0
    b[0] = 0.0
    b[0, np.diff(A.indptr) > 64] = 1.0  # the hubs themselves
    rhs = cuda.from_numpy(b).cuda()
    out = cuda.empty_like(rhs)
    solver.diffuse(rhs, out)
    assert solver.last_stats["heat_refinements"] > 1
    for x, source in zip(out.cpu().numpy(), b):
        assert np.all(np.abs(source - A @ x) <= 2e-11 * (abs(A) @ np.abs(x) + np.abs(source)))

    b = (L @ rng.standard_normal((n, columns))).T.copy()
    rhs = cuda.from_numpy(b).cuda()
    solver.solve_poisson(rhs, out)
    for x, source in zip(out.cpu().numpy(), b):
        bar = np.maximum(abs(L) @ np.abs(x) + np.abs(source), np.abs(source).max())
        assert np.all(np.abs(source - L @ x) <= 2e-11 * bar)


@pytest.mark.parametrize("name", sorted(FACTORED))
def test_distances_match_the_oracle(cuda, name):
    from oracle import heat_oracle as oracle
    from ordito_amd import heat

    v, f = FACTORED[name]()
    mesh = heat.Trimesh(v, f)
    solver = mesh.heat_solver(method="meshlab")
    assert solver.factor()
    want = oracle.geodesic(v, f.reshape(-1), [1]).distance
    reached = want != 0.0  # other components hold no distance from this source
    reached[1] = True
    for columns in (1, 3, 8):
        sets = [cuda.tensor([1], dtype=cuda.int32, device="cuda")] * columns
        for got in solver.geodesic(sets).cpu().numpy().reshape(columns, -1):
            assert oracle.relative_error(got[reached], want[reached])[0] <= 1e-9
