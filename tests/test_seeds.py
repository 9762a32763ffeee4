"""
The seeds of fields stored by rows (``csrc/assembly.hip``): one launch that clears and seeds up to 4,096
sources, a clear and a launch beyond, and the bitmap of seeded rows that the heat step's residual reads
its right-hand side by. Row counts off a multiple of 32 and below it, 1 to 65 columns, repeated and empty
sets, every vertex a source, and sources out of range on both paths.

Bar: 1e-9 of the range against the oracle, as for every direct query.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import heat_oracle as oracle

pytestmark = pytest.mark.gpu


def _mesh(name):
    from ordito_amd import creation

    return {"tiny": creation.planar_grid(5, 4, 1.0, 0.2, 6),
            "grid": creation.planar_grid(61, 47, 1.0, 0.2, 6)}[name]


@pytest.mark.parametrize("name", ["tiny", "grid"])
@pytest.mark.parametrize("columns,each", [(1, 1), (5, 3), (6, 900), (64, 2), (64, 70), (65, 63), (65, 64)])
def test_columns_match_the_oracle(cuda, name, columns, each):
    from ordito_amd import heat

    v, f = _mesh(name)
    mesh = heat.Trimesh(v, f)
    solver = mesh.heat_solver(method="meshlab")
    assert solver.factor()
    rng = np.random.default_rng(columns + each)
    sets = [rng.integers(0, len(v), each).astype(np.int32) for _ in range(columns)]
    if columns > 1:
        sets[1] = np.arange(len(v), dtype=np.int32)
        sets[2] = np.asarray([], np.int32)
    for _ in range(2):  # the second call's field starts from the first's
        got = solver.geodesic([cuda.tensor(s, dtype=cuda.int32, device="cuda") for s in sets])
        got = got.cpu().numpy().reshape(columns, len(v))
        for c in sorted({0, columns - 1}):
            want = oracle.geodesic(v, f, sets[c]).distance
            assert oracle.relative_error(got[c], want)[0] <= 1e-9, c
        sets = sets[::-1]


@pytest.mark.parametrize("entries", [1, 4096, 5000])
@pytest.mark.parametrize("bad", [-1, 2867])
def test_a_source_out_of_range_fails_the_call(cuda, entries, bad):
    from ordito_amd import heat

    v, f = _mesh("grid")
    assert len(v) == 2867
    mesh = heat.Trimesh(v, f)
    solver = mesh.heat_solver(method="meshlab")
    assert solver.factor()
    good = np.arange(entries, dtype=np.int32) % len(v)
    wrong = good.copy()
    wrong[-1] = bad
    for values, fails in ((wrong, True), (good, False)):
        sources = [cuda.tensor(values, dtype=cuda.int32, device="cuda")]
        if fails:
            with pytest.raises(ValueError):
                solver.geodesic(sources)
        else:
            assert np.isfinite(solver.geodesic(sources).cpu().numpy()).all()
