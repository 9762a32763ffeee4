"""
Calls of several threads on one device (``csrc/flow.hip``, ``WaitClaim``): sweeps of a few columns as one
launch, whose blocks wait for each other, run for one call at a time, the others' level by level, and a
conjugate gradient waits its turn. Each field equals the one its mesh gives alone, whichever way it went;
``igl``'s second heat solve, whose sweeps run beside the first's, and columns that end a wide batch among
them.

Bar: 1e-10 of the range, as between any two direct solves of one system (1e-6 for the iterated call, whose
solver stops at a tolerance).
"""

from __future__ import annotations

import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _jobs():
    from ordito_amd import creation

    torus = creation.torus(300, 150, 1.0, 0.3, 0.1, 3)
    grid = creation.planar_grid(220, 150, 1.0, 0.2, 6)
    sphere = creation.icosphere(5)
    # mesh, method, columns (None: a one-shot call)
    return [(torus, "meshlab", 1), (grid, "igl", 2), (torus, "meshlab", 4), (grid, "igl", 66),
            (sphere, "meshlab", 3), (sphere, "meshlab", None)]


def _call(cuda, job, held):
    from ordito_amd import heat

    (v, f), method, columns = job
    rng = np.random.default_rng(columns or 0)
    sources = [cuda.tensor(rng.integers(0, len(v), 2).astype(np.int32), device="cuda")
               for _ in range(columns or 1)]
    if columns is None:
        return heat.heat_geodesic(v, f, sources[0].cpu().numpy())
    if not held:
        held["mesh"] = heat.Trimesh(v, f)
        held["solver"] = held["mesh"].heat_solver(method=method)
        assert held["solver"].factor()
    return held["solver"].geodesic(sources).cpu().numpy()


@pytest.mark.parametrize("graphs", [True, False])
def test_threads_get_the_fields_of_calls_alone(cuda, graphs):
    jobs = _jobs()
    held = [{} for _ in jobs]
    alone = [np.asarray(_call(cuda, job, h)) for job, h in zip(jobs, held)]
    for h in held:
        if "solver" in h:
            h["solver"].set_graphs(graphs)
    failures = []

    def work(i):
        try:
            with cuda.cuda.stream(cuda.cuda.Stream()):
                for _ in range(2 if jobs[i][2] is None else 12):
                    got = np.asarray(_call(cuda, jobs[i], held[i]))
                    bar = 1e-6 if jobs[i][2] is None else 1e-10
                    worst = np.max(np.abs(got - alone[i])) / np.ptp(alone[i])
                    if not worst <= bar:
                        failures.append((i, worst))
        except Exception as error:  # reported by the test's thread
            failures.append((i, repr(error)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures
