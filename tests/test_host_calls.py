"""
The library's host code with a HIP runtime that only keeps memory and a log of launches
(``tests/fake_hip.cpp``): what a call allocates and launches, in what order and beside which other
calls, where no GPU is needed to tell. Kernels do nothing there, so device memory stays zero and a
mesh's pattern is empty; the solves' sequences of launches are the real ones.

Each test runs in a process of its own, which binds the library to that runtime.
"""

from __future__ import annotations

import contextlib
import ctypes
import subprocess
import sys
import threading
from pathlib import Path

import numpy as np

ROOT = Path(__file__).resolve().parents[1]
HEAT, POISSON = 1, 2
ITERATE, FACTORED = 0, 1


class Library:
    """libheatgeo over the fake runtime; a call that fails raises its message."""

    def __init__(self, fake: str) -> None:
        self.fake = ctypes.CDLL(fake, mode=ctypes.RTLD_GLOBAL)
        self.lib = ctypes.CDLL(str(ROOT / "ordito_amd" / "libheatgeo.so"))
        self.lib.hg_last_error.restype = ctypes.c_char_p
        for name in ("fake_live_bytes", "fake_launches", "fake_thread_launches"):
            getattr(self.fake, name).restype = ctypes.c_long

    def call(self, name: str, *args) -> None:
        values = [a.ctypes.data_as(ctypes.c_void_p) if isinstance(a, np.ndarray)
                  else ctypes.c_int64(a) if isinstance(a, int) else a for a in args]
        if getattr(self.lib, name)(*values):
            raise RuntimeError(self.lib.hg_last_error().decode())

    def launches(self, part: str) -> int:
        return self.fake.fake_launches(part.encode())

    def mesh(self, n: int) -> ctypes.c_void_p:
        xyz = np.random.default_rng(n).random((n, 3), dtype=np.float32)
        faces = (np.arange(3 * n, dtype=np.int32) % n)
        handle = ctypes.c_void_p()
        self.call("hg_mesh_create", xyz, n, faces, n, None, ctypes.byref(handle))
        return handle

    def geodesic(self, mesh, n: int, columns: int, mode: int = FACTORED) -> None:
        sources = np.zeros(columns, np.int32)
        out = np.zeros((columns, n))
        self.call("hg_geodesic", mesh, sources, np.arange(columns + 1), columns, out, mode, 0, None)

    def diffuse(self, mesh, n: int, columns: int) -> None:
        fields = np.zeros((2, columns, n))
        self.call("hg_diffuse", mesh, fields[0], fields[1], columns, ITERATE, 0, None)

    def solve_poisson(self, mesh, n: int, columns: int) -> None:
        fields = np.zeros((2, columns, n))
        self.call("hg_solve_poisson", mesh, fields[0], fields[1], columns, ITERATE, 0)

    def device_bytes(self, mesh) -> int:
        out = ctypes.c_int64()
        self.call("hg_device_bytes", mesh, ctypes.byref(out))
        return out.value


def _alone(name: str, tmp_path) -> None:
    fake = tmp_path / "fake_hip.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", str(ROOT / "tests" / "fake_hip.cpp"), "-o", str(fake)],
                   check=True)
    run = subprocess.run([sys.executable, __file__, name, str(fake)], capture_output=True, text=True,
                         timeout=100)
    assert run.returncode == 0, run.stdout + run.stderr


def _failing(lib: Library, attempt) -> None:
    """`attempt` with each of its allocations failing in turn: `attempt(None)` is one that may fail,
    `attempt(error)` what must hold after it did."""
    for n in range(1, 1000):
        state = attempt(None)
        lib.fake.fake_fail_allocation(n)
        try:
            state()
            error = None
        except RuntimeError as raised:
            error = str(raised)
        if lib.fake.fake_failure_pending():
            assert error is None and n > 1
            return
        # (A capture that runs out of memory falls back to an eager solve.)
        assert error is None or "out of memory" in error, (n, error)
        attempt(n)
    raise AssertionError("the call never ran out of allocations")


@contextlib.contextmanager
def _held(lib: Library, kernel: str, call):
    """`call` running on another thread, held where it launches `kernel` until the block ends."""
    failures = []

    def work():
        try:
            call()
        except Exception as error:  # reported by the test's thread
            failures.append(error)

    lib.fake.fake_gate(kernel.encode())
    thread = threading.Thread(target=work)
    thread.start()
    try:
        assert lib.fake.fake_held(), f"{kernel} was not launched {failures}"
        yield
        assert thread.is_alive()
    finally:
        lib.fake.fake_open()
        thread.join(20)
    assert not thread.is_alive() and not failures, failures


def _beside(call, seconds: float = 20.0) -> dict:
    """`call` on a thread of its own: what it returned, or that it did not end in time."""
    out = {}

    def work():
        try:
            out["value"] = call()
        except Exception as error:  # reported by the test's thread
            out["error"] = error

    thread = threading.Thread(target=work, daemon=True)
    thread.start()
    thread.join(seconds)
    out["ended"] = not thread.is_alive()
    out["thread"] = thread
    assert "error" not in out, out["error"]
    return out


def iterations_of_one_block_run_beside_others(lib: Library) -> None:
    """Conjugate gradients of one block wait for no other block, so they run whatever else does; two
    of several blocks take turns."""
    large, other, small, middle = (lib.mesh(n) for n in (2000, 2100, 300, 3000))
    with _held(lib, "cg_resident_kernel", lambda: lib.solve_poisson(large, 2000, 1)):
        assert _beside(lambda: lib.diffuse(small, 300, 1))["ended"]
        assert _beside(lambda: lib.solve_poisson(small, 300, 1))["ended"]
        assert _beside(lambda: lib.diffuse(middle, 3000, 4))["ended"]
        waits = _beside(lambda: lib.solve_poisson(other, 2100, 1), 0.3)
        assert not waits["ended"]
    waits["thread"].join(20)
    assert not waits["thread"].is_alive()


def preparation_leaves_the_device_unclaimed(lib: Library) -> None:
    """Only solves keep others from sweeping in one launch: not a call that is still factoring, nor
    one that iterates."""
    small, large, fresh = lib.mesh(300), lib.mesh(2000), lib.mesh(400)

    def swept() -> int:
        before = lib.fake.fake_thread_launches(b"flow_kernel")
        fields = np.zeros((2, 1, 300))
        lib.call("hg_diffuse", small, fields[0], fields[1], 1, FACTORED, 0, None)
        return lib.fake.fake_thread_launches(b"flow_kernel") - before

    def iterates():
        lib.solve_poisson(large, 2000, 1)

    assert swept() == 1
    for kernel, call in (("panel_diag", lambda: lib.geodesic(fresh, 400, 1)),
                         ("cg_resident_kernel", lambda: lib.geodesic(lib.mesh(500), 500, 1, ITERATE))):
        with _held(lib, kernel, call):
            assert _beside(swept)["value"] == 1, kernel
            assert _beside(iterates)["ended"], kernel
    # One that does hold the claim: a sweep in one launch, and a solve of several blocks.
    for kernel, call in (("flow_kernel", lambda: lib.geodesic(fresh, 400, 2)),
                         ("cg_resident_kernel", iterates)):
        with _held(lib, kernel, call):
            assert _beside(swept)["value"] == 0, kernel
    assert swept() == 1


def workspaces_after_a_failed_allocation(lib: Library) -> None:
    """A call that could not allocate says so, holds no more than the mesh counts, and leaves
    workspaces that a narrower call can trust: none of theirs is missing."""
    n = 300
    held = {}

    def attempt(failed):
        if failed is None:
            held["mesh"] = lib.mesh(n)
            lib.geodesic(held["mesh"], n, 1)
            lib.diffuse(held["mesh"], n, 2)
            held["bytes"] = lib.device_bytes(held["mesh"])

            def wide():
                lib.geodesic(held["mesh"], n, 4)
                lib.call("hg_release", held["mesh"])
                lib.diffuse(held["mesh"], n, 3)

            return wide
        assert lib.device_bytes(held["mesh"]) <= lib.fake.fake_live_bytes(), failed
        lib.geodesic(held["mesh"], n, 1)
        lib.call("hg_release", held["mesh"])
        lib.diffuse(held["mesh"], n, 2)
        lib.geodesic(held["mesh"], n, 1)
        assert lib.device_bytes(held["mesh"]) >= held["bytes"], failed
        lib.call("hg_mesh_destroy", held["mesh"])
        return None

    _failing(lib, attempt)


def server_after_a_failed_allocation(lib: Library) -> None:
    """A query that a worker's buffers could not grow for fails alone: the next one is answered."""
    n = 300
    xyz = np.random.default_rng(n).random((n, 3), dtype=np.float32)
    faces = np.arange(3 * n, dtype=np.int32) % n
    out = np.zeros(n)
    held = {}

    def query():
        ticket, done = ctypes.c_int64(), ctypes.c_int32()
        sources = np.zeros(2000, np.int32)
        lib.call("hg_server_submit", held["server"], held["id"].value, sources, len(sources), out,
                 ctypes.byref(ticket))
        lib.call("hg_server_wait", held["server"], ticket.value, ctypes.c_double(20000.0),
                 ctypes.byref(done))
        assert done.value

    def attempt(failed):
        if failed is None:
            server, held["id"] = ctypes.c_void_p(), ctypes.c_int64()
            lib.call("hg_server_create", 1 << 40, 1, 8, 0, ctypes.byref(server))
            held["server"] = server
            lib.call("hg_server_add_mesh", server, xyz, n, faces, n, ctypes.byref(held["id"]))
            return query
        query()
        lib.call("hg_server_destroy", held["server"])
        return None

    _failing(lib, attempt)


def row_order_after_a_failed_allocation(lib: Library) -> None:
    """A solve whose state stays on the chip indexes by the rows' order, which must have been built."""
    n = 2000
    held = {}

    def attempt(failed):
        if failed is None:
            held["mesh"] = lib.mesh(n)
            held["inverted"] = lib.launches("invert_kernel")
            return lambda: lib.solve_poisson(held["mesh"], n, 1)
        solves = lib.launches("cg_resident_kernel")
        lib.solve_poisson(held["mesh"], n, 1)
        assert lib.launches("cg_resident_kernel") == solves + 1, failed
        assert lib.launches("invert_kernel") > held["inverted"], failed
        lib.call("hg_mesh_destroy", held["mesh"])
        return None

    _failing(lib, attempt)


def a_wait_is_bounded(lib: Library) -> None:
    """The waits count their polls in 32 bits: a patience such a count cannot pass is refused."""
    mesh = lib.mesh(300)
    for polls in (0, 1 << 21, 2**31 - 2):
        lib.call("hg_set_sweep_patience", mesh, polls)
    for polls in (-1, 2**31 - 1, 2**31, 1 << 40, 2**63 - 1):
        try:
            lib.call("hg_set_sweep_patience", mesh, polls)
        except RuntimeError as error:
            assert "2147483646" in str(error)
        else:
            raise AssertionError(f"{polls} polls accepted")


def test_workspaces_after_a_failed_allocation(tmp_path):
    _alone("workspaces_after_a_failed_allocation", tmp_path)


def test_server_after_a_failed_allocation(tmp_path):
    _alone("server_after_a_failed_allocation", tmp_path)


def test_row_order_after_a_failed_allocation(tmp_path):
    _alone("row_order_after_a_failed_allocation", tmp_path)


def test_a_wait_is_bounded(tmp_path):
    _alone("a_wait_is_bounded", tmp_path)


def test_iterations_of_one_block_run_beside_others(tmp_path):
    _alone("iterations_of_one_block_run_beside_others", tmp_path)


def test_preparation_leaves_the_device_unclaimed(tmp_path):
    _alone("preparation_leaves_the_device_unclaimed", tmp_path)


if __name__ == "__main__":
    globals()[sys.argv[1]](Library(sys.argv[2]))
