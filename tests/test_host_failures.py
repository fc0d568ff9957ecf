"""The library's host code on a stand-in for the HIP runtime (fake_hip.c: no
kernel runs): what it leaves behind when an allocation fails, and that copies
keep to their allocations.  Each test is a process of its own, which loads the
stand-in before the library."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PRELUDE = """
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_watch_table.argtypes = fake.fake_launched.argtypes = [ctypes.c_size_t]
sys.path.insert(0, sys.argv[2])
import numpy as np
import sph_amd as A
S, BOX = A.settings(mass=0.02, h=0.1), A.box((-2.0,) * 3, (2.0,) * 3)
def frame(n):
    return A.update_particles(A.make_particles(np.zeros((n, 3), np.float32)), S, 1e-3, BOX)
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    lib = tmp_path_factory.mktemp("fake") / "libfake_hip.so"
    subprocess.run(["gcc", "-O1", "-Wall", "-shared", "-fPIC", "-o", str(lib), os.path.join(HERE, "fake_hip.c")],
                   check=True)
    python = os.path.join(os.path.dirname(HERE), "sph-fluid-simulator_amd", "python")

    def _run(body):
        r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(body), str(lib), python],
                           capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stdout + r.stderr

    return _run


def test_wave_tasks_after_a_failed_allocation(run):
    """Whichever allocation of a larger frame fails, the next frame of the
    former size finds its table of wave tasks on the device."""
    run("""
    n, tasks = 1000, np.array([[0, 64 * k] for k in range(16)], np.uint32)
    fake.fake_watch_table(tasks.nbytes)
    for k in range(1, 200):
        frame(n)
        assert fake.fake_table_holds(A._ptr(tasks)) == 1, ("before", k)
        fake.fake_fail_in(k)
        try:
            frame(20000 + 1024 * k)
        except A.SphError:
            pass
        if fake.fake_pending_failure():  # it made fewer allocations
            break
        frame(n)
        assert fake.fake_table_holds(A._ptr(tasks)) == 1, ("allocation", k)
    assert 20 < k < 199, k
    """)


def test_counters_after_a_failed_allocation(run):
    """... and the larger frame tried again clears the counters its passes
    expect at zero (parts finished, 4 bytes per wave task: the only array of
    that size that a kernel, the clearing one, gets first)."""
    run("""
    for k in range(1, 200):
        n = 100000 + 4096 * k
        fake.fake_fail_in(k)
        try:
            frame(n)
        except A.SphError:
            pass
        if fake.fake_pending_failure():
            break
        frame(n)
        assert fake.fake_launched(4 * ((n + 63) // 64)) == 1, k
    assert 20 < k < 199, k
    """)


def test_downloads_copy_within_their_allocations(run):
    """Records and transforms of n particles, n a multiple of 1024, end on a
    page, and the next allocation may begin there: each is copied by itself
    (16,384: through small pinned memory, 40,960: in pieces)."""
    run("""
    for n in (1024, 2048, 15360, 16384, 40960):
        frame(n)
        pos = np.zeros((n, 3), np.float32)
        with A.Context(n, S, BOX, 1e-3) as c:
            c.upload(pos)
            c.step(1)
            c.download_particles()
            c.download()
        with A.Batch([A.scene_desc(n, S, BOX, 1e-3)] * 2) as b:
            for k in range(2):
                b.upload(k, pos)
            b.step(1)
            b.download_particles(1)
            b.download(1)
    """)
