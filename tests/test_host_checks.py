"""Host parts of the library that the C ABI does not show
(tests/host_checks.cpp): the interaction lists, entry by entry in order,
against the reference's walks in one thread, the check that the near
field's items cover every pair and target, and that a call uses the threads
that are there."""
import ctypes
import os
import subprocess
import threading

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def checks(tmp_path_factory):
    import barytree_amd
    if not os.path.exists(barytree_amd.LIB_PATH):
        from barytree_amd import build
        build.build()
    out = str(tmp_path_factory.mktemp("host_checks") / "libhost_checks.so")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    lib = os.path.abspath(barytree_amd.LIB_PATH)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-std=c++17", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__",
                    f"-I{rocm}/include", os.path.join(ROOT, "tests", "host_checks.cpp"), lib,
                    f"-Wl,-rpath,{os.path.dirname(lib)}", "-o", out], check=True, capture_output=True)
    return ctypes.CDLL(out)


@pytest.mark.parametrize("cc", [0, 1])
@pytest.mark.parametrize("n,m", [(9000, 9000), (20000, 300), (300, 20000)])
@pytest.mark.parametrize("degree", [1, 3])
def test_lists_have_the_order_of_one_walk(checks, cc, n, m, degree):
    """Trees above 1024 nodes, whose lists several threads write: sums run
    over the lists and pairs are numbered by them, so the order counts."""
    rng = np.random.default_rng(n + m)
    dp = lambda a: a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))  # noqa: E731
    pts = [np.sign(u) * np.abs(u) ** rng.uniform(2.0, 4.0)
           for u in (rng.uniform(-1, 1, k) for k in (n, n, n, m, m, m))]
    keys = ctypes.c_int(0)
    bad = checks.check_lists(ctypes.c_int(cc), ctypes.c_int(n), *map(dp, pts[:3]), ctypes.c_int(m), *map(dp, pts[3:]),
                             ctypes.c_double(0.7), ctypes.c_int(degree), ctypes.c_int(6), ctypes.byref(keys))
    assert bad == 0
    assert m < 9000 or keys.value > 1024


def test_items_cover_check(checks):
    assert checks.check_cover() == 0


def next_thread_id():
    """The id of a thread started now; ids are given in sequence."""
    out = []
    t = threading.Thread(target=lambda: out.append(threading.get_native_id()))
    t.start()
    t.join()
    return out[0]


@pytest.mark.parametrize("ct", [1, 2, 3])
def test_a_call_starts_no_threads(checks, ct):
    """Plans of one system, once the first call has started the threads of its
    parallel loops: later calls start none (the least of several calls, for
    other processes take ids too).  A parallel region within another starts
    its threads anew each time, which costs milliseconds and now and then
    tens of them."""
    import barytree_amd as bt
    from tests.helpers import uniform_cube
    t, s = uniform_cube(12000, 12000, seed=ct)
    started = []
    for _ in range(8):
        before = next_thread_id()
        a = bt.analyze(t, s, 1, [0.5], 1, 1, ct, 0.7, 1, 6, 6)
        started.append(next_thread_id() - before - 1)
    assert max(a["source_nodes"], a["target_nodes"]) > 1024
    assert min(started[1:]) == 0, started
