"""Host parts of the library that the C ABI does not show
(tests/host_checks.cpp): the check that the near field's items cover every
pair and target."""
import ctypes
import os
import subprocess

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


def test_items_cover_check(checks):
    assert checks.check_cover() == 0
