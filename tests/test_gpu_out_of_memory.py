"""Calls that find no device memory: every device allocation of a call fails in turn, in a
process of its own whose hipMalloc is the test's (device_oom/fail_malloc.cpp).  The call does
without that memory or reports BLEST_ERR_OUT_OF_DEVICE_MEMORY, and the handles it worked on
give the oracle's results afterwards."""
import subprocess
import sys
from pathlib import Path

import pytest
from conftest import progress

pytestmark = pytest.mark.gpu

HERE = Path(__file__).resolve().parent / "device_oom"


@pytest.fixture(scope="module")
def fail_malloc(tmp_path_factory):
    lib = tmp_path_factory.mktemp("oom") / "libfail_malloc.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", str(HERE / "fail_malloc.cpp"), "-o", str(lib), "-ldl"],
                   check=True)
    return lib


@pytest.mark.parametrize("group", ["query_state", "creation", "construction"])
def test_failed_allocations(fail_malloc, group):
    progress(f"case failed allocations {group}")
    r = subprocess.run([sys.executable, "-u", str(HERE / "child.py"), str(fail_malloc), group], capture_output=True,
                       text=True, timeout=110)
    assert r.returncode == 0 and "OOM GROUP OK" in r.stdout, (r.stdout + r.stderr)[-4000:]
