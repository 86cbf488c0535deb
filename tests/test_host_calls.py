"""The library's host side without a GPU: tests/cpp/host_calls_test.cpp stands in for the HIP runtime,
runs no kernel and notes what the library queues and allocates."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXE = os.path.join(ROOT, "tests", "cpp", "host_calls_test")


@pytest.mark.skipif(not os.path.exists(EXE), reason="host call test not built")
@pytest.mark.parametrize("check", ["--failed-step", "--create"])
def test_host_calls(check):
    r = subprocess.run([EXE, check], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
