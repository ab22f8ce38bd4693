"""Result entries of the build server's slots (csrc/result_ring.h): requests in
flight never share one, also past requests that failed before they got to the
slot (tests/cpp/result_ring_test.cc, on the CPU)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_requests_in_flight_have_entries_of_their_own(tmp_path):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "result_ring_test")
    subprocess.run([gxx, "-O1", "-std=c++17", "-Wall", "-Wextra", "-Werror",
                    "-I", os.path.join(ROOT, "webgpu-lvbh-demo_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "result_ring_test.cc"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip() == "ok"
