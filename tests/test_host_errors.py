"""The library's host code on a HIP runtime without a GPU
(tests/fake_hip/fake_hip.cpp): what it leaves behind when a HIP call fails."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
FAKE = os.path.join(HERE, "fake_hip")


@pytest.fixture(scope="module")
def fake_hip(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-shared", "-fPIC", os.path.join(FAKE, "fake_hip.cpp"), "-o", lib], check=True)
    return lib


def test_every_error_waits_for_the_staging_areas(fake_hip):
    # each HIP call of a forward and a sampler call fails in turn: the call
    # reports it, and no work that may read the pinned staging areas, which the
    # next call writes, is still queued
    p = subprocess.run([sys.executable, os.path.join(FAKE, "errors_wait.py"), fake_hip],
                       capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stderr
    lines = p.stdout.splitlines()
    assert len(lines) == 5, p.stdout
    for line in lines:
        calls, errors, left = [int(part.split()[0]) for part in line.split(": ")[1].split(", ")[:3]]
        assert calls == errors and left == 0, line
