"""The library's host code on a HIP runtime without a GPU
(tests/fake_hip/fake_hip.cpp): what it leaves behind when a HIP call fails, and what
a decode plan costs."""
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
    # each HIP call of a forward, a sampler call and a plan's making fails in turn:
    # the call reports it, and no work that may read the staging areas, which are
    # then written or freed, is still queued
    p = subprocess.run([sys.executable, os.path.join(FAKE, "errors_wait.py"), fake_hip],
                       capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stderr
    lines = p.stdout.splitlines()
    assert len(lines) == 6, p.stdout
    for line in lines:
        calls, errors, left = [int(part.split()[0]) for part in line.split(": ")[1].split(", ")[:3]]
        assert calls == errors and left == 0, line


# a plan of short rows (a group per arena type), of long ones, of a shared prefix
PLANS = """
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
import numpy as np, orion_hip as oh
be = oh.HipBackend(0)
for context, shared in [(300, 0), (3000, 0), (3000, 128)]:
    n = (context + 15) // 16
    ids = np.arange(4 * n, dtype=np.uint32).reshape(4, n)
    ids[:, :shared] = ids[0, :shared]
    before = fake.fake_hip_mallocs(), fake.fake_hip_copies()
    plan = oh.DecodePlan(be, [context - 1] * 4, np.arange(4), np.arange(5) * n, ids.reshape(-1), 32,
                         4, 64, 16)
    print(fake.fake_hip_mallocs() - before[0], fake.fake_hip_copies() - before[1],
          plan.info()["packed_items"] > 0)
    plan.close()
"""


def test_a_plan_is_one_list_buffer_and_one_copy(fake_hip):
    # what a program that plans each step pays: the lists (for both arena types
    # where they differ) in one allocation and one copy, and the workspace
    pkg = os.path.join(os.path.dirname(HERE), "orionserve-rs_amd")
    p = subprocess.run([sys.executable, "-c", PLANS, fake_hip, pkg], capture_output=True, text=True,
                       timeout=120)
    assert p.returncode == 0, p.stderr
    assert p.stdout.splitlines() == ["2 1 False", "2 1 False", "2 1 True"]
