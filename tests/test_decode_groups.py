"""Grouped decode plans (short contexts: one workgroup per row and KV head, its
waves' pieces merged in LDS): the planner's properties on the CPU
(tests/plan/group_plan_check.cpp), and on the MI355X the grouped pass against
the oracle and against the separate split and merge launches
(ORION_DECODE_GROUP=0)."""
import os
import subprocess

import numpy as np
import pytest

from paged_cases import PagedCase

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "orionserve-rs_amd", "csrc")


def test_grouped_plans_cover_every_context_once(tmp_path):
    exe = str(tmp_path / "group_plan_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + CSRC, os.path.join(ROOT, "tests", "plan", "group_plan_check.cpp"),
                    os.path.join(CSRC, "decode_plan.cpp"), "-o", exe], check=True)
    p = subprocess.run([exe, "3000"], capture_output=True, text=True)
    assert p.returncode == 0, p.stdout
    assert int(p.stdout.split()[2]) > 300  # grouped plans were built and checked


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,G,d,bs,head_major", [
    ("bf16", 8, 64, 16, False), ("bf16", 1, 64, 8, True), ("bf16", 5, 64, 32, False),
    ("bf16", 4, 128, 16, True), ("bf16", 7, 128, 4, False), ("bf16", 8, 128, 32, False),
    ("f32", 4, 64, 16, False), ("f32", 1, 64, 4, True), ("f32", 8, 64, 16, False),
    ("f32", 5, 64, 32, True)])
def test_grouped_decode_matches_oracle_and_split(backend, monkeypatch, dtype, G, d, bs, head_major):
    from test_gpu_attention import run_decode

    longest = 512 if d == 64 and (dtype == "bf16" or G <= 4) else 256  # 32 tokens a wave
    ctxs = [longest, 1, 15, 16, 17, 63, 64, 65, longest - 1, longest // 2 + 3]
    case = PagedCase(G * d + bs, ctxs, 2 * G, 2, d, bs, dtype=dtype, pool_factor=1.25,
                     head_major=head_major)
    got = run_decode(backend, case)
    want = case.oracle()
    # f32 accumulation over exact operands; bf16 arenas split Q and P to 16 bits
    assert np.abs(got - want).max() <= (2e-6 if dtype == "f32" else 1e-4)
    monkeypatch.setenv("ORION_DECODE_GROUP", "0")
    split = run_decode(backend, case)
    monkeypatch.delenv("ORION_DECODE_GROUP")
    # other piece boundaries only
    assert np.abs(got - split).max() <= (2e-6 if dtype == "f32" else 2e-5)
