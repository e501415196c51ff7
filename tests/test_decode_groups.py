"""Grouped decode plans (short contexts: one workgroup per row and KV head, its
waves' pieces merged in LDS): the planner's properties on the CPU
(tests/plan/group_plan_check.cpp), and on the MI355X the grouped pass against
the oracle and against the separate split and merge launches
(ORION_DECODE_GROUP=0): alone, and in a model's forward, where past 8 rows every
decode kernel writes the next GEMM's operand in fragment order."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle as orc
import orion_hip as oh
from decode_cases import decode_case
from model_fixtures import oracle_model, random_weights
from paged_cases import PagedCase
from test_gpu_model import batch, gpu_model, rel_err
from test_host_errors import FAKE, fake_hip  # noqa: F401

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


# (rows, head_dim, longest context, kernels of the attention).  Up to 8 rows the
# rows stay f32; 32 tokens a wave is the longest that runs grouped, 256 (row, KV
# head) pairs the most.
GROUPED, SPLIT = ["paged_decode_group_kernel"], ["paged_decode_mfma2_kernel"]
MERGED = ["paged_decode_combine_kernel"] + SPLIT
FORWARDS = [(8, 64, 300, GROUPED), (9, 64, 500, GROUPED), (17, 64, 512, GROUPED),
            (40, 64, 200, GROUPED), (64, 64, 333, GROUPED), (9, 128, 256, GROUPED),
            (33, 128, 129, GROUPED), (9, 64, 513, MERGED), (20, 128, 700, MERGED),
            (64, 128, 300, MERGED), (16, 64, 40, SPLIT), (48, 128, 60, SPLIT)]


def attention_kernels(fake_lib, cases, **env):
    p = subprocess.run([sys.executable, os.path.join(FAKE, "decode_kernels.py"), fake_lib,
                        json.dumps(cases)], capture_output=True, text=True, timeout=120,
                       env=dict(os.environ, **env))
    assert p.returncode == 0, p.stderr
    return [[k for k in json.loads(line) if k.startswith("paged")] for line in p.stdout.splitlines()]


def test_the_forwards_below_run_the_kernels_they_are_for(fake_hip):  # noqa: F811
    cases = [f[:3] for f in FORWARDS]
    assert attention_kernels(fake_hip, cases) == [f[3] for f in FORWARDS]
    split = [MERGED if f[3] == GROUPED else f[3] for f in FORWARDS]
    assert attention_kernels(fake_hip, cases, ORION_DECODE_GROUP="0") == split


@pytest.mark.gpu
@pytest.mark.parametrize("rows,d,longest", [f[:3] for f in FORWARDS])
def test_decode_forward_at_serving_contexts(backend, monkeypatch, rows, d, longest):
    spec, ctxs, tables = decode_case(rows, d, longest)
    W = random_weights(spec, np.random.default_rng(rows + d), std=0.05)
    rng = np.random.default_rng(longest)
    lens = [c - 1 for c in ctxs]
    toks = rng.integers(0, spec.V, sum(lens)).tolist()
    pos = [p for n in lens for p in range(n)]
    nxt = rng.integers(0, spec.V, rows).tolist()
    print(f"[decode forward] rows={rows} d={d} longest={longest}", flush=True)
    om = oracle_model(spec, W, kv_bf16=True)
    om.forward(toks, pos, lens, lens, tables)
    want = om.forward(nxt, lens, [1] * rows, ctxs, tables)
    om.close()
    gm = gpu_model(backend, spec, W, oh.BF16)
    gm.forward(batch(toks, pos, lens, tables))
    got = gm.forward(batch(nxt, lens, [1] * rows, tables, ctxs)).logits
    # the same step without grouping (it rewrites its row of the cache)
    monkeypatch.setenv("ORION_DECODE_GROUP", "0")
    split = gm.forward(batch(nxt, lens, [1] * rows, tables, ctxs)).logits
    gm.close()
    # bf16 KV: a value of K or V may be rounded to the other neighbour (2^-8 of
    # it), in the prompt against the oracle, in one row between the two
    assert rel_err(got, want) <= 2e-2, rel_err(got, want)
    assert [orc.argmax(r) for r in got] == [orc.argmax(r) for r in split]
    assert rel_err(got, split) <= 4e-3, rel_err(got, split)
