"""The tiled GEMM's choice of workgroup shape and K splits up to 1024 rows, seen on
the CPU through the kernels it launches (tests/fake_hip): against what the shapes
were measured to take on an MI355X, weights not in a cache."""
import json
import os
import subprocess
import sys

import pytest

from test_host_errors import FAKE, fake_hip  # noqa: F401

STORE, ACCUMULATE, SWIGLU = 0, 1, 2
QWEN, LLAMA = (3584, 18944, 28, 4, 128), (4096, 14336, 32, 8, 128)

# (call, which tiled GEMM of it, us of (column tiles, row tiles, k-steps in LDS,
# splits)).  Calls of [M, N, K, epilogue] take f32 activations; the others are
# prompts of M tokens through a layer: its QKV (0) and gate/up (2) GEMMs.
MEASURED = [
    ([320, 37888, 3584, SWIGLU], 0, {(8, 4, 2, 1): 204, (4, 3, 2, 1): 234, (4, 2, 4, 1): 235,
        (4, 4, 2, 1): 244, (4, 4, 3, 1): 246, (4, 3, 3, 1): 269}),
    ([450, 32000, 2048, STORE], 0, {(8, 4, 2, 1): 131, (4, 3, 2, 1): 153, (4, 4, 2, 1): 154,
        (4, 4, 3, 1): 159, (8, 4, 2, 2): 162, (4, 4, 2, 2): 168}),
    ([1000, 32000, 2048, STORE], 0, {(8, 4, 2, 1): 248, (4, 3, 2, 1): 287, (4, 4, 2, 1): 293,
        (4, 4, 3, 1): 308, (4, 3, 3, 1): 344, (4, 2, 4, 1): 351}),
    ([512, 28672, 4096, STORE], 0, {(8, 4, 2, 1): 230, (8, 4, 2, 2): 268, (4, 4, 2, 2): 272,
        (4, 4, 2, 1): 274, (4, 4, 3, 1): 280, (4, 4, 3, 2): 291}),
    ([640, 2048, 2048, ACCUMULATE], 0, {(4, 3, 2, 4): 27.2, (4, 3, 3, 4): 28.3, (4, 2, 4, 2): 28.8,
        (4, 4, 2, 4): 29.8, (4, 5, 3, 4): 30.0, (4, 4, 2, 1): 54.5}),
    ([512, 2560, 2048, STORE], 0, {(4, 3, 2, 4): 27.2, (4, 3, 3, 4): 28.0, (4, 2, 4, 2): 28.1,
        (4, 4, 2, 4): 29.2, (4, 4, 3, 4): 30.1, (4, 4, 2, 1): 56.6}),
    ([320, *QWEN], 2, {(8, 4, 2, 1): 175, (4, 4, 3, 1): 191, (4, 3, 3, 1): 200, (4, 2, 4, 1): 201,
        (4, 3, 2, 1): 205, (4, 4, 2, 1): 216}),
    ([640, *QWEN], 2, {(8, 4, 2, 1): 288, (4, 4, 2, 1): 304, (4, 4, 3, 1): 311, (4, 3, 2, 1): 337,
        (4, 3, 3, 1): 349, (4, 2, 4, 1): 356}),
    ([743, *LLAMA], 2, {(4, 3, 2, 1): 294, (8, 4, 2, 1): 309, (4, 4, 2, 1): 323, (4, 3, 3, 1): 324,
        (4, 4, 3, 1): 329, (4, 2, 4, 1): 356}),
    ([743, *LLAMA], 0, {(4, 3, 3, 1): 83.3, (4, 5, 3, 1): 93.3, (4, 4, 3, 1): 99.2,
        (4, 3, 2, 1): 101, (4, 2, 4, 1): 106, (4, 4, 2, 1): 107}),
]


@pytest.fixture(scope="module")
def chosen(fake_hip):  # noqa: F811
    p = subprocess.run([sys.executable, os.path.join(FAKE, "gemm_shapes.py"), fake_hip,
                        json.dumps([call for call, _, _ in MEASURED])],
                       capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stderr
    return [json.loads(line) for line in p.stdout.splitlines()]


@pytest.mark.parametrize("i", range(len(MEASURED)), ids=lambda i: f"{MEASURED[i][0]}-{MEASURED[i][1]}")
def test_the_shape_is_near_the_fastest(chosen, i):
    call, which, us = MEASURED[i]
    ntw, mtw, st, splits, presplit, rope = chosen[i][which]
    assert (presplit, rope) == ((0, 0) if len(call) == 4 else (1, int(which == 0)))
    # (shapes not listed were slower than those that are)
    assert us.get((ntw, mtw, st, splits), 1e9) <= 1.05 * min(us.values()), (ntw, mtw, st, splits)
