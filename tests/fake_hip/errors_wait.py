"""Fails each HIP call of a forward, of a sampler call and of making a decode plan in
turn, on the fake runtime, and prints what was still queued when the call returned
(the staging areas it reads are then overwritten or freed).
usage: errors_wait.py FAKE_HIP_LIBRARY"""
import ctypes
import os
import sys

fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path.insert(0, os.path.join(ROOT, "orionserve-rs_amd"))

import numpy as np  # noqa: E402
import orion_hip as oh  # noqa: E402

META = oh.ModelMetadata(hidden_size=256, num_layers=2, num_attention_heads=4, num_kv_heads=2,
                        head_dim=64, vocab_size=1000, intermediate_size=512,
                        max_position_embeddings=1024, rope_theta=1.0e4, rms_norm_eps=1e-5,
                        architecture="llama", tied_lm_head=True)


def decode(rows, context):
    tables = [[(r * 40 + j) % 4096 for j in range((context + 15) // 16)] for r in range(rows)]
    return oh.ForwardBatch([1] * rows, [context - 1] * rows, list(range(rows)), [1] * rows,
                           [context] * rows, tables, False)


def prompt(tokens):
    return oh.ForwardBatch([1] * tokens, list(range(tokens)), [0], [tokens], [tokens],
                           [list(range((tokens + 15) // 16))], True)


def forward(*batches):
    def run():
        be = oh.HipBackend(0)
        m = oh.HipTransformerModel(META, 4096, 16, be, oh.BF16)
        try:
            for b in batches:
                m.forward(b, want_argmax=True)
        finally:
            results.append(fake.fake_hip_queued())
            m.close()
            be.close()
    return run


def sample():
    be = oh.HipBackend(0)
    logits = be.alloc(4 * 1000 * 4)
    try:
        oh.sample(be, logits.ptr, 4, 1000, [oh.SamplingParams(temperature=1.0)] * 4,
                  [np.array([1, 2], np.uint32)] * 4, np.full(4, 0.5, np.float32))
    finally:
        results.append(fake.fake_hip_queued())
        be.close()


def plan():
    be = oh.HipBackend(0)
    logits = be.alloc(1000 * 4)
    try:
        # (the sampler's pinned memory: from here on queued work is counted)
        oh.sample(be, logits.ptr, 1, 1000, [oh.SamplingParams(temperature=1.0)],
                  [np.array([], np.uint32)], np.full(1, 0.5, np.float32))
        oh.DecodePlan(be, [299], np.zeros(1, np.int32), np.array([0, 19]), np.arange(19), 32, 4, 64,
                      16).close()
    finally:
        results.append(fake.fake_hip_queued())
        be.close()


for name, run in [("decode 1 row", forward(decode(1, 40))),
                  ("decode 9 rows, then longer", forward(decode(9, 30), decode(40, 600))),
                  ("decode 96 rows", forward(decode(96, 100))),
                  ("prompt", forward(prompt(300))), ("sample", sample), ("plan", plan)]:
    results = []
    fake.fake_hip_fail_at(0)
    run()
    calls, bad, refused = fake.fake_hip_calls(), [], 0
    for n in range(1, calls + 1):
        fake.fake_hip_fail_at(n)
        results = []
        try:
            run()
        except oh.EngineError:
            refused += 1
        if results and results[0]:
            bad.append((n, results[0]))
        fake.fake_hip_fail_at(0)
    print(f"{name}: {calls} calls, {refused} errors, {len(bad)} left queued {bad[:5]}", flush=True)
