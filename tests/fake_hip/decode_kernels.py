"""The kernels of one decode forward on the fake runtime, by name.
usage: decode_kernels.py FAKE_HIP_LIBRARY CASES, where CASES is a JSON list of
[rows, head_dim, longest context]; prints one JSON line per case."""
import ctypes
import json
import os
import re
import sys

fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_hip_launched.restype = ctypes.c_char_p
TESTS = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROOT = os.path.dirname(TESTS)
sys.path[:0] = [os.path.join(ROOT, "orionserve-rs_amd"), ROOT, TESTS]

import orion_hip as oh  # noqa: E402
from decode_cases import decode_case  # noqa: E402

be = oh.HipBackend(0)
for rows, d, longest in json.loads(sys.argv[2]):
    spec, ctxs, tables = decode_case(rows, d, longest)
    meta = oh.ModelMetadata(hidden_size=spec.H, num_layers=spec.L, num_attention_heads=spec.hq,
                            num_kv_heads=spec.hkv, head_dim=spec.d, vocab_size=spec.V,
                            intermediate_size=spec.F, max_position_embeddings=spec.max_pos,
                            rope_theta=spec.theta, rms_norm_eps=spec.eps, architecture="llama",
                            tied_lm_head=spec.tied)
    m = oh.HipTransformerModel(meta, spec.num_blocks, spec.block_size, be, oh.BF16)
    fake.fake_hip_clear_launched()
    m.forward(oh.ForwardBatch([1] * rows, [c - 1 for c in ctxs], list(range(rows)), [1] * rows, ctxs,
                              tables, False))
    names = re.findall(r"\d+(paged_\w*?kernel|gemm_\w*?kernel)", fake.fake_hip_launched().decode())
    print(json.dumps(sorted(set(names))), flush=True)
    m.close()
