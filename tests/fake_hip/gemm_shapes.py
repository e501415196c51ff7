"""The tiled GEMM's workgroup shape and K splits for given calls, from the kernels
launched on the fake runtime.
usage: gemm_shapes.py FAKE_HIP_LIBRARY CALLS, where CALLS is a JSON list of
[M, N, K, epilogue] (op-level calls) and [M, hidden, ffn, hq, hkv, head_dim] (one
prompt of M tokens through a one-layer model).  Prints one JSON line per call:
a list of [column tiles, row tiles, k-steps, splits, x split before, RoPE]."""
import ctypes
import json
import os
import re
import sys

fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_hip_launched.restype = ctypes.c_char_p
ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path.insert(0, os.path.join(ROOT, "orionserve-rs_amd"))

import orion_hip as oh  # noqa: E402

be = oh.HipBackend(0)


def prompt(M, H, F, hq, hkv, d):
    meta = oh.ModelMetadata(hidden_size=H, num_layers=1, num_attention_heads=hq, num_kv_heads=hkv,
                            head_dim=d, vocab_size=64, intermediate_size=F,
                            max_position_embeddings=2048, rope_theta=1.0e4, rms_norm_eps=1e-5,
                            architecture="llama", tied_lm_head=True)
    m = oh.HipTransformerModel(meta, 160, 16, be, oh.BF16)
    m.forward(oh.ForwardBatch([1] * M, list(range(M)), [0], [M], [M],
                              [list(range((M + 15) // 16))], True))
    m.close()


for call in json.loads(sys.argv[2]):
    fake.fake_hip_clear_launched()
    if len(call) == 4:
        M, N, K, ep = call
        oh.gemm(be, 4096, 4096, None, M, N, K, ep, 4096)  # (no kernel reads them here)
    else:
        prompt(*call)
    shapes = []
    for line in fake.fake_hip_launched().decode().splitlines():
        name, z = line.split()
        t = re.search(r"gemm_tiled_kernelILb\dELi(\d+)ELb(\d)ELi(\d+)ELi(\d+)ELb(\d)E", name)
        if t:
            ntw, xs, mtw, st, rope = (int(v) for v in t.groups())
            shapes.append([ntw, mtw, st, int(z), xs, rope])
    print(json.dumps(shapes), flush=True)
