"""The decode route's projections on the MI355X (launch_gemm_rows: whole K per
workgroup, RMSNorm and RoPE + KV write inside, activations as f32 rows or in
fragment order) through the model forward, against the CPU oracle: row counts
around its 8-row and 16-row edges, widths with a partial column tile, a K long
enough to be split over workgroups, and heads that are not whole 16-column
tiles (their RoPE is a launch of its own)."""
import numpy as np
import pytest

import oracle as orc
import orion_hip as oh
from model_fixtures import Spec, oracle_model, random_weights
from test_gpu_model import batch, gpu_model, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,H,F,hq,hkv,d,V", [
    (1, 256, 2048, 4, 2, 64, 517), (8, 96, 160, 4, 1, 24, 33), (9, 256, 352, 4, 2, 64, 1000),
    (16, 160, 2048, 5, 1, 32, 517), (17, 256, 352, 2, 1, 128, 130), (33, 320, 2080, 4, 2, 80, 515),
    (48, 256, 4128, 8, 2, 32, 700), (49, 96, 1056, 4, 2, 24, 257), (64, 512, 4096, 8, 8, 64, 4100)])
def test_decode_rows_match_oracle(backend, S, H, F, hq, hkv, d, V):
    rng = np.random.default_rng(S * H + F)
    spec = Spec(2, H, hq, hkv, d, F, V, max_pos=64, bias=S % 2 == 0, tied=S % 3 == 0,
                num_blocks=2 * S, block_size=16)
    W = random_weights(spec, rng, std=0.05)
    gm = gpu_model(backend, spec, W, oh.F32)
    om = oracle_model(spec, W)
    tables = [[2 * s, 2 * s + 1] for s in range(S)]
    toks = rng.integers(0, V, S).tolist()
    print(f"[decode gemms] S={S} H={H} F={F} hq={hq} hkv={hkv} d={d} V={V}", flush=True)
    for pos in range(3):  # decode rows from the first position on
        b = batch(toks, [pos] * S, [1] * S, tables, [pos + 1] * S)
        g = gm.forward(b, want_argmax=True)
        o = om.forward(toks, [pos] * S, [1] * S, [pos + 1] * S, tables)
        # f32 KV: the split operands keep 17 bits of each activation, so the
        # logits are off by far less than the 1e-4 the forward tests allow
        assert rel_err(g.logits, o) <= 1e-4, (pos, rel_err(g.logits, o))
        toks = [orc.argmax(r) for r in o]
    om.close()
    gm.close()
