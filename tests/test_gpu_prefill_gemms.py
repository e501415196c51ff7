"""The prefill route's projections on the MI355X: the LDS-tiled GEMM's workgroup
shapes (2 to 5 row tiles per wave, 2 to 4 k-steps in LDS) at row counts around
their tile edges, and the QKV GEMM with RoPE and the KV write in its epilogue
against the CPU oracle and the separate launches (ORION_GEMM_FUSE=0)."""
import numpy as np
import pytest

import oracle as orc
import orion_hip as oh
from model_fixtures import Spec, oracle_model, random_weights
from test_gpu_model import batch, gpu_model, rel_err
from test_gpu_ops import gemm_case

pytestmark = pytest.mark.gpu


# (a K of one to three k-steps is shorter than the copies in flight)
@pytest.mark.parametrize("M,N,K", [
    (256, 8200, 96), (256, 28672, 32), (257, 16384, 64), (320, 24576, 96), (321, 520, 2080),
    (384, 6144, 1056), (480, 136, 4096), (576, 28688, 64), (743, 6152, 512), (768, 4096, 160),
    (961, 40, 32), (1024, 9216, 96), (1025, 9216, 96), (1300, 8200, 64)])
def test_tiled_shapes_match_linear(backend, M, N, K):
    for kw in (dict(bias=True), dict(accumulate=True)):
        got, _, ref64 = gemm_case(backend, M, N, K, seed=M + N, **kw)
        # the hi/lo split keeps x to ~2^-17 relative; the rest is summation order
        assert np.abs(got - ref64).max() <= 2e-5 * np.abs(ref64).max() + 1e-6, kw


@pytest.mark.parametrize("n,H,F,hq,hkv,d,kv", [
    (65, 256, 352, 4, 2, 64, oh.F32), (97, 256, 4096, 2, 1, 128, oh.BF16),
    (160, 96, 14336, 8, 4, 32, oh.F32), (161, 2048, 512, 4, 2, 64, oh.F32),
    (193, 128, 160, 3, 1, 96, oh.F32), (257, 256, 352, 4, 2, 80, oh.F32),
    (320, 64, 7168, 16, 16, 64, oh.F32), (640, 160, 2048, 5, 5, 32, oh.BF16),
    (1030, 128, 4160, 4, 1, 128, oh.F32),
    # 8192 QKV columns: 256-column tiles, with RoPE and with the permuted store
    (1030, 64, 160, 64, 32, 64, oh.F32)])
def test_prefill_rows_match_oracle_and_separate_rope(backend, monkeypatch, n, H, F, hq, hkv, d, kv):
    rng = np.random.default_rng(n * H + F)
    lens = [n // 2, 3, n - n // 2 - 3]  # ragged prompts, one below a row tile
    bs = 16
    blocks = [(L + 1 + bs - 1) // bs for L in lens]
    spec = Spec(2, H, hq, hkv, d, F, 300, max_pos=2048, bias=n % 2 == 0, tied=False,
                num_blocks=sum(blocks), block_size=bs)
    W = random_weights(spec, rng, std=0.05)
    perm = rng.permutation(spec.num_blocks).tolist()
    tables = [[perm.pop() for _ in range(k)] for k in blocks]
    toks = rng.integers(0, 300, n).tolist()
    pos = [p for L in lens for p in range(L)]
    om = oracle_model(spec, W)
    want = om.forward(toks, pos, lens, lens, tables)
    nxt = [orc.argmax(r) for r in want]
    ctx = [L + 1 for L in lens]
    want2 = om.forward(nxt, lens, [1, 1, 1], ctx, tables)
    om.close()
    got = {}
    for fuse in (None, "0"):
        if fuse:
            monkeypatch.setenv("ORION_GEMM_FUSE", fuse)
        gm = gpu_model(backend, spec, W, kv)
        print(f"[prefill gemms] n={n} H={H} F={F} hq={hq} hkv={hkv} d={d} fuse={fuse}", flush=True)
        a = gm.forward(batch(toks, pos, lens, tables), want_argmax=True).logits
        # one decode step reads the cache that the prompt wrote
        b = gm.forward(batch(nxt, lens, [1, 1, 1], tables, ctx), want_argmax=True).logits
        got[fuse] = (a, b)
        gm.close()
    monkeypatch.delenv("ORION_GEMM_FUSE")
    # f32 KV: 17 bits of each activation; bf16 KV rounds K and V (2^-9)
    tol = 1e-4 if kv == oh.F32 else 2e-2
    assert rel_err(got[None][0], want) <= tol and rel_err(got[None][1], want2) <= tol
    # the same f32 rotation; K splits differ where the separate route takes them
    # (an f32 sum's order, which in bf16 can turn a rounding of K or V: 2^-8)
    tol = 1e-5 if kv == oh.F32 else 4e-3
    assert rel_err(got[None][0], got["0"][0]) <= tol and rel_err(got[None][1], got["0"][1]) <= tol
