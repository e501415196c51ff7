"""The work this library is used for, as cases that can be timed and compared.

Three kinds of call, over the ranges a serving program meets:

* ``model``: one LanguageModel forward (HipTransformerModel.forward) on a
  prepared batch of decode rows and / or prefill chunks.  The one-layer models
  are a whole decoder layer (norms, projections, RoPE, KV write, paged
  attention, MLP) between a gather and a small head, at the layer shapes the
  benchmarks use; the 22-layer one is the benchmark's full model.
* ``attn_decode`` / ``attn_prefill``: the paged attention entry points alone,
  on a cache filled with N(0, 1) and scattered block tables.
* ``sample``: the device sampler on one step's logits, rows of mixed settings.

Sizes of a case (context lengths, chunk lengths) follow from the case alone;
weights, cache contents, tokens and block tables from the seed.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "orionserve-rs_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import orion_hip as oh  # noqa: E402

MASKED = -1.0e30  # the value the sampler gives a filtered logit
MAX_POS = 20480

# Decoder shapes of the benchmarks.  The one-layer shapes cut the vocabulary
# to 1024, so the layer and not the head is what counts.
SHAPES = {
    "tinyllama": dict(layers=22, hidden=2048, hq=32, hkv=4, d=64, ffn=5632, vocab=32000,
                      bias=False, theta=1.0e4, eps=1e-5),
    "tinyllama-layer": dict(layers=1, hidden=2048, hq=32, hkv=4, d=64, ffn=5632, vocab=1024,
                            bias=False, theta=1.0e4, eps=1e-5),
    "llama3-8b-layer": dict(layers=1, hidden=4096, hq=32, hkv=8, d=128, ffn=14336, vocab=1024,
                            bias=False, theta=5.0e5, eps=1e-5),
    "qwen2-7b-layer": dict(layers=1, hidden=3584, hq=28, hkv=4, d=128, ffn=18944, vocab=1024,
                           bias=True, theta=1.0e6, eps=1e-6),
}


def _model(name, shape, decodes=0, ctx=(0, 0), chunks=0, chunk=(0, 0), prefix=0, shared=0,
           block=16, lens=1):
    """decodes rows at contexts in ctx; chunks prefill chunks of lengths in
    chunk, each on a cached prefix of 0 .. prefix tokens; every other sequence
    of a shared batch starts with the same `shared` cached tokens."""
    c = dict(kind="model", shape=shape, decodes=decodes, ctx_lo=ctx[0], ctx_hi=ctx[1],
             chunks=chunks, chunk_lo=chunk[0], chunk_hi=chunk[1], prefix=prefix, shared=shared,
             block=block, lens=lens)
    return dict(c, name=name) if name else c


def _attn(name, kind, rows, lo, hi, hq, hkv, d, kv="bf16", chunk=0, block=16, lens=1):
    c = dict(kind=kind, rows=rows, lo=lo, hi=hi, hq=hq, hkv=hkv, d=d, kv=kv, chunk=chunk,
             block=block, lens=lens)
    return dict(c, name=name) if name else c


def _sample(name, rows, vocab, prev, lens=1):
    c = dict(kind="sample", rows=rows, vocab=vocab, prev=prev, lens=lens)
    return dict(c, name=name) if name else c


def listed():
    return [
        # One user's token: the latency of a whole decode step, one sequence.
        _model("step_1", "tinyllama", decodes=1, ctx=(700, 700)),
        # The benchmark's decode batch: 32 sequences of 16 .. 1024 tokens, full model.
        _model("step_32", "tinyllama", decodes=32, ctx=(16, 1024), lens=2),
        # One layer's share of a decode step, a handful of sequences, 8B layer.
        _model("layer_decode_6", "llama3-8b-layer", decodes=6, ctx=(128, 4096), lens=3),
        # An ordinary decode batch of an odd size on a layer with QKV bias.
        _model("layer_decode_45", "qwen2-7b-layer", decodes=45, ctx=(128, 4096), lens=4),
        # A busy server's decode batch: past 64 rows, below a prefill's.
        _model("layer_decode_160", "llama3-8b-layer", decodes=160, ctx=(64, 2048), lens=5),
        # One user's prompt through one layer.
        _model("layer_prompt_1", "llama3-8b-layer", chunks=1, chunk=(743, 743), lens=6),
        # The benchmark's prefill batch through one layer: 32 prompts, about 17,000 tokens.
        _model("layer_prompts_32", "tinyllama-layer", chunks=32, chunk=(16, 1024), lens=20),
        # Continuous batching: decode rows and prefill chunks together, half of
        # the sequences on one cached prefix.
        _model("layer_mixed", "qwen2-7b-layer", decodes=192, ctx=(256, 6000), chunks=8,
               chunk=(256, 256), prefix=4000, shared=2048, lens=8),
        # Paged attention alone, the smallest call: four short f32 sequences.
        _attn("attn_decode_4_f32", "attn_decode", 4, 1, 512, 8, 2, 64, kv="f32", lens=9),
        # The headline: 64 rows over 128 .. 4096 cached tokens, bf16.
        _attn("attn_decode_64", "attn_decode", 64, 128, 4096, 32, 8, 128, lens=10),
        # Chunked prefill attention: 8 chunks of 512 on prefixes of up to 7680.
        _attn("attn_prefill_8", "attn_prefill", 8, 0, 7680, 32, 8, 128, chunk=512, lens=11),
        # Sampling one decode step: rows of mixed settings, a vocabulary of 32,000.
        _sample("sample_32", 32, 32000, 200, lens=12),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "decode", "decode", "prompt", "mixed", "attn_decode",
                       "attn_prefill", "sample"])
    lens = rng.randrange(1, 1 << 30)
    layer = rng.choice(["tinyllama-layer", "llama3-8b-layer", "qwen2-7b-layer"])
    if kind == "step":
        hi = _log(rng, 64, 2048)
        return _model(None, "tinyllama", decodes=_log(rng, 1, 64), ctx=(16, hi), lens=lens)
    if kind == "decode":
        hi = _log(rng, 256, 4096)
        return _model(None, layer, decodes=_log(rng, 1, 256), ctx=(16, hi),
                      block=rng.choice([8, 16, 16, 32]), lens=lens)
    if kind == "prompt":
        n = _log(rng, 1, 8)
        hi = _log(rng, 24, min(1536, 3000 // n))
        return _model(None, layer, chunks=n, chunk=(16, hi), prefix=rng.choice([0, 0, 2000]),
                      lens=lens)
    if kind == "mixed":
        return _model(None, layer, decodes=_log(rng, 4, 160), ctx=(16, _log(rng, 512, 4096)),
                      chunks=rng.randrange(1, 6), chunk=(32, _log(rng, 64, 512)),
                      prefix=rng.choice([0, 3000]), lens=lens)
    hq, hkv, d = rng.choice([(32, 8, 128), (28, 4, 128), (32, 4, 64), (8, 2, 64)])
    if kind == "attn_decode":
        kv = rng.choice(["bf16", "bf16", "f32"])
        return _attn(None, kind, _log(rng, 1, 96), 1, _log(rng, 128, 8192), hq, hkv, d, kv=kv,
                     block=rng.choice([8, 16, 32]), lens=lens)
    if kind == "attn_prefill":
        return _attn(None, kind, rng.randrange(1, 9), 0, _log(rng, 64, 8000), hq, hkv, d,
                     chunk=_log(rng, 33, 512), lens=lens)
    return _sample(None, _log(rng, 1, 64), _log(rng, 4000, 152000), rng.randrange(1, 800),
                   lens=lens)


# ---------------------------------------------------------------------------
# Sizes that follow from the case
# ---------------------------------------------------------------------------


def _lens(case, n, lo, hi, salt):
    if n == 0:
        return np.zeros(0, np.int64)
    r = np.random.default_rng((case["lens"], salt))
    return r.integers(lo, max(hi, lo) + 1, size=n)


def _sequences(case):
    """[(first position, new tokens)] of the batch's sequences, decodes first,
    and which of them start with the shared cached tokens."""
    ctx = _lens(case, case["decodes"], case["ctx_lo"], case["ctx_hi"], 1)
    new = _lens(case, case["chunks"], case["chunk_lo"], case["chunk_hi"], 2)
    old = _lens(case, case["chunks"], 0, case["prefix"], 3)
    seqs = [[int(c) - 1, 1] for c in ctx] + [[int(p), int(c)] for p, c in zip(old, new)]
    on_shared = [bool(case["shared"]) and i % 2 == 0 for i in range(len(seqs))]
    for s, on in zip(seqs, on_shared):
        if on:
            s[0] += case["shared"]
    return [(max(a, 0), n) for a, n in seqs], on_shared


def _tables(seqs, on_shared, shared, block, rng):
    """Scattered block tables over a pool of 1.25x the blocks needed; those of
    on_shared begin with the same whole blocks."""
    nshared = shared // block
    need = [(a + n + block - 1) // block for a, n in seqs]
    own = [n - (nshared if on else 0) for n, on in zip(need, on_shared)]
    total = sum(own) + (nshared if any(on_shared) else 0)
    pool = max(1, total * 5 // 4)
    ids = rng.permutation(pool)
    head, at = ids[:nshared], nshared if any(on_shared) else 0
    tables = []
    for n, on in zip(own, on_shared):
        t = ids[at:at + n]
        at += n
        tables.append(np.concatenate([head, t]) if on else t)
    return [t.astype(np.uint32) for t in tables], pool


def _weights(s):
    """Elements of one layer's matrices, and of the head."""
    qkv = (s["hq"] + 2 * s["hkv"]) * s["d"] * s["hidden"]
    layer = qkv + s["hidden"] * s["hq"] * s["d"] + 3 * s["hidden"] * s["ffn"]
    return layer, s["vocab"] * s["hidden"]


def work(case):
    if case["kind"] == "model":
        s = SHAPES[case["shape"]]
        seqs, on = _sequences(case)
        rows = sum(n for _, n in seqs)
        layer, head = _weights(s)
        vec = 2 * s["hkv"] * s["d"] * 2  # K and V of one token, bf16
        nsh = case["shared"] // case["block"] * case["block"]
        old = sum(a - (nsh if o else 0) for (a, _), o in zip(seqs, on)) + (nsh if any(on) else 0)
        pairs = sum(a * n + n * (n + 1) // 2 for a, n in seqs)
        nbytes = s["layers"] * (2 * layer + vec * (old + rows)) + 2 * head
        nbytes += rows * s["hidden"] * 2 + len(seqs) * s["vocab"] * 4
        flops = s["layers"] * (2.0 * rows * layer + 4.0 * s["hq"] * s["d"] * pairs)
        return dict(bytes=nbytes, flops=flops + 2.0 * len(seqs) * head)
    if case["kind"] == "sample":
        n = case["rows"] * case["vocab"]
        return dict(bytes=8 * n, flops=4.0 * n)
    esz = 4 if case["kv"] == "f32" else 2
    lens = _lens(case, case["rows"], case["lo"], case["hi"], 1)
    per = case["hq"] * case["d"]
    if case["kind"] == "attn_decode":
        tokens, rows, pairs = int(lens.sum()), case["rows"], int(lens.sum())
    else:
        c = case["chunk"]
        tokens, rows = int(lens.sum()) + c * len(lens), c * case["rows"]
        pairs = int(sum(int(a) * c + c * (c + 1) // 2 for a in lens))
    return dict(bytes=tokens * 2 * case["hkv"] * case["d"] * esz + 2 * rows * per * 4,
                flops=4.0 * per * pairs)


def tolerance(case):
    if case["kind"] == "sample":
        # values are copied or scaled; a candidate on the edge of the nucleus may
        # fall either way (one of rows x vocab masked values)
        return {"rel": 5e-3, "max": 0.99, "differ": 0.01}
    if case["kind"] == "attn_decode":
        return {"rel": 4e-5, "max": 2e-3}
    if case["kind"] == "attn_prefill":
        return {"rel": 4e-5, "max": 2e-3}
    if case["shape"] == "tinyllama":
        # 22 layers: each new K/V vector is rounded to bf16, and a rounding that
        # falls the other way travels through the layers after it
        return {"rel": 4e-3, "max": 6e-2}
    return {"rel": 1e-3, "max": 4e-2}


# ---------------------------------------------------------------------------
# States
# ---------------------------------------------------------------------------

_BE = None


def _backend():
    global _BE
    if _BE is None:
        _BE = oh.HipBackend(0)
    return _BE


class _Memory:
    """Device memory of the library, seen as a tensor; `keep` owns it."""

    def __init__(self, ptr, count, keep):
        self.keep = keep
        self.__cuda_array_interface__ = dict(shape=(count,), typestr="<i2", data=(ptr, False),
                                             version=2)


class _Model:
    def __init__(self, case):
        s = SHAPES[case["shape"]]
        self.model = None
        self.shape, self.case = s, case
        self.seqs, self.on_shared = _sequences(case)

    def open(self, num_blocks):
        s = self.shape
        meta = oh.ModelMetadata(
            hidden_size=s["hidden"], num_layers=s["layers"], num_attention_heads=s["hq"],
            num_kv_heads=s["hkv"], head_dim=s["d"], vocab_size=s["vocab"],
            intermediate_size=s["ffn"], max_position_embeddings=MAX_POS, rope_theta=s["theta"],
            rms_norm_eps=s["eps"], architecture="qwen2" if s["bias"] else "llama")
        self.model = oh.HipTransformerModel(meta, num_blocks, self.case["block"], _backend(),
                                            oh.BF16)
        ptr, nbytes = self.model.kv_arena()
        self.arena_ptr, self.arena_bytes = ptr, nbytes

    def arena(self):
        t = torch.as_tensor(_Memory(self.arena_ptr, self.arena_bytes // 2, self), device="cuda")
        return t.view(torch.bfloat16)

    def __del__(self):
        if self.model is not None:
            self.model.close()
            self.model = None


def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000003 + salt)
    return g


def _randn(g, *shape, std=1.0, base=0.0, dtype=torch.bfloat16):
    """N(base, std) rounded to dtype, drawn in pieces of 64 M values."""
    n = int(np.prod(shape))
    out = torch.empty(n, dtype=dtype, device="cuda")
    for a in range(0, n, 1 << 26):
        b = min(n, a + (1 << 26))
        out[a:b] = (torch.randn(b - a, generator=g, device="cuda") * std + base).to(dtype)
    return out.view(*shape)


def _layer_tensors(s, seed):
    """The weights of a one-layer model, bf16 on the GPU (norms and biases f32)."""
    g = _gen(seed, 1)
    H, F, qd, kvd = s["hidden"], s["ffn"], s["hq"] * s["d"], s["hkv"] * s["d"]
    f32 = torch.float32
    w = {oh.W_EMBED: _randn(g, s["vocab"], H, std=0.02),
         oh.W_FINAL_NORM: _randn(g, H, std=0.1, base=1.0, dtype=f32),
         oh.W_LM_HEAD: _randn(g, s["vocab"], H, std=0.02),
         oh.W_INPUT_NORM: _randn(g, H, std=0.1, base=1.0, dtype=f32),
         oh.W_Q: _randn(g, qd, H, std=0.02), oh.W_K: _randn(g, kvd, H, std=0.02),
         oh.W_V: _randn(g, kvd, H, std=0.02), oh.W_O: _randn(g, H, qd, std=0.02),
         oh.W_POST_NORM: _randn(g, H, std=0.1, base=1.0, dtype=f32),
         oh.W_GATE: _randn(g, F, H, std=0.02), oh.W_UP: _randn(g, F, H, std=0.02),
         oh.W_DOWN: _randn(g, H, F, std=0.02)}
    if s["bias"]:
        w[oh.W_Q_BIAS] = _randn(g, qd, std=0.02, dtype=f32)
        w[oh.W_K_BIAS] = _randn(g, kvd, std=0.02, dtype=f32)
        w[oh.W_V_BIAS] = _randn(g, kvd, std=0.02, dtype=f32)
    return w


def _cache(case, s, pool, seed):
    """What earlier steps left in the cache: N(0, 1) in bf16, every layer and block."""
    return _randn(_gen(seed, 2), s["layers"] * pool * 2 * case["block"] * s["hkv"] * s["d"])


def _tokens(case, s, rows, seed):
    return np.random.default_rng((seed, 3)).integers(0, s["vocab"], rows)


def _prepare_model(case, seed):
    st = _Model(case)
    s, seqs = st.shape, st.seqs
    tables, pool = _tables(seqs, st.on_shared, case["shared"], case["block"],
                           np.random.default_rng((seed, 4)))
    st.open(pool)
    if s["layers"] == 1:
        for which, t in _layer_tensors(s, seed).items():
            a = t.cpu() if t.dtype == torch.float32 else t.view(torch.int16).cpu()
            a = a.numpy() if t.dtype == torch.float32 else a.numpy().view(np.uint16)
            st.model.upload_weight(which, 0, a)
    else:
        st.model.init_synthetic(seed, 0.02)
    cache = _cache(case, s, pool, seed)
    torch.cuda.synchronize()
    _backend().memcpy_d2d(st.arena_ptr, cache.data_ptr(), st.arena_bytes)
    _backend().synchronize()
    rows = sum(n for _, n in seqs)
    pos = [p for a, n in seqs for p in range(a, a + n)]
    st.batch = oh.ForwardBatch(
        _tokens(case, s, rows, seed).tolist(), pos, list(range(len(seqs))),
        [n for _, n in seqs], [a + n for a, n in seqs], [t.tolist() for t in tables],
        case["chunks"] > 0).prepare()
    return st


class _Attn:
    plan = None

    def __del__(self):
        if self.plan is not None:
            self.plan.close()
            self.plan = None


def _attn_inputs(case, seed):
    """Tensors of an attention call: cache, queries, positions and tables."""
    c = case
    lens = _lens(c, c["rows"], c["lo"], c["hi"], 1)
    if c["kind"] == "attn_decode":
        seqs = [(int(n) - 1, 1) for n in lens]
    else:
        seqs = [(int(n), c["chunk"]) for n in lens]
    tables, pool = _tables(seqs, [False] * len(seqs), 0, c["block"],
                           np.random.default_rng((seed, 4)))
    dt = torch.float32 if c["kv"] == "f32" else torch.bfloat16
    arena = _randn(_gen(seed, 2), pool, 2, c["block"], c["hkv"], c["d"], dtype=dt)
    q = _randn(_gen(seed, 5), sum(n for _, n in seqs), c["hq"], c["d"], dtype=torch.float32)
    return seqs, tables, pool, arena, q


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _prepare_attn(case, seed):
    c, st, be = case, _Attn(), _backend()
    seqs, tables, pool, st.arena, st.q = _attn_inputs(case, seed)
    st.case, st.pool, st.out = case, pool, torch.empty_like(st.q)
    st.kv = oh.kv_layout(1, pool, c["block"], c["hkv"], c["d"],
                         oh.F32 if c["kv"] == "f32" else oh.BF16)
    offs = np.cumsum([0] + [len(t) for t in tables]).astype(np.int64)
    ids = np.concatenate(tables)
    st.offs, st.ids = _dev(offs), _dev(ids.view(np.int32))
    first = np.array([a for a, _ in seqs], np.uint32)
    if c["kind"] == "attn_decode":
        rows = np.arange(len(seqs), dtype=np.int32)
        st.pos, st.seq = _dev(first.view(np.int32)), _dev(rows)
        st.plan = oh.DecodePlan(be, first, rows, offs, ids, c["hq"], c["hkv"], c["d"], c["block"])
    else:
        n = len(seqs)
        st.start = _dev((np.arange(n) * c["chunk"]).astype(np.int32))
        st.count = _dev(np.full(n, c["chunk"], np.int32))
        st.first = _dev(first.view(np.int32))
        st.max_pos = int(first.max()) + c["chunk"] - 1
    torch.cuda.synchronize()
    return st


class _Sample:
    pass


def _settings(case):
    """Per-row (temperature, top_k, top_p, repetition_penalty): a quarter each
    greedy, nucleus only, top-k + nucleus + penalty, and plain temperature."""
    kinds = [(0.0, 0, 1.0, 1.0), (1.0, 0, 0.95, 1.0), (0.8, 50, 0.9, 1.1), (0.7, 0, 1.0, 1.05)]
    r = np.random.default_rng((case["lens"], 6))
    return [kinds[(i + int(r.integers(0, 2))) % 4] for i in range(case["rows"])]


def _sample_inputs(case, seed):
    n, V = case["rows"], case["vocab"]
    logits = _randn(_gen(seed, 7), n, V, std=2.0, dtype=torch.float32)
    r = np.random.default_rng((seed, 8))
    prev = [r.integers(0, V, case["prev"]).astype(np.uint32) for _ in range(n)]
    return logits, prev, r.random(n, dtype=np.float32)


def _prepare_sample(case, seed):
    st = _Sample()
    st.case = case
    st.logits, st.prev, st.uniform = _sample_inputs(case, seed)
    st.work = torch.empty_like(st.logits)
    st.params = [oh.SamplingParams(*p) for p in _settings(case)]
    torch.cuda.synchronize()
    return st


def prepare(case, seed):
    if case["kind"] == "model":
        return _prepare_model(case, seed)
    if case["kind"] == "sample":
        return _prepare_sample(case, seed)
    return _prepare_attn(case, seed)


def run(st):
    c = st.case
    if c["kind"] == "model":
        if st.shape["layers"] > 1:
            # the step's logits and greedy tokens, and the cache it wrote into
            out = st.model.forward(st.batch, want_logits=True, want_argmax=True)
        else:
            out = st.model.forward(st.batch)
        return {"logits": out.logits, "cache": st.arena()}
    be = _backend()
    if c["kind"] == "sample":
        # the sampler filters its logits in place: each pass takes the step's anew
        be.memcpy_d2d(st.work.data_ptr(), st.logits.data_ptr(), st.logits.numel() * 4)
        tokens = oh.sample(be, st.work.data_ptr(), c["rows"], c["vocab"], st.params, st.prev,
                           st.uniform)
        return {"filtered": st.work, "tokens": np.asarray(tokens, np.int64)}
    if c["kind"] == "attn_decode":
        oh.paged_attention_decode(be, st.kv, st.arena.data_ptr(), 0, st.q.data_ptr(), c["rows"],
                                  c["hq"], st.pos.data_ptr(), st.seq.data_ptr(),
                                  st.offs.data_ptr(), st.ids.data_ptr(), st.plan,
                                  st.out.data_ptr())
    else:
        # Q and P as hi + lo pairs: what the forward asks for
        oh.paged_attention_prefill(be, st.kv, st.arena.data_ptr(), 0, st.q.data_ptr(), c["hq"],
                                   c["rows"], st.start.data_ptr(), st.count.data_ptr(),
                                   st.first.data_ptr(), st.offs.data_ptr(), st.ids.data_ptr(),
                                   c["chunk"], st.max_pos, st.out.data_ptr(), hilo=True)
    return st.out


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------

F64 = torch.float64


def _attend(q, k, v, first):
    """q [n, hq, d] at positions first .. first + n - 1 over k, v [m, hkv, d]."""
    n, hq, d = q.shape
    m, hkv, _ = k.shape
    G = hq // hkv
    out = torch.empty(n, hq, d, dtype=F64, device="cuda")
    mask = None
    if n > 1:
        mask = torch.arange(m, device="cuda")[None, :] > torch.arange(n, device="cuda")[:, None] + first
    for h in range(hkv):
        kt = k[:, h].t().contiguous()
        vh = v[:, h].contiguous()
        for g in range(h * G, (h + 1) * G):
            s = torch.mm(q[:, g].contiguous(), kt) / math.sqrt(d)
            if mask is not None:
                s = s.masked_fill(mask, -math.inf)
            out[:, g] = torch.mm(torch.softmax(s, dim=1), vh)
    return out


def _exact_attn(case, seed):
    seqs, tables, pool, arena, q = _attn_inputs(case, seed)
    out = torch.empty(q.shape, dtype=F64, device="cuda")
    r = 0
    for (a, n), t in zip(seqs, tables):
        kv = arena[_dev(t.astype(np.int64))].to(F64)  # [blocks, 2, block, hkv, d]
        k = kv[:, 0].reshape(-1, case["hkv"], case["d"])[:a + n]
        v = kv[:, 1].reshape(-1, case["hkv"], case["d"])[:a + n]
        out[r:r + n] = _attend(q[r:r + n].to(F64), k, v, a)
        r += n
    return out


def _exact_model(case, seed):
    s = SHAPES[case["shape"]]
    if s["layers"] > 1:
        return None
    seqs, on = _sequences(case)
    tables, pool = _tables(seqs, on, case["shared"], case["block"],
                           np.random.default_rng((seed, 4)))
    w = _layer_tensors(s, seed)
    bs, hq, hkv, d = case["block"], s["hq"], s["hkv"], s["d"]
    cache = _cache(case, s, pool, seed).view(pool, 2, bs, hkv, d)
    rows = sum(n for _, n in seqs)
    tok = _dev(_tokens(case, s, rows, seed).astype(np.int64))
    pos = np.concatenate([np.arange(a, a + n) for a, n in seqs])

    def mul(x, which):
        return torch.mm(x, w[which].to(F64).t().contiguous())

    def norm(x, which):
        return x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + s["eps"]) * w[which].to(F64)

    h = w[oh.W_EMBED][tok].to(F64)
    x = norm(h, oh.W_INPUT_NORM)
    q, k, v = mul(x, oh.W_Q), mul(x, oh.W_K), mul(x, oh.W_V)
    if s["bias"]:
        q, k, v = q + w[oh.W_Q_BIAS].to(F64), k + w[oh.W_K_BIAS].to(F64), v + w[oh.W_V_BIAS].to(F64)
    # the model's rotation angles are f32 products of an f32 table
    half = d // 2
    i = np.arange(half, dtype=np.float32)
    inv = np.float32(1.0) / np.power(np.float32(s["theta"]), np.float32(2.0) * i / np.float32(d))
    ang = (pos.astype(np.float32)[:, None] * inv[None, :].astype(np.float32)).astype(np.float64)
    cos, sin = _dev(np.cos(ang))[:, None, :], _dev(np.sin(ang))[:, None, :]

    def rope(t, heads):
        t = t.view(rows, heads, d)
        a, b = t[..., :half], t[..., half:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], dim=-1)

    q, k, v = rope(q, hq), rope(k, hkv), v.view(rows, hkv, d)
    seq_of = np.concatenate([np.full(n, j) for j, (_, n) in enumerate(seqs)])
    blk = _dev(np.array([tables[j][p // bs] for j, p in zip(seq_of, pos)], np.int64))
    slot = _dev((pos % bs).astype(np.int64))
    cache[blk, 0, slot] = k.to(torch.bfloat16)  # the cache holds bf16
    cache[blk, 1, slot] = v.to(torch.bfloat16)
    att = torch.empty(rows, hq, d, dtype=F64, device="cuda")
    r = 0
    for (a, n), t in zip(seqs, tables):
        kv = cache[_dev(t.astype(np.int64))].to(F64)
        att[r:r + n] = _attend(q[r:r + n], kv[:, 0].reshape(-1, hkv, d)[:a + n],
                               kv[:, 1].reshape(-1, hkv, d)[:a + n], a)
        r += n
    h = h + mul(att.view(rows, hq * d), oh.W_O)
    x = norm(h, oh.W_POST_NORM)
    gate = mul(x, oh.W_GATE)
    h = h + mul(gate * torch.sigmoid(gate) * mul(x, oh.W_UP), oh.W_DOWN)
    last = _dev(np.cumsum([n for _, n in seqs]) - 1)
    logits = mul(norm(h[last], oh.W_FINAL_NORM), oh.W_LM_HEAD)
    return {"logits": logits.cpu().numpy(), "cache": cache.view(-1).to(F64)}


def _exact_sample(case, seed):
    logits, prev, _ = _sample_inputs(case, seed)
    x = logits.to(F64)
    for r, (temp, top_k, top_p, pen) in enumerate(_settings(case)):
        row = x[r]
        if pen != 1.0:
            t = _dev(np.unique(prev[r]).astype(np.int64))
            pen = float(np.float32(pen))
            row[t] = torch.where(row[t] > 0, row[t] / pen, row[t] * pen)
        if temp == 0.0:
            continue
        row *= float(np.float32(1.0) / np.float32(temp))
        if 0 < top_k < case["vocab"]:
            row[row < torch.topk(row, top_k).values[-1]] = MASKED
        if top_p < 1.0:
            p = torch.softmax(torch.where(row <= MASKED, -math.inf, row), dim=0)
            v, order = torch.sort(p, descending=True)
            before = torch.cumsum(v, dim=0) - v
            row[order[before >= float(np.float32(top_p))]] = MASKED
    return {"filtered": x, "tokens": None}


def exact(case, seed):
    if case["kind"] == "model":
        return _exact_model(case, seed)
    if case["kind"] == "sample":
        return _exact_sample(case, seed)
    return _exact_attn(case, seed)
