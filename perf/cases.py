"""Performance cases: one layer's worth of a serving engine's GPU work at a time, and one whole model step.

Each case calls the package's public entry points the way an engine does, on
inputs of the shapes the framework serves.  ``listed()`` holds the fixed
cases, ``draw()`` makes more of the same ranges.  Two attention shapes recur,
each with 16-token KV blocks: 32 query / 8 KV heads of 64 dims (the 1B model)
or of 128 dims (the 8B model), and 64 / 8 heads of 128 dims (a 70B layer).

Kinds
  decode   write_kv + decode attention of one layer, one new token a sequence
  prefill  write_kv + prefill attention of one layer; sequences with one new
           token in such a step are decode rows of a mixed step
  block    a layer's attention half: QKV projection, RoPE + cache write,
           attention, output projection
  mlp      a layer's MLP half: RMSNorm, gate/up projection, SwiGLU, down
           projection
  head     the step's end: last rows' RMSNorm, LM head, greedy argmax
  model    a whole model's decode or prefill step, logits out
"""
import importlib.util
import math
import pathlib
import sys

import numpy as np
import torch

ROOT = pathlib.Path(__file__).resolve().parents[1]
DEV = "cuda:0"
BS = 16                 # tokens of a KV block
FILL = 8192             # rows of a write_kv call while the cached context is laid down
EPS = 1e-5
THETA = 500000.0
NO_SCALING = dict(factor=1.0, low_freq_factor=1.0, high_freq_factor=4.0,
                  original_max_position_embeddings=8192)

# name: (query heads, KV heads, head dim)
SHAPES = {"1b": (32, 8, 64), "8b": (32, 8, 128), "70b": (64, 8, 128)}
# name: (hidden, FFN, vocabulary, layers)
MODELS = {"1b": (2048, 8192, 128256, 16), "8b": (4096, 14336, 128256, 32)}


def _package(sub=None):
    """The package (its folder's name is no identifier), or its module `sub`."""
    name = "vllm_oxide_amd"
    if name not in sys.modules:
        folder = ROOT / "vllm-oxide_amd"
        spec = importlib.util.spec_from_file_location(name, folder / "__init__.py",
                                                      submodule_search_locations=[str(folder)])
        module = importlib.util.module_from_spec(spec)
        sys.modules[name] = module
        spec.loader.exec_module(module)
    return importlib.import_module(f"{name}.{sub}") if sub else sys.modules[name]


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------


def _step(kind, shape, seqs, lo, hi, rows=1, prefix=0, lone=0, chunks=0, dist="uniform", **more):
    """A step over paged KV: `seqs` sequences of lo..hi cached tokens (after a
    `prefix` that all of them share) with `rows` new ones each, `lone` > 0:
    one more of that many cached tokens, `chunks` > 0: that many more with
    512-row prompt chunks beside the decode rows."""
    return dict(kind=kind, shape=shape, seqs=seqs, lo=lo, hi=hi, rows=rows, prefix=prefix,
                lone=lone, chunks=chunks, dist=dist, **more)


def listed():
    return [
        # One user, a short chat: the 1B model's attention at batch 1, 238-token prompt.
        dict(_step("decode", "1b", 1, 238, 238), name="decode_1_short"),
        # Two users with long chats: few rows, so the keys are the only parallelism.
        dict(_step("decode", "8b", 2, 5000, 8100), name="decode_2_long"),
        # The headline: 64 sequences of 512 to 4096 cached tokens.
        dict(_step("decode", "8b", 64, 512, 4096), name="decode_64"),
        # Prefix caching: 64 sequences over one 4096-token prefix, and one of 32768 tokens.
        dict(_step("decode", "70b", 64, 256, 1024, prefix=4096, lone=32768), name="decode_prefix"),
        # A first prompt of ordinary length, nothing cached.
        dict(_step("prefill", "1b", 1, 0, 0, rows=238), name="prefill_prompt"),
        # Chunked prefill: eight 512-row chunks over up to 8192 cached tokens.
        dict(_step("prefill", "8b", 8, 0, 8192, rows=512), name="prefill_chunks"),
        # The same with 8 query heads to a KV head and chunks that are no whole tiles.
        dict(_step("prefill", "70b", 3, 0, 6000, rows=451), name="prefill_ragged"),
        # A continuous-batching step: 256 decode rows and two prompt chunks.
        dict(_step("prefill", "8b", 256, 128, 8192, chunks=2, dist="lognormal"), name="mixed_step"),
        # A layer's attention half for a batch of two 700-token prompts behind a 512-token one.
        dict(_step("block", "1b", 2, 512, 512, rows=700), name="block_prefill"),
        # A layer's MLP half for a small decode batch: the weights are the work.
        dict(kind="mlp", shape="8b", rows=16, name="mlp_16"),
        # The end of a decode step of 40 sequences: logits and next tokens.
        dict(kind="head", shape="1b", rows=40, name="head_40"),
        # A whole decode step of four sequences.
        dict(_step("model", "1b", 4, 200, 2000), name="model_decode_4"),
    ]


def _log(rng, lo, hi):
    """A whole number of lo..hi, even over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "mixed", "block",
                       "block", "mlp", "mlp", "head", "model"])
    shape = rng.choice(list(SHAPES))
    if kind == "decode":
        seqs, hi = _log(rng, 1, 200), _log(rng, 20, 30000)
        hi = max(20, min(hi, 350000 // seqs))
        prefix = rng.choice([0, 0, 0, BS * _log(rng, 4, 256)])
        return _step("decode", shape, seqs, max(1, int(hi * rng.random())), hi,
                     prefix=prefix if seqs > 1 else 0)
    if kind == "prefill":
        seqs, rows = _log(rng, 1, 8), _log(rng, 17, 512)
        hi = rng.choice([0, _log(rng, 16, 8000)])
        return _step("prefill", shape, seqs, int(hi * rng.random()), hi, rows=rows)
    if kind == "mixed":
        seqs, hi = _log(rng, 4, 200), _log(rng, 256, 8000)
        return _step("prefill", shape, seqs, min(128, hi), hi, chunks=rng.randint(1, 2),
                     dist="lognormal")
    if kind == "block":
        shape = rng.choice(list(MODELS))
        rows = rng.choice([1, _log(rng, 2, 512)])
        seqs = _log(rng, 1, 64) if rows == 1 else rng.randint(1, 3)
        return _step("block", shape, seqs, 0, _log(rng, 16, 4000), rows=rows)
    shape = rng.choice(list(MODELS))
    if kind in ("mlp", "head"):
        rows = _log(rng, 1, 600 if kind == "mlp" else 128)
        return dict(kind=kind, shape=shape, rows=rows + (rows in (16, 40)))  # no listed case again
    rows = rng.choice([1, 1, _log(rng, 17, 300)])
    seqs = _log(rng, 1, 32) if rows == 1 else 1
    return _step("model", "1b", seqs, 0 if rows > 1 else 16, _log(rng, 16, 1500), rows=rows)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


class _Step:
    """Sequences, block tables and, where `kv`, one layer's cached K/V of a step."""

    def __init__(self, case, seed, kv=True):
        rng = np.random.default_rng(seed)
        self.heads, self.kv_heads, self.hd = SHAPES[case["shape"]]
        n, lo, hi = case["seqs"], case["lo"], case["hi"]
        if case["dist"] == "lognormal":
            ctx = np.clip(np.round(np.exp(math.log(1024) + rng.standard_normal(n))), lo, hi)
        else:
            ctx = rng.integers(lo, hi + 1, n)
        new = np.full(n, case["rows"], np.int64)
        prefix = case["prefix"]
        ctx = ctx.astype(np.int64) + prefix
        if case["lone"]:
            ctx, new = np.append(ctx, case["lone"]), np.append(new, 1)
        for c in range(case["chunks"]):
            ctx, new = np.append(ctx, 1536 * c), np.append(new, 512)
        self.ctx, self.new = ctx, new
        self.rows = int(new.sum())
        self.starts = np.concatenate([[0], np.cumsum(new)])
        blocks = -(-(ctx + new) // BS)
        shared = prefix // BS
        own = blocks - np.where(np.arange(len(ctx)) < n, shared, 0)
        self.num_blocks = int(own.sum()) + shared + 64
        perm = rng.permutation(self.num_blocks).astype(np.uint32)
        head, at, self.tables = perm[:shared], shared, []
        for s in range(len(ctx)):
            mine = perm[at:at + own[s]]
            at += own[s]
            self.tables.append(np.concatenate([head, mine]) if s < n and shared else mine)
        self.used_blocks = at
        self.gen = torch.Generator(device=DEV)
        self.gen.manual_seed(int(seed) + 1)
        if kv:
            width = self.kv_heads * self.hd
            self.k, self.v = self.randn(self.num_blocks * BS, width), self.randn(self.num_blocks * BS, width)

    def randn(self, *shape, scale=1.0):
        return (torch.randn(shape, generator=self.gen, device=DEV) * scale).to(torch.bfloat16)

    def slots(self, s):
        """Pool slots of every position of sequence s."""
        pos = np.arange(int(self.ctx[s] + self.new[s]))
        return torch.from_numpy(self.tables[s][pos // BS].astype(np.int64) * BS + pos % BS).to(DEV)

    def decode(self):
        return bool((self.new == 1).all())

    def meta(self, vo):
        if self.decode():
            return vo.DecodeMeta.new([vo.DecodeSeq(int(c), t) for c, t in zip(self.ctx, self.tables)], BS)
        return vo.PrefillMeta.new([vo.PrefillSeq(int(c), int(n), t)
                                   for c, n, t in zip(self.ctx, self.new, self.tables)], BS)

    def backend(self, vo):
        return vo.HipBackend(0, max_seqs=len(self.ctx), max_rows=max(self.rows, FILL),
                             max_table_entries=sum(len(t) for t in self.tables),
                             max_query_heads=self.heads)

    def fill(self, backend, pool, layer, k, v):
        for a in range(0, self.num_blocks * BS, FILL):
            b = min(a + FILL, self.num_blocks * BS)
            backend.write_kv(pool, layer, k[a:b], v[a:b], np.arange(a, b, dtype=np.uint32))


def _attention_inputs(st):
    width, kvw = st.heads * st.hd, st.kv_heads * st.hd
    return st.randn(st.rows, width), st.randn(st.rows, kvw), st.randn(st.rows, kvw)


def _weight(gen, out, inp, std=0.02):
    return (torch.randn((out, inp), generator=gen, device=DEV) * std).to(torch.bfloat16)


def _block_inputs(case, st):
    hidden = MODELS[case["shape"]][0]
    qd, kvd = st.heads * st.hd, st.kv_heads * st.hd
    return (st.randn(st.rows, hidden), _weight(st.gen, qd + 2 * kvd, hidden), _weight(st.gen, hidden, qd))


def _rows_inputs(case, seed):
    """mlp and head: a residual stream with the few large channels that trained models have."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed))
    hidden, ffn, vocab, _ = MODELS[case["shape"]]
    x = torch.randn((case["rows"], hidden), generator=gen, device=DEV)
    x[:, ::257] *= 20.0
    norm = (1.0 + 0.1 * torch.randn(hidden, generator=gen, device=DEV)).to(torch.bfloat16)
    if case["kind"] == "mlp":
        return x, norm, _weight(gen, 2 * ffn, hidden), _weight(gen, hidden, ffn)
    table = _weight(gen, vocab, hidden)
    # A sure next token for each row, as a trained model mostly has one.
    likely = torch.randint(0, vocab, (case["rows"],), generator=gen, device=DEV)
    x = x + 100.0 * table[likely].float()
    return x, norm, table


def _model_inputs(case, st):
    hidden, ffn, vocab, layers = MODELS[case["shape"]]
    qd, kvd = st.heads * st.hd, st.kv_heads * st.hd
    g = st.gen
    # The projections into the residual stream are smaller in deeper models and
    # its first values are of the size of what the layers add in all, as in a
    # trained model: the stream neither grows nor turns over with the depth.
    into = 0.02 / math.sqrt(2 * layers)
    one = lambda: (1.0 + 0.1 * torch.randn(hidden, generator=g, device=DEV)).to(torch.bfloat16)  # noqa: E731
    weights = dict(embed=_weight(g, vocab, hidden, 0.3), final_norm=one(), layers=[
        dict(attn_norm=one(), wq=_weight(g, qd, hidden), wk=_weight(g, kvd, hidden),
             wv=_weight(g, kvd, hidden), wo=_weight(g, hidden, qd, into), mlp_norm=one(),
             w_gate=_weight(g, ffn, hidden), w_up=_weight(g, ffn, hidden),
             w_down=_weight(g, hidden, ffn, into)) for _ in range(layers)])
    kv = [(st.randn(st.num_blocks * BS, kvd), st.randn(st.num_blocks * BS, kvd)) for _ in range(layers)]
    tokens = torch.randint(0, vocab, (st.rows,), generator=g, device=DEV).tolist()
    return weights, kv, tokens


def prepare(case, seed):
    vo = _package()
    if case["kind"] in ("mlp", "head"):
        state = dict(case=case, vo=vo)
        if case["kind"] == "mlp":
            state["x"], state["norm"], state["wgu"], state["wd"] = _rows_inputs(case, seed)
            state["backend"] = vo.HipBackend(0)
            state["backend"].gemm()
            return state
        state["x"], state["norm"], state["table"] = _rows_inputs(case, seed)
        rows = case["rows"]
        backend = vo.HipBackend(0, max_seqs=rows, max_rows=rows, max_table_entries=rows, max_query_heads=32)
        backend.gemm()
        pool = backend.alloc_kv_pool(vo.KvLayout(1, rows, BS, 8, 64))
        meta = vo.DecodeMeta.new([vo.DecodeSeq(0, [i]) for i in range(rows)], BS)
        return dict(state, backend=backend, pool=pool, meta=meta)
    if case["kind"] == "model":
        M = _package("model")
        st = _Step(case, seed, kv=False)
        weights, kv, tokens = _model_inputs(case, st)
        hidden, ffn, vocab, layers = MODELS[case["shape"]]
        backend = st.backend(vo)
        config = M.ModelConfig(hidden, ffn, layers, st.heads, st.kv_heads, vocab, 8192, EPS, THETA,
                               dict(NO_SCALING))
        engine = M.EngineConfig(max_batch_tokens=max(st.rows, 64), max_seqs=len(st.ctx), max_model_len=8192,
                                block_size=BS, num_blocks=st.num_blocks)
        model = M.Llama(backend, config, engine, weights)
        pool = model.alloc_kv_pool()
        for layer, (k, v) in enumerate(kv):
            st.fill(backend, pool, layer, k, v)
        return dict(case=case, vo=vo, model=model, pool=pool, st=st, tokens=tokens)
    st = _Step(case, seed)
    backend = st.backend(vo)
    pool = backend.alloc_kv_pool(vo.KvLayout(1, st.num_blocks, BS, st.kv_heads, st.hd))
    st.fill(backend, pool, 0, st.k, st.v)
    st.k = st.v = None
    state = dict(case=case, vo=vo, backend=backend, pool=pool, meta=st.meta(vo), decode=st.decode())
    if case["kind"] == "block":
        state["x"], state["wqkv"], state["wo"] = _block_inputs(case, st)
        state["rope"] = vo.RopeTable(st.hd, THETA, 8192, 0, **NO_SCALING)
        state["qd"], state["kvd"] = st.heads * st.hd, st.kv_heads * st.hd
        state["q"] = torch.empty((st.rows, state["qd"]), dtype=torch.bfloat16, device=DEV)
        backend.gemm()
    else:
        state["q"], state["k"], state["v"] = _attention_inputs(st)
    return state


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------


def run(state):
    case, vo = state["case"], state["vo"]
    kind = case["kind"]
    if kind == "model":
        st = state["st"]
        step = state["model"].decode if st.decode() else state["model"].prefill
        step(state["pool"], state["tokens"], st.meta(vo))
        return state["model"].logits[:len(st.ctx)]
    backend = state["backend"]
    if kind == "decode":
        return backend.decode_attention_write_kv(state["q"], state["k"], state["v"], state["pool"], 0,
                                                 state["meta"])
    if kind == "prefill":
        backend.write_kv(state["pool"], 0, state["k"], state["v"], state["meta"])
        return backend.prefill_attention(state["q"], state["pool"], 0, state["meta"])
    if kind == "block":
        pool, meta, q = state["pool"], state["meta"], state["q"]
        qkv = backend.matmul(state["x"], state["wqkv"])
        holder = backend.step_meta(pool)
        if holder.holds is not meta:
            holder.upload(meta)
        status = vo.lib.vo_qkv_rope_write_kv(
            pool.handle, 0, state["rope"].handle, qkv.data_ptr(), q.shape[0], state["qd"], state["kvd"],
            holder.handle, q.data_ptr(), torch.cuda.current_stream().cuda_stream)
        if status != vo.VO_OK:
            raise RuntimeError(f"vo_qkv_rope_write_kv: {status}")
        attention = backend.decode_attention if state["decode"] else backend.prefill_attention
        return backend.matmul(attention(q, pool, 0, meta), state["wo"], out_dtype=torch.float32)
    if kind == "mlp":
        ffn = state["wd"].shape[1]
        gu = backend.matmul(backend.rmsnorm(state["x"], state["norm"], EPS), state["wgu"])
        act = backend.silu_mul(gu[:, :ffn], gu[:, ffn:])
        return backend.matmul(act, state["wd"], out_dtype=torch.float32)
    last = backend.rmsnorm_last_rows(state["x"], state["norm"], EPS, state["pool"], state["meta"])
    logits = backend.matmul(last, state["table"], out_dtype=torch.float32)
    return {"logits": logits, "ids": backend.argmax(logits).astype(np.int64)}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------


def _attention_work(case):
    """Bytes and operations of the attention itself and of the new K/V, at the
    expected sizes (the contexts are drawn from the seed: their mean)."""
    heads, kv_heads, hd = SHAPES[case["shape"]]
    n, lo, hi, rows = case["seqs"], case["lo"], case["hi"], case["rows"]
    if case["dist"] == "lognormal":
        mean = float(np.clip(np.exp(math.log(1024) + np.random.default_rng(0).standard_normal(20000)), lo, hi).mean())
    else:
        mean = (lo + hi) / 2
    parts = [(n, mean, rows, case["prefix"])]
    if case["lone"]:
        parts.append((1, case["lone"], 1, 0))
    parts += [(1, 1536 * c, 512, 0) for c in range(case["chunks"])]
    keys = case["prefix"] + sum(m * (ctx + r) for m, ctx, r, _ in parts)
    total = sum(m * r for m, _, r, _ in parts)
    seen = sum(m * r * (p + ctx + (r + 1) / 2) for m, ctx, r, p in parts)
    return dict(kv=keys * kv_heads * hd * 4, new=total * kv_heads * hd * 4, qo=total * heads * hd * 4,
                flops=seen * heads * hd * 4, rows=total, seqs=sum(m for m, *_ in parts))


def work(case):
    kind = case["kind"]
    if kind in ("mlp", "head"):
        hidden, ffn, vocab, _ = MODELS[case["shape"]]
        rows = case["rows"]
        if kind == "mlp":
            return {"bytes": 3 * hidden * ffn * 2 + rows * hidden * 8 + hidden * 2,
                    "flops": 6 * rows * hidden * ffn}
        return {"bytes": vocab * hidden * 2 + rows * (hidden * 4 + vocab * 4) + hidden * 2,
                "flops": 2 * rows * hidden * vocab}
    w = _attention_work(case)
    if kind in ("decode", "prefill"):
        return {"bytes": w["kv"] + w["new"] + w["qo"], "flops": w["flops"]}
    heads, kv_heads, hd = SHAPES[case["shape"]]
    hidden, ffn, vocab, layers = MODELS[case["shape"]]
    matrix = hidden * (2 * heads + 2 * kv_heads) * hd  # weights of the QKV and output projections
    if kind == "block":
        return {"bytes": w["kv"] + 2 * matrix + w["rows"] * hidden * 6,
                "flops": w["flops"] + 2 * w["rows"] * matrix}
    matrix += 3 * hidden * ffn
    return {"bytes": layers * (w["kv"] + 2 * matrix) + 2 * vocab * hidden + w["seqs"] * vocab * 4,
            "flops": layers * (w["flops"] + 2 * w["rows"] * matrix) + 2 * w["seqs"] * vocab * hidden}


def tolerance(case):
    """About four times each kind's distance from ``exact``: 0.0017 (decode:
    the rounding of a bf16 output), 0.0023 (prefill: bf16 probabilities),
    0.0033 (block), 0.0039 (mlp), 0.0016 (head), 0.008 (model)."""
    return {"decode": {"rel": 0.007}, "prefill": {"rel": 0.009}, "block": {"rel": 0.013},
            "mlp": {"rel": 0.015}, "head": {"rel": 0.007, "differ": 0.01},
            "model": {"rel": 0.03}}[case["kind"]]


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------


def _exact_attention(st, q, k, v, pool_k, pool_v):
    """q [rows, heads*hd], k, v [rows, kv_heads*hd] f64 over the cached bf16 pools."""
    group = st.heads // st.kv_heads
    out = torch.empty_like(q)
    for s in range(len(st.ctx)):
        a, b, ctx, new = int(st.starts[s]), int(st.starts[s + 1]), int(st.ctx[s]), int(st.new[s])
        at = st.slots(s)[:ctx]
        ks = torch.cat([pool_k[at].double(), k[a:b]]).view(ctx + new, st.kv_heads, st.hd)
        vs = torch.cat([pool_v[at].double(), v[a:b]]).view(ctx + new, st.kv_heads, st.hd)
        qs = q[a:b].view(new, st.kv_heads, group, st.hd)
        hidden = (torch.arange(ctx + new, device=DEV)[None, :]
                  > ctx + torch.arange(new, device=DEV)[:, None]).repeat_interleave(group, 0)
        for h in range(st.kv_heads):
            score = qs[:, h].reshape(new * group, st.hd) @ ks[:, h].T.contiguous() / math.sqrt(st.hd)
            score.masked_fill_(hidden, -math.inf)
            o = torch.softmax(score, dim=1) @ vs[:, h].contiguous()
            out[a:b].view(new, st.kv_heads, group, st.hd)[:, h] = o.view(new, group, st.hd)
    return out


def _exact_rope(st, x):
    """NO_SCALING leaves every frequency as it is."""
    half = st.hd // 2
    pos = np.concatenate([c + np.arange(n) for c, n in zip(st.ctx, st.new)]).astype(np.float64)
    angle = torch.from_numpy(pos[:, None] * THETA ** (-np.arange(half) / half)).to(DEV)[:, None, :]
    x = x.view(st.rows, -1, st.hd)
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin()],
                     dim=-1).reshape(st.rows, -1)


def _exact_norm(x, w):
    return w.double() * (x * torch.rsqrt(x.square().mean(dim=1, keepdim=True) + EPS))


def _exact_mlp(x, wgu, wd):
    g, u = (x @ wgu.double().T).chunk(2, dim=1)
    return (g * torch.sigmoid(g) * u) @ wd.double().T


def _exact_block(st, x, wqkv, wo, pool_k, pool_v):
    qd, kvd = st.heads * st.hd, st.kv_heads * st.hd
    qkv = x @ wqkv.double().T
    q, k, v = qkv[:, :qd], qkv[:, qd:qd + kvd], qkv[:, qd + kvd:]
    attn = _exact_attention(st, _exact_rope(st, q), _exact_rope(st, k), v, pool_k, pool_v)
    return attn @ wo.double().T


def exact(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        x, norm, wgu, wd = _rows_inputs(case, seed)
        return _exact_mlp(_exact_norm(x.double(), norm), wgu, wd)
    if kind == "head":
        x, norm, table = _rows_inputs(case, seed)
        return {"logits": _exact_norm(x.double(), norm) @ table.double().T, "ids": None}
    if kind == "model":
        st = _Step(case, seed, kv=False)
        W, kv, tokens = _model_inputs(case, st)
        x = W["embed"][torch.tensor(tokens, device=DEV)].double()
        for L, (pool_k, pool_v) in zip(W["layers"], kv):
            wqkv = torch.cat([L["wq"], L["wk"], L["wv"]])
            x = x + _exact_block(st, _exact_norm(x, L["attn_norm"]), wqkv, L["wo"], pool_k, pool_v)
            x = x + _exact_mlp(_exact_norm(x, L["mlp_norm"]), torch.cat([L["w_gate"], L["w_up"]]), L["w_down"])
        last = torch.from_numpy(st.starts[1:] - 1).to(DEV)
        return _exact_norm(x[last], W["final_norm"]) @ W["embed"].double().T
    st = _Step(case, seed)
    if kind == "block":
        x, wqkv, wo = _block_inputs(case, st)
        return _exact_block(st, x.double(), wqkv, wo, st.k, st.v)
    q, k, v = _attention_inputs(st)
    return _exact_attention(st, q.double(), k.double(), v.double(), st.k, st.v)
