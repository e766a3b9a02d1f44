"""The framework's work as its users have it done: single layers and blocks of the decoder, the paged
attention, sampling and acceptance, and whole forward calls, each through a public entry point.

Sizes come from the package's own configurations: the tiny float32 model (4 layers, d 256, 8/4 heads,
ffn 688, vocabulary 512), the 1B shape (d 2048, 32/8 heads, head_dim 64, ffn 8192, vocabulary 32000) and
the 8B shape (d 4096, 32/8 heads, head_dim 128, ffn 14336, vocabulary 128256), with the batches, windows
and contexts that the benchmark, the Engine workload and the tests run.

A case names its `kind` and that kind's sizes. Lengths that differ from row to row (contexts, prompts)
are drawn from the case's `sizes` number, so that they belong to the case; the values (weights, caches,
activations, token ids, noise) are drawn from the seed.
"""

import math
import random

import torch

import forgeserve_amd as fa
from forgeserve_amd import ops

DEV = "cuda"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
SHAPES = {
    "tiny": dict(vocab_size=512, d_model=256, n_heads=8, n_kv_heads=4, ffn_dim=688, max_seq_len=512),
    "1b": dict(vocab_size=32000, d_model=2048, n_heads=32, n_kv_heads=8, ffn_dim=8192, max_seq_len=2048),
    "8b": dict(vocab_size=128256, d_model=4096, n_heads=32, n_kv_heads=8, ffn_dim=14336, max_seq_len=32768),
}
BLOCK = 16


# ------------------------------------------------------------------------------------------------
# the cases
# ------------------------------------------------------------------------------------------------
def listed():
    return [
        # one request decoding on the tiny float32 model (the package's default dtype): the smallest call
        dict(name="decode_tiny_f32", kind="decode", shape="tiny", dtype="f32", layers=4, batch=1, t=1, lo=100, hi=100,
             layout="slots", sizes=1),
        # the tiny float32 model over whole sequences, logits at every position (teacher forcing, evaluation)
        dict(name="forward_tiny_f32", kind="forward", shape="tiny", dtype="f32", layers=4, batch=4, t=160),
        # one Engine decode step of 16 running requests at the 1B shape (4 of its 16 layers, and the head)
        dict(name="decode_1b", kind="decode", shape="1b", dtype="bf16", layers=4, batch=16, t=1, lo=128, hi=1280,
             layout="slots", sizes=2),
        # the prompts that an Engine admits at once, prefilled packed (4 layers of the 1B shape)
        dict(name="prefill_1b", kind="prefill", shape="1b", dtype="bf16", layers=4, rows=12, lo=128, hi=1024, sizes=3),
        # one decoder block of the 8B verify pass: 64 sequences, a window of k + 1 = 7 tokens
        dict(name="block_verify_8b", kind="block", shape="8b", dtype="bf16", batch=64, t=7, lo=2048, hi=8192,
             layout="groups", sizes=4),
        # one decoder block of a small decoding batch at the 8B shape
        dict(name="block_decode_8b", kind="block", shape="8b", dtype="bf16", batch=8, t=1, lo=512, hi=4096,
             layout="slots", sizes=5),
        # the paged verify attention alone, 32 sequences with a window of 5
        dict(name="attn_verify", kind="attn", heads=32, kv_heads=8, hd=128, batch=32, t=5, lo=512, hi=4096,
             layout="slots", sizes=6),
        # a few requests with long contexts, one token each
        dict(name="attn_long", kind="attn", heads=32, kv_heads=8, hd=128, batch=3, t=1, lo=8000, hi=30000,
             layout="groups", sizes=7),
        # the attention of a packed prefill of ragged prompts
        dict(name="attn_prefill", kind="attn_prefill", heads=32, kv_heads=8, hd=128, rows=5, lo=300, hi=4096,
             layout="groups", sizes=8),
        # the MLP over a long packed prefill (an odd number of tokens)
        dict(name="mlp_prefill_8b", kind="mlp", shape="8b", dtype="bf16", m=8005),
        # the fused acceptance of one verify pass, every logit row read
        dict(name="accept_8b", kind="accept", dtype="bf16", batch=64, k=6, vocab=128256),
        # a draft step's draws (64 rows sampled from their logits), and one row's probabilities
        dict(name="sample_8b", kind="sample", dtype="bf16", rows=64, vocab=128256),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "forward", "prefill", "block", "attn", "attn_prefill", "mlp", "accept", "sample"])
    sizes = rng.randrange(1000)
    layout = rng.choice(["slots", "groups"])
    if kind == "decode":   # one token, or a speculative window, per running request
        if rng.random() < 0.4:
            hi = rng.randint(40, 400)
            return dict(kind=kind, shape="tiny", dtype="f32", layers=4, batch=_log_int(rng, 1, 16),
                        t=rng.choice([1, 1, 5]), lo=20, hi=hi, layout=layout, sizes=sizes)
        hi = rng.randint(300, 2000)
        return dict(kind=kind, shape="1b", dtype="bf16", layers=rng.randint(1, 4), batch=_log_int(rng, 1, 16),
                    t=rng.choice([1, 1, 5]), lo=128, hi=hi, layout=layout, sizes=sizes)
    if kind == "forward":
        return dict(kind=kind, shape="tiny", dtype="f32", layers=4, batch=_log_int(rng, 1, 4), t=_log_int(rng, 2, 160))
    if kind == "prefill":
        return dict(kind=kind, shape="1b", dtype="bf16", layers=rng.randint(1, 4), rows=_log_int(rng, 1, 12), lo=128,
                    hi=rng.randint(200, 1024), sizes=sizes)
    if kind == "block":
        shape = rng.choice(["1b", "8b"])
        batch, t = _log_int(rng, 1, 64), rng.choice([1, 1, 5, 7])
        hi = rng.randint(600, 2000) if shape == "1b" else _log_int(rng, 600, 8192)
        return dict(kind=kind, shape=shape, dtype="bf16", batch=batch, t=t, lo=hi // 8 + 8, hi=hi, layout=layout,
                    sizes=sizes)
    if kind == "attn":
        hd, kv_heads = rng.choice([64, 128]), 8
        hi = _log_int(rng, 200, 30000)
        batch = max(1, min(64, _log_int(rng, 1, 64), 120000 // hi))
        return dict(kind=kind, heads=kv_heads * rng.choice([1, 4, 4, 8]), kv_heads=kv_heads, hd=hd, batch=batch,
                    t=rng.choice([1, 1, 3, 5, 7, 9]), lo=hi // 8 + 9, hi=hi, layout=layout, sizes=sizes)
    if kind == "attn_prefill":
        hi = _log_int(rng, 300, 4096)
        return dict(kind=kind, heads=32, kv_heads=8, hd=rng.choice([64, 128]), rows=max(1, min(8, 8000 // hi)),
                    lo=hi // 8 + 64, hi=hi, layout=layout, sizes=sizes)
    if kind == "mlp":
        shape = rng.choice(["1b", "8b"])
        return dict(kind=kind, shape=shape, dtype="bf16", m=_log_int(rng, 1, 8000))
    vocab = rng.choice([32000, 128256, _log_int(rng, 500, 128256)])
    if kind == "accept":
        dtype = rng.choice(["f32", "bf16"])
        k = rng.randint(1, 8)
        return dict(kind=kind, dtype=dtype, batch=max(1, min(_log_int(rng, 1, 64), int(200e6 / (vocab * k * 8)))), k=k,
                    vocab=vocab)
    return dict(kind=kind, dtype=rng.choice(["f32", "bf16"]), rows=_log_int(rng, 1, 64), vocab=vocab)


# ------------------------------------------------------------------------------------------------
# what a case's sizes and seed stand for
# ------------------------------------------------------------------------------------------------
def _config(case, layers=1):
    return dict(SHAPES[case["shape"]], n_layers=case.get("layers", layers))


def _lengths(case, n):
    """n context or prompt lengths in lo..hi (the first is hi)."""
    r = random.Random(case["sizes"])
    return [case["hi"]] + [r.randint(case["lo"], case["hi"]) for _ in range(n - 1)]


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, *shape, dtype=torch.float32, std=1.0):
    return torch.randn(*shape, device=DEV, generator=g).mul_(std).to(dtype)


def _weights(case, g):
    """A decoder's parameters by name: N(0, 0.02) matrices, norms near 1. The layers of one case share
    nothing; the head is the embedding."""
    c, dt = _config(case), DTYPES[case["dtype"]]
    d, f, hd = c["d_model"], c["ffn_dim"], c["d_model"] // c["n_heads"]
    w = {}
    if case["kind"] in ("decode", "forward", "prefill"):
        w["tok_emb.weight"] = _normal(g, c["vocab_size"], d, dtype=dt, std=0.02)
    for i in range(c["n_layers"]):
        p = f"layers.{i}."
        for name, rows, cols in (("attn.wq", c["n_heads"] * hd, d), ("attn.wk", c["n_kv_heads"] * hd, d),
                                 ("attn.wv", c["n_kv_heads"] * hd, d), ("attn.wo", d, c["n_heads"] * hd),
                                 ("mlp.w_gate", f, d), ("mlp.w_up", f, d), ("mlp.w_down", d, f)):
            w[f"{p}{name}.weight"] = _normal(g, rows, cols, dtype=dt, std=0.02)
        for name in ("attn_norm", "mlp_norm"):
            w[f"{p}{name}.weight"] = (1 + _normal(g, d, std=0.1)).to(dt)
    w["norm.weight"] = (1 + _normal(g, d, std=0.1)).to(dt)
    return w


def _module(dtype, make):
    """make()'s module with parameters of this dtype, on the GPU from the start."""
    prev = torch.get_default_dtype()
    torch.set_default_dtype(dtype)
    try:
        with torch.device(DEV):
            return make().eval()
    finally:
        torch.set_default_dtype(prev)


def _model(case, w):
    c = _config(case)
    if "tok_emb.weight" not in w:   # a block alone: the embedding and head are not used
        c["vocab_size"] = 16
    model = _module(DTYPES[case["dtype"]], lambda: fa.ForgeModel(fa.ModelConfig(**c)))
    with torch.no_grad():
        for name, p in model.named_parameters():
            if name in w:
                p.copy_(w[name])
    for layer in model.layers:   # the fused weights that a program's first call lays out once
        layer.attn.qkv_weight()
        layer.mlp.gate_up_weight()
    return model


def _tables(case, lens):
    """Block ids of each row (a random permutation of the pool), as lists."""
    counts = [-(-n // BLOCK) for n in lens]
    ids = list(range(sum(counts) + 5))
    random.Random(case["sizes"] + 1).shuffle(ids)
    out, at = [], 0
    for n in counts:
        out.append(ids[at: at + n])
        at += n
    return out, len(ids)


def _table_tensor(lists):
    t = torch.zeros(len(lists), max(len(x) for x in lists), dtype=torch.int32)
    for i, x in enumerate(lists):
        t[i, : len(x)] = torch.tensor(x, dtype=torch.int32)
    return t


def _caches(g, layers, blocks, heads, hd, dtype):
    """N(0, 1) keys and values of every layer, (layers, blocks, heads, BLOCK, hd)."""
    shape = (layers, blocks, heads, BLOCK, hd)
    return [(_normal(g, *shape[1:], dtype=dtype), _normal(g, *shape[1:], dtype=dtype)) for _ in range(layers)]


def _pool(cfg, blocks, dtype, layout, caches=None):
    pool = fa.PagedKVPool(fa.ModelConfig(**cfg), blocks, BLOCK, dtype=dtype, device=DEV, key_layout=layout)
    for i, (k, v) in enumerate(caches or ()):
        pool.k[i].copy_(k.unflatten(-1, (-1, 8)) if layout == "groups" else k)
        pool.v[i].copy_(v)
    return pool


def _attn_config(case):
    return dict(vocab_size=8, d_model=case["heads"] * case["hd"], n_layers=1, n_heads=case["heads"],
                n_kv_heads=case["kv_heads"], max_seq_len=16)


def _window(lens, t):
    """Positions (B, t) of the last t tokens of each context."""
    return torch.tensor([[n - t + i for i in range(t)] for n in lens])


# the inputs of each kind, from the case and the seed alone
def _decode_inputs(case, seed):
    g = _generator(seed)
    c, dt = _config(case), DTYPES[case["dtype"]]
    lens = _lengths(case, case["batch"])
    lists, blocks = _tables(case, lens)
    w = _weights(case, g)
    caches = _caches(g, c["n_layers"], blocks, c["n_kv_heads"], c["d_model"] // c["n_heads"], dt)
    idx = torch.randint(0, c["vocab_size"], (case["batch"], case["t"]), generator=torch.Generator().manual_seed(seed))
    return c, w, caches, lists, blocks, idx, _window(lens, case["t"])


def _block_inputs(case, seed):
    g = _generator(seed)
    c, dt = _config(case), DTYPES[case["dtype"]]
    lens = _lengths(case, case["batch"])
    lists, blocks = _tables(case, lens)
    w = _weights(case, g)
    caches = _caches(g, 1, blocks, c["n_kv_heads"], c["d_model"] // c["n_heads"], dt)
    x = _normal(g, case["batch"] * case["t"], c["d_model"], dtype=dt)
    return c, w, caches, lists, blocks, x, _window(lens, case["t"])


def _prefill_inputs(case, seed):
    g, r = _generator(seed), torch.Generator().manual_seed(seed)
    c = _config(case)
    lens = _lengths(case, case["rows"])
    lists, blocks = _tables(case, lens)
    tokens = [torch.randint(0, c["vocab_size"], (n,), generator=r).tolist() for n in lens]
    return c, _weights(case, g), lists, blocks, tokens


def _attn_inputs(case, seed):
    g = _generator(seed)
    lens = _lengths(case, case["batch"])
    lists, blocks = _tables(case, lens)
    caches = _caches(g, 1, blocks, case["kv_heads"], case["hd"], torch.bfloat16)
    q = _normal(g, case["batch"], case["t"], case["heads"], case["hd"], dtype=torch.bfloat16)
    return caches, lists, blocks, q, _window(lens, case["t"])


def _attn_prefill_inputs(case, seed):
    g = _generator(seed)
    lens = _lengths(case, case["rows"])
    lists, blocks = _tables(case, lens)
    caches = _caches(g, 1, blocks, case["kv_heads"], case["hd"], torch.bfloat16)
    q = _normal(g, sum(lens), case["heads"], case["hd"], dtype=torch.bfloat16)
    return caches, lists, blocks, q, lens


def _mlp_inputs(case, seed):
    g = _generator(seed)
    c, dt = _config(case), DTYPES[case["dtype"]]
    d, f = c["d_model"], c["ffn_dim"]
    w = {n: _normal(g, r, k, dtype=dt, std=0.02) for n, r, k in (("w_gate", f, d), ("w_up", f, d), ("w_down", d, f))}
    return w, _normal(g, case["m"], d, dtype=dt), _normal(g, case["m"], d, dtype=dt)


def _accept_inputs(case, seed):
    """Target logits N(0, 2^2), the draft's near them, proposals drawn from the draft's distribution,
    a third of the rows each at temperature 1, 0.7 and 0."""
    g, dt = _generator(seed), DTYPES[case["dtype"]]
    b, k, v = case["batch"], case["k"], case["vocab"]
    tgt = _normal(g, b, k + 1, v, dtype=dt, std=2.0)
    dft = (tgt[:, :k].float() + _normal(g, b, k, v, std=0.5)).to(dt)
    temps = torch.tensor([(1.0, 0.7, 0.0)[i % 3] for i in range(b)], device=DEV)
    div = torch.where(temps > 0, temps, torch.ones_like(temps))[:, None]
    xs = torch.empty(b, k, dtype=torch.int32, device=DEV)
    for i in range(k):
        y = dft[:, i].float() / div
        e = torch.empty_like(y).exponential_(generator=g)
        xs[:, i] = torch.where(temps > 0, (y - e.log()).argmax(-1), y.argmax(-1)).int()
    u = torch.rand(b, k, device=DEV, generator=g)
    noise = torch.empty(b, v, device=DEV).exponential_(generator=g)
    return tgt, dft, xs, temps, u, noise


def _sample_inputs(case, seed):
    g, dt = _generator(seed), DTYPES[case["dtype"]]
    x = _normal(g, case["rows"], case["vocab"], dtype=dt, std=2.0)
    noise = torch.empty(case["rows"], case["vocab"], device=DEV).exponential_(generator=g)
    temps = torch.tensor([(0.7, 1.0, 0.0)[i % 3] for i in range(case["rows"])], device=DEV)
    return x, temps, noise


# ------------------------------------------------------------------------------------------------
# a program's state and one pass
# ------------------------------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        c, w, caches, lists, blocks, idx, pos = _decode_inputs(case, seed)
        pool = _pool(c, blocks, DTYPES[case["dtype"]], case["layout"], caches)
        return case, _model(case, w), pool, _table_tensor(lists), idx, pos
    if kind == "forward":
        r = torch.Generator().manual_seed(seed)
        idx = torch.randint(0, _config(case)["vocab_size"], (case["batch"], case["t"]), generator=r)
        return case, _model(case, _weights(case, _generator(seed))), idx
    if kind == "prefill":
        c, w, lists, blocks, tokens = _prefill_inputs(case, seed)
        return case, _model(case, w), _pool(c, blocks, DTYPES[case["dtype"]], "groups"), tokens, lists
    if kind == "block":
        c, w, caches, lists, blocks, x, pos = _block_inputs(case, seed)
        pool = _pool(c, blocks, DTYPES[case["dtype"]], case["layout"], caches)
        model = _model(case, w)
        rope = model.rope_cos.float().contiguous(), model.rope_sin.float().contiguous()
        return case, model, rope, pool, _table_tensor(lists).to(DEV), x, pos.to(torch.int32).to(DEV)
    if kind == "attn":
        caches, lists, blocks, q, pos = _attn_inputs(case, seed)
        pool = _pool(_attn_config(case), blocks, torch.bfloat16, case["layout"], caches)
        return case, pool, _table_tensor(lists).to(DEV), q, pos.to(torch.int32).to(DEV)
    if kind == "attn_prefill":
        caches, lists, blocks, q, lens = _attn_prefill_inputs(case, seed)
        pool = _pool(_attn_config(case), blocks, torch.bfloat16, case["layout"], caches)
        pos = torch.full((len(lens), max(lens)), -1, dtype=torch.int32)
        for i, n in enumerate(lens):
            pos[i, :n] = torch.arange(n, dtype=torch.int32)
        cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
        return case, pool, _table_tensor(lists).to(DEV), q, pos.to(DEV), cu.to(DEV)
    if kind == "mlp":
        w, x, residual = _mlp_inputs(case, seed)
        mlp = _module(DTYPES[case["dtype"]], lambda: fa.model.SwiGLU(fa.ModelConfig(**_config(case)), fa.SINGLE))
        with torch.no_grad():
            for name, t in w.items():
                getattr(mlp, name).weight.copy_(t)
        mlp.gate_up_weight()
        return case, mlp, x, residual
    if kind == "accept":
        return (case,) + _accept_inputs(case, seed)
    return (case,) + _sample_inputs(case, seed)


def run(state):
    case, kind = state[0], state[0]["kind"]
    with torch.no_grad():
        if kind == "decode":
            _, model, pool, tables, idx, pos = state
            return model(idx, pos, pool.views(tables, pos))
        if kind == "forward":
            _, model, idx = state
            return model(idx)
        if kind == "prefill":
            _, model, pool, tokens, lists = state
            return fa.prefill_packed(model, pool, tokens, lists), pool.k_store, pool.v_store
        if kind == "block":
            _, model, rope, pool, tables, x, pos = state
            view = pool.views(tables, pos)[0]
            return model.layers[0].step(x, case["batch"], case["t"], pos, view, rope, next_norm=model.norm)
        if kind == "attn":
            _, pool, tables, q, pos = state
            return ops.paged_attention(q, pool.layout(0), tables, pos, case["hd"] ** -0.5)
        if kind == "attn_prefill":
            _, pool, tables, q, pos, cu = state
            return ops.paged_attention_varlen(q, pool.layout(0), tables, pos, cu, case["hd"] ** -0.5)
        if kind == "mlp":
            _, mlp, x, residual = state
            return mlp(x, residual=residual)
        if kind == "accept":
            _, tgt, dft, xs, temps, u, noise = state
            return ops.spec_accept(tgt, dft, xs, None, temps, u, noise)
        _, x, temps, noise = state
        return ops.sample_logits(x, temps, noise), ops.probs_from_logits(x[:1], 0.7)


# ------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ------------------------------------------------------------------------------------------------
def _layer_weights(c):
    d, hd = c["d_model"], c["d_model"] // c["n_heads"]
    return d * (c["n_heads"] + 2 * c["n_kv_heads"]) * hd + c["n_heads"] * hd * d + 3 * d * c["ffn_dim"]


def _causal(lens, t=None):
    """Query-key pairs: the last t tokens of each context (all of them when t is None)."""
    return sum(n * (n + 1) // 2 if t is None else t * n - t * (t - 1) // 2 for n in lens)


def work(case):
    kind = case["kind"]
    s = 4 if case.get("dtype") == "f32" else 2
    if kind in ("decode", "forward", "prefill", "block"):
        c = _config(case)
        hd, v = c["d_model"] // c["n_heads"], c["vocab_size"]
        kv = 2 * c["n_kv_heads"] * hd * s   # bytes of one token's keys and values in one layer
        if kind in ("decode", "block"):
            lens, t = _lengths(case, case["batch"]), case["t"]
            m, pairs, cached = case["batch"] * t, _causal(lens, t), sum(lens) - case["batch"] * t
        elif kind == "forward":
            lens = [case["t"]] * case["batch"]
            m, pairs, cached = sum(lens), _causal(lens), 0
        else:
            lens = _lengths(case, case["rows"])
            m, pairs, cached = sum(lens), _causal(lens), 0
        flops = c["n_layers"] * (2.0 * m * _layer_weights(c) + 4.0 * c["n_heads"] * hd * pairs)
        nbytes = c["n_layers"] * (_layer_weights(c) * s + kv * (cached + m))
        if kind == "block":
            return {"bytes": nbytes + 3 * m * c["d_model"] * s, "flops": flops}
        out = case["rows"] if kind == "prefill" else m
        flops += 2.0 * out * v * c["d_model"]
        return {"bytes": nbytes + v * c["d_model"] * s + out * v * s, "flops": flops}
    if kind in ("attn", "attn_prefill"):
        lens = _lengths(case, case["batch"] if kind == "attn" else case["rows"])
        m = case["batch"] * case["t"] if kind == "attn" else sum(lens)
        pairs = _causal(lens, case["t"] if kind == "attn" else None)
        return {"bytes": 4.0 * sum(lens) * case["kv_heads"] * case["hd"] + 4.0 * m * case["heads"] * case["hd"],
                "flops": 4.0 * case["heads"] * case["hd"] * pairs}
    if kind == "mlp":
        c = _config(case)
        n = 3 * c["d_model"] * c["ffn_dim"]
        return {"bytes": n * s + 3.0 * case["m"] * c["d_model"] * s, "flops": 2.0 * case["m"] * n}
    if kind == "accept":
        b, k, v = case["batch"], case["k"], case["vocab"]
        return {"bytes": float(s * b * v * (2 * k + 1) + 4 * b * v + 8 * b * k + 4 * b * (k + 2)), "flops": 0.0}
    return {"bytes": float(case["rows"] * case["vocab"] * (s + 4) + 4 * case["vocab"]), "flops": 0.0}


def tolerance(case):
    # about four times what each kind is off the 64-bit results (measured: 7e-7 in float32, 0.017 after four
    # bf16 blocks and the head, 0.006 after one block, 0.004 after an MLP, 0.002 after attention); decisions and
    # draws are whole numbers, which another order of the softmax sums moves only where two candidates nearly tie
    kind = case["kind"]
    if kind in ("accept", "sample"):
        return {"rel": 1e-5, "differ": 0.01}
    if kind in ("decode", "forward") and case["dtype"] == "f32":
        return {"rel": 1e-5}
    return {"rel": {"decode": 3e-2, "prefill": 3e-2, "block": 2e-2, "attn": 1e-2, "attn_prefill": 1e-2,
                    "mlp": 1.5e-2}[kind]}


# ------------------------------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ------------------------------------------------------------------------------------------------
def _norm64(x, w, eps=1e-5):
    return x * (x.square().mean(-1, keepdim=True) + eps).rsqrt() * w.double()


def _rotate64(x, pos, theta=10000.0):
    """Half-split rotary of x (tokens, heads, hd) at pos (tokens,); the angles are float32, as the tables' are."""
    hd = x.shape[-1]
    inv = 1.0 / (theta ** (torch.arange(0, hd, 2).float() / hd))
    ang = (pos.float().cpu()[:, None] * inv[None]).to(x.device).double()
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x[..., : hd // 2], x[..., hd // 2:]
    return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)


def _attend64(q, k, v, pos):
    """q (T, H, hd) at pos over keys and values (Hkv, S, hd), causal by position: (T, H, hd)."""
    t, h, hd = q.shape
    hkv, s, _ = k.shape
    seen = torch.arange(s, device=q.device)
    out = torch.empty_like(q)
    for a in range(0, t, 1024):   # in pieces of queries, to bound the scores' memory
        qq = q[a: a + 1024].view(-1, hkv, h // hkv, hd).permute(1, 2, 0, 3)
        n = qq.shape[2]
        sc = torch.matmul(qq.reshape(hkv, -1, hd), k.transpose(1, 2).contiguous()).view(hkv, h // hkv, n, s) * hd ** -0.5
        sc = sc.masked_fill(seen > pos[a: a + 1024, None], float("-inf"))
        o = torch.matmul(sc.softmax(-1).reshape(hkv, -1, s), v).view(hkv, h // hkv, n, hd)
        out[a: a + 1024] = o.permute(2, 0, 1, 3).reshape(n, h, hd)
    return out


def _rows64(cache, blocks, n):
    """The first n positions of a row's cache (blocks, heads, BLOCK, hd): (heads, n, hd)."""
    x = cache[torch.tensor(blocks, device=cache.device)].double()
    return x.permute(1, 0, 2, 3).reshape(x.shape[1], -1, x.shape[3])[:, :n]


def _block64(c, w, p, x, rows, cached):
    """One decoder block on x (tokens, d). rows: (first token, tokens, their positions) of each sequence;
    cached(row): its earlier keys and values (Hkv, S, hd), or None."""
    h, hkv = c["n_heads"], c["n_kv_heads"]
    hd = c["d_model"] // h
    lin = lambda y, name: torch.matmul(y, w[f"{p}{name}.weight"].double().t().contiguous())
    y = _norm64(x, w[f"{p}attn_norm.weight"])
    q, k, v = (lin(y, f"attn.{n}").view(x.shape[0], -1, hd) for n in ("wq", "wk", "wv"))
    att = torch.empty_like(q)
    for r, (a, n, pos) in enumerate(rows):
        qr, kr = _rotate64(q[a: a + n], pos), _rotate64(k[a: a + n], pos).transpose(0, 1)
        vr = v[a: a + n].transpose(0, 1)
        old = cached(r)
        if old is not None:
            kr, vr = torch.cat([old[0], kr], 1), torch.cat([old[1], vr], 1)
        att[a: a + n] = _attend64(qr, kr.contiguous(), vr.contiguous(), pos)
    x = x + lin(att.view(x.shape[0], -1), "attn.wo")
    y = _norm64(x, w[f"{p}mlp_norm.weight"])
    return x + lin(torch.nn.functional.silu(lin(y, "mlp.w_gate")) * lin(y, "mlp.w_up"), "mlp.w_down")


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind in ("decode", "forward", "prefill"):
            return _model64(case, seed)
        if kind == "block":
            c, w, caches, lists, _, x, pos = _block_inputs(case, seed)
            t = case["t"]
            pos = pos.to(DEV)
            rows = [(r * t, t, pos[r]) for r in range(case["batch"])]
            got = _block64(c, w, "layers.0.", x.double(), rows, lambda r: tuple(
                _rows64(m, lists[r], int(pos[r, 0])) for m in caches[0]))
            return got, _norm64(got, w["norm.weight"])
        if kind == "attn":
            caches, lists, _, q, pos = _attn_inputs(case, seed)
            pos = pos.to(DEV)
            return torch.stack([_attend64(q[r].double(), *(_rows64(m, lists[r], int(pos[r, -1]) + 1) for m in caches[0]),
                                          pos[r]) for r in range(case["batch"])])
        if kind == "attn_prefill":
            caches, lists, _, q, lens = _attn_prefill_inputs(case, seed)
            out, a = [], 0
            for r, n in enumerate(lens):
                out.append(_attend64(q[a: a + n].double(), *(_rows64(m, lists[r], n) for m in caches[0]),
                                     torch.arange(n, device=DEV)))
                a += n
            return torch.cat(out)
        if kind == "mlp":
            w, x, residual = _mlp_inputs(case, seed)
            lin = lambda y, name: torch.matmul(y, w[name].double().t().contiguous())
            x = x.double()
            return residual.double() + lin(torch.nn.functional.silu(lin(x, "w_gate")) * lin(x, "w_up"), "w_down")
        if kind == "accept":
            return _accept64(case, seed)
        x, temps, noise = _sample_inputs(case, seed)
        return _draw64(x, temps, noise), (x[:1].double() / 0.7).softmax(-1)


def _model64(case, seed):
    if case["kind"] == "decode":
        c, w, caches, lists, _, idx, pos = _decode_inputs(case, seed)
        t, pos = case["t"], pos.to(DEV)
        rows = [(r * t, t, pos[r]) for r in range(case["batch"])]
        cached = lambda i: (lambda r: tuple(_rows64(m, lists[r], int(pos[r, 0])) for m in caches[i]))
        idx = idx.reshape(-1)
    else:
        if case["kind"] == "forward":
            c, w = _config(case), _weights(case, _generator(seed))
            r = torch.Generator().manual_seed(seed)
            idx = torch.randint(0, c["vocab_size"], (case["batch"], case["t"]), generator=r)
            lens, idx = [case["t"]] * case["batch"], idx.reshape(-1)
        else:
            c, w, _, _, tokens = _prefill_inputs(case, seed)
            lens, idx = [len(x) for x in tokens], torch.tensor([x for t in tokens for x in t])
        starts = [sum(lens[:r]) for r in range(len(lens))]
        rows = [(a, n, torch.arange(n, device=DEV)) for a, n in zip(starts, lens)]
        cached = lambda i: (lambda r: None)
    x = w["tok_emb.weight"][idx.to(DEV)].double()
    for i in range(c["n_layers"]):
        x = _block64(c, w, f"layers.{i}.", x, rows, cached(i))
    if case["kind"] == "prefill":
        x = x[torch.tensor([a + n - 1 for a, n, _ in rows], device=DEV)]
    y = _norm64(x, w["norm.weight"])
    logits = torch.matmul(y, w["tok_emb.weight"].double().t().contiguous())
    if case["kind"] == "prefill":
        return logits, None, None
    return logits.view(case["batch"], case["t"], -1)


def _probs64(x, temps):
    """softmax(x / T) of rows x (R, V) in 64 bits (T = 1 where it is 0)."""
    return (x.double() / torch.where(temps > 0, temps, torch.ones_like(temps)).double()[:, None]).softmax(-1)


def _draw64(x, temps, noise):
    return torch.where(temps > 0, (_probs64(x, temps) / noise.double()).argmax(-1), x.double().argmax(-1))


def _accept64(case, seed):
    """Rejection sampling in 64 bits: accept proposal i while u_i < min(1, p_i / q_i), then one draw from the
    rejected position's residual max(p - q, 0), or from the target past the last proposal; a row at
    temperature 0 accepts while the proposal is the target's argmax."""
    tgt, dft, xs, temps, u, noise = _accept_inputs(case, seed)
    b, k, v = case["batch"], case["k"], case["vocab"]
    greedy = temps == 0
    out = torch.full((b, k + 1), -1, dtype=torch.int32, device=DEV)
    n = torch.zeros(b, dtype=torch.int32, device=DEV)
    live = torch.ones(b, dtype=torch.bool, device=DEV)
    extra = torch.zeros(b, dtype=torch.int32, device=DEV)
    for i in range(k + 1):
        p = _probs64(tgt[:, i], temps)
        p = torch.where(greedy[:, None], torch.nn.functional.one_hot(tgt[:, i].double().argmax(-1), v).double(), p)
        if i < k:
            q = _probs64(dft[:, i], temps)
            q = torch.where(greedy[:, None], torch.nn.functional.one_hot(dft[:, i].double().argmax(-1), v).double(), q)
            x = xs[:, i].long()[:, None]
            px, qx = p.gather(1, x)[:, 0], q.gather(1, x)[:, 0]
            ok = u[:, i].double() < torch.where(qx > 0, px / qx, torch.ones_like(px)).clamp(max=1)
            w = (p - q).clamp(min=0)
            w = torch.where(w.sum(-1, keepdim=True) > 0, w, p)
        else:
            ok, w = torch.zeros_like(live), p
        stop = live & ~ok
        extra = torch.where(stop, (w / noise.double()).argmax(-1).int(), extra)
        if i < k:
            go = live & ok
            out[:, i] = torch.where(go, xs[:, i], out[:, i])
            n += go.int()
        live = live & ok
    out.scatter_(1, n.long()[:, None], extra[:, None])
    return out, n
