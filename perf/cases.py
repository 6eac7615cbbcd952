"""Performance cases of the int4 GPT-2 path: what a program does with this framework, through its public entry points.

Two kinds of program use it.  Most load a model (Int4Gpt2Model) and generate: greedy or sampled, one sequence or a
batch, or they only want the logits of a text, whole or in chunks over the KV cache.  The others compose the operators
(`ops`) themselves, as the reference's transformer block does, over a prompt or over one new token with their own cache.

listed() names the cases, draw() gives more of the same ranges: model widths of 2 to 25 heads of 64 and 2 to 48 layers,
batches of 1 to 16, prompts of 1 to 1000 tokens, scale groups of 32, 64 and 128, int4 and f32 LM head, and for the
operators 1 to 2048 rows, odd ones among them.  The model shapes are those of workloads.py, bench.py and bench_configs.py (small, medium-,
large- and XL-shaped) with random weights: speed does not depend on their values.
"""
import math

import numpy as np
import torch

import __graft_entry__ as entry

entry.load_package()
from async_gpu_amd import _lib, gpt2, ops  # noqa: E402

DH = 64


def listed():
    return [
        # The headline use: one user, greedy continuation of a short prompt by the small model, token after token.
        dict(name="generate_small_b1", kind="generate", layers=12, heads=12, group=32, head="int4", batch=1, prompt=64, new=128, vocab=50257),
        # A serving batch on the largest model: 16 prompts of 256 tokens, then 64 tokens each.
        dict(name="generate_xl_b16", kind="generate", layers=48, heads=25, group=32, head="int4", batch=16, prompt=256, new=64, vocab=50257),
        # A few users at once on a mid-sized model, a prompt of no round length.
        dict(name="generate_medium_b3", kind="generate", layers=24, heads=16, group=32, head="int4", batch=3, prompt=100, new=64, vocab=50257),
        # What a program written for the reference gets: its default group of 128 and its f32 LM head, 50 tokens from a short
        # prompt as in the example program.
        dict(name="generate_reference_defaults", kind="generate", layers=12, heads=12, group=128, head="f32", batch=1, prompt=7, new=50, vocab=50257),
        # Top-k sampling, one user, large-shaped model: a host draw between any two tokens.
        dict(name="sample_large_top40", kind="sample", layers=36, heads=20, group=32, head="int4", batch=1, prompt=33, new=48, vocab=50257),
        # A long prompt whose next token is wanted (time to first token).
        dict(name="prefill_large_1000", kind="prefill", layers=36, heads=20, group=32, head="int4", batch=1, prompt=1000, vocab=50257),
        # Scoring a text: the logits of every position, the reference's forward() at its benchmark's 128 tokens.
        dict(name="forward_small_128", kind="forward", layers=12, heads=12, group=32, head="int4", batch=1, prompt=128, vocab=50257),
        # A conversation: turns of 150 tokens appended to what is cached already.
        dict(name="chunks_medium_5x150", kind="chunks", layers=24, heads=16, group=32, head="int4", batch=1, prompt=150, chunks=5, vocab=50257),
        # One Linear on one row, the smallest call there is (the MLP's first Linear of the small model).
        dict(name="linear_1x768x3072", kind="linear", rows=1, k=768, n=3072, group=32),
        # One new token through a transformer block put together from operators, with a KV cache of the caller's own.
        dict(name="block_decode_kv777", kind="block_decode", heads=12, group=32, kv=777),
        # The same block over a prompt: a middling, odd number of rows with the reference's group of 128 ...
        dict(name="block_small_333", kind="block", heads=12, group=128, rows=333),
        # ... and the widest over a long one.
        dict(name="block_xl_2048", kind="block", heads=25, group=32, rows=2048),
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["generate", "generate", "generate", "sample", "prefill", "forward", "chunks", "linear", "block_decode", "block"])
    group = rng.choice([32, 32, 32, 64, 128])
    if kind == "linear":
        while True:
            c = dict(kind=kind, rows=_log(rng, 1, 2048), k=8 * _log(rng, 8, 800), n=_log(rng, 64, 6400), group=group)
            if rng.random() < 0.7:  # the widths of Linears are mostly round
                c["k"], c["n"] = 64 * max(1, c["k"] // 64), 64 * max(1, c["n"] // 64)
            return c
    if kind == "block_decode":
        return dict(kind=kind, heads=_log(rng, 2, 25), group=group, kv=_log(rng, 1, 1024))
    if kind == "block":
        return dict(kind=kind, heads=_log(rng, 2, 25), group=group, rows=_log(rng, 1, 2048))
    while True:
        c = dict(kind=kind, layers=_log(rng, 2, 48), heads=_log(rng, 2, 25), group=group, head=rng.choice(["int4", "int4", "int4", "f32"]),
                 batch=1, prompt=_log(rng, 1, 1000), vocab=50257 if rng.random() < 0.7 else rng.randint(500, 50256))
        if kind in ("generate", "prefill"):
            c["batch"] = rng.choice([1, 1, rng.randint(2, 4), rng.randint(5, 16)])
        if kind in ("generate", "sample"):
            c["new"] = _log(rng, 8, 128)
        if kind == "forward":
            c["prompt"] = _log(rng, 1, 256)
        if kind == "chunks":
            c["chunks"] = rng.randint(2, 6)
        # inside the 1024 positions, and no dearer than the largest listed case in steps, prompt work or logits
        if (c["prompt"] * c.get("chunks", 1) + c.get("new", 0) <= 1024 and c["layers"] * c.get("new", 0) <= 48 * 56
                and c["batch"] * c["prompt"] * c.get("chunks", 1) * c["layers"] * c["heads"] ** 2 <= 16 * 256 * 48 * 625):
            return c


# ---- inputs ------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, std=1.0, mean=0.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std + mean


def _int4(g, k, n, group):
    """A trained Linear's likes: N(0, 0.02) weights, quantized as the offline script does."""
    packed, scales = ops.int4_quantize(_randn(g, k, n, std=0.02), group, _lib.QUANT_SCRIPT)
    return packed, scales, _randn(g, n, std=0.02)


def _block(g, d, group):
    w = {name: _int4(g, k, n, group) for name, k, n in (("qkv", d, 3 * d), ("proj", d, d), ("fc", d, 4 * d), ("fc_proj", 4 * d, d))}
    for name in ("ln1_g", "ln2_g"):
        w[name] = _randn(g, d, std=0.1, mean=1.0)
    for name in ("ln1_b", "ln2_b"):
        w[name] = _randn(g, d, std=0.1)
    return w


def _model(case, g):
    d, vocab, group, positions = DH * case["heads"], case["vocab"], case["group"], 1024
    host = lambda t: t.cpu().numpy()
    layers = []
    for _ in range(case["layers"]):
        w = _block(g, d, group)
        layers.append({k: tuple(host(t) for t in v) if isinstance(v, tuple) else host(v) for k, v in w.items()})
    wte = _randn(g, vocab, d, std=0.02)
    qz = dict(wte=host(wte), wpe=host(_randn(g, positions, d, std=0.02)), lnf_g=host(_randn(g, d, std=0.1, mean=1.0)),
              lnf_b=host(_randn(g, d, std=0.1)), layers=layers, lm_head=None)
    if case["head"] == "int4":
        qz["lm_head"] = tuple(host(t) for t in ops.int4_quantize(wte.t().contiguous(), group, _lib.QUANT_SCRIPT))
    config = gpt2.Gpt2Config(case["layers"], d, case["heads"], vocab_size=vocab, n_positions=positions, group_size=group,
                             max_batch=case["batch"], lm_head=gpt2.LM_HEAD_INT4 if case["head"] == "int4" else gpt2.LM_HEAD_F32)
    return gpt2.Int4Gpt2Model.from_quantized(config, qz)


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    state = dict(case=case)
    if kind == "linear":
        state["w"] = _int4(g, case["k"], case["n"], case["group"])
        state["x"] = _randn(g, case["rows"], case["k"])
    elif kind == "block":
        d = DH * case["heads"]
        state["w"] = _block(g, d, case["group"])
        state["x"] = _randn(g, case["rows"], d)
    elif kind == "block_decode":
        d = DH * case["heads"]
        state["w"] = _block(g, d, case["group"])
        state["x"] = _randn(g, 1, d)
        # kv positions are cached, the new token's row goes behind them
        state["k"], state["v"] = (_randn(g, case["heads"], case["kv"] + 1, DH) for _ in range(2))
    else:
        state["model"] = _model(case, g)
        r = np.random.default_rng(seed)
        tokens = r.integers(0, case["vocab"], size=(case["batch"], case["prompt"] * case.get("chunks", 1))).astype(np.uint32)
        state["tokens"] = tokens
        state["chunks"] = np.split(tokens, case.get("chunks", 1), axis=1)
        state["seed"] = seed
    return state


# ---- one pass ----------------------------------------------------------------------------

def _run_block(s):
    """Int4TransformerBlock::forward in operators: x += Attn(LN1 x), x += MLP(LN2 x)."""
    c, w, x = s["case"], s["w"], s["x"]
    heads, group, rows = c["heads"], c["group"], x.shape[0]
    qkv = ops.int4_linear(ops.layer_norm(x, w["ln1_g"], w["ln1_b"]), *w["qkv"], group=group)
    q, k, v = ops.split_qkv(qkv, heads, DH)
    att = ops.multi_head_flash_attention(*(t.view(heads * rows, DH) for t in (q, k, v)), rows, heads, DH)
    h = ops.int4_linear(ops.concat_heads(att.view(heads, rows, DH)), *w["proj"], residual=x, group=group)
    m = ops.int4_linear(ops.layer_norm(h, w["ln2_g"], w["ln2_b"]), *w["fc"], group=group, flags=_lib.EPI_GELU_TANH)
    return ops.int4_linear(m, *w["fc_proj"], residual=h, group=group)


def _run_block_decode(s):
    """The same block for one new token: its K and V rows are appended to the caller's cache, LayerNorm inside the Linears."""
    c, w, x = s["case"], s["w"], s["x"]
    heads, group, kv = c["heads"], c["group"], c["kv"]
    qkv = ops.int4_linear(x, *w["qkv"], group=group, ln=(w["ln1_g"], w["ln1_b"], 1e-5))
    q, k, v = ops.split_qkv(qkv, heads, DH)
    ops.kv_append(k, s["k"], kv)
    ops.kv_append(v, s["v"], kv)
    att = ops.attention(q, s["k"], s["v"], kv_len=kv + 1, q_offset=kv)
    h = ops.int4_linear(ops.concat_heads(att), *w["proj"], residual=x, group=group)
    m = ops.int4_linear(h, *w["fc"], group=group, flags=_lib.EPI_GELU_TANH, ln=(w["ln2_g"], w["ln2_b"], 1e-5))
    return ops.int4_linear(m, *w["fc_proj"], residual=h, group=group), s["k"], s["v"]


def run(state):
    c, kind = state["case"], state["case"]["kind"]
    if kind == "linear":
        return ops.int4_linear(state["x"], *state["w"], group=c["group"])
    if kind == "block":
        return _run_block(state)
    if kind == "block_decode":
        return _run_block_decode(state)
    m = state["model"]
    if kind == "generate":
        tokens, _ = m.generate_cached(state["tokens"], c["new"], eos=-1)
        return tokens, m.last_logits(c["batch"])
    if kind == "sample":
        return m.generate_cached_sampling(state["tokens"], c["new"], 40, 0.8, ops.SimpleRng(state["seed"]), eos=-1), m.last_logits()
    if kind == "forward":
        return m.forward(state["tokens"])
    m.reset_cache()  # prefill, chunks
    return [m.forward_cached(t, all_rows=False) for t in state["chunks"]]


# ---- what a pass cannot do without -------------------------------------------------------

def _linear_bytes(k, n, group):
    return k * n / 2 + math.ceil(k / group) * n * 4 + n * 4


def _block_weights(d, group):
    return sum(_linear_bytes(k, n, group) for k, n in ((d, 3 * d), (d, d), (d, 4 * d), (4 * d, d))) + 4 * d * 4


def _attention_flops(d, new, cached):
    """QK^T and PV of `new` queries behind `cached` positions under the causal mask."""
    return 4 * d * (new * cached + new * (new + 1) / 2)


def work(case):
    kind, group = case["kind"], case["group"]
    if kind == "linear":
        m, k, n = case["rows"], case["k"], case["n"]
        return {"bytes": _linear_bytes(k, n, group) + 4 * m * (k + n), "flops": 2 * m * k * n}
    d = DH * case["heads"]
    if kind == "block":
        m = case["rows"]
        return {"bytes": _block_weights(d, group) + 8 * m * d, "flops": 24 * m * d * d + _attention_flops(d, m, 0)}
    if kind == "block_decode":
        return {"bytes": _block_weights(d, group) + 8 * d + 8 * d * (case["kv"] + 2), "flops": 24 * d * d + _attention_flops(d, 1, case["kv"])}
    layers, batch, vocab, chunks = case["layers"], case["batch"], case["vocab"], case.get("chunks", 1)
    head = _linear_bytes(d, vocab, group) if case["head"] == "int4" else 4 * d * vocab
    weights = layers * _block_weights(d, group) + head
    kv_row = layers * 8 * d
    bytes_, flops, cached = 0, 0, 0
    for _ in range(chunks):  # the prompt: weights once, the cached rows read, the new ones written, embeddings, logits
        new = case["prompt"]
        rows_out = new if kind == "forward" else 1
        bytes_ += weights + batch * (kv_row * (cached + new) + 8 * d * new + 4 * vocab * rows_out)
        flops += batch * (layers * (24 * new * d * d + _attention_flops(d, new, cached)) + 2 * rows_out * d * vocab)
        cached += new
    for _ in range(case.get("new", 1) - 1):  # every further token: weights once for the batch, its cache read
        bytes_ += weights + batch * (kv_row * (cached + 2) + 8 * d)
        flops += batch * (layers * (24 * d * d + _attention_flops(d, 1, cached)) + 2 * d * vocab)
        cached += 1
    if kind in ("generate", "sample"):
        bytes_ += 4 * batch * vocab  # the logits handed out at the end
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """Token ids are whole numbers and stay the same.  Everything is fp32: sums of up to 6400 products in another order
    differ by about 1e-6 of the result, and a model of 48 layers carries that to a few 1e-6 of its logits."""
    return {"rel": 1e-5 if case["kind"] in ("linear", "block", "block_decode") else 3e-5}
