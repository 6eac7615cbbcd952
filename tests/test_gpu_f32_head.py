"""The f32 LM head that reads the embedding table row by row (gemv_f32_rows_kernel): one and several rows, widths whose last 256 elements are whole,
partial or the only ones, vocabularies that leave workgroups and rows of a wave without a row."""
import numpy as np
import pytest

from conftest import build_oracle_model, gpu_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,heads,vocab", [(1, 4, 63), (2, 5, 257), (3, 12, 1001), (4, 13, 2), (5, 16, 130), (16, 25, 301), (7, 8, 65), (1, 32, 1003)])
def test_logits_and_tokens_of_the_f32_head(orc, agpu, dev, rows, heads, vocab):
    """Logits of the last position of `rows` prompts, and the tokens that follow, against the f64 oracle.  The head's sums of up to 2048 products round
    at 2^-24 of a partial sum in chains of some 16 additions: 0.3 x 4 x 2^-24 = 0.7e-7 of the result; the four Linears of the layer in front
    1e-7 each: 2.1e-7 of the logits' rms (of two tokens one row's logits may both be small).  Twice that is allowed."""
    from async_gpu_amd import gpt2, workloads
    cfg = dict(n_layer=1, n_embd=64 * heads, n_head=heads, vocab=vocab, n_positions=32)
    w = workloads.gpt2_fp32_weights(cfg, 7, std=0.02, nonzero_bias=True, random_ln=True)
    qz = workloads.quantize_gpt2(w, 32, lambda wt, g: orc.quantize_weight_int4(wt, g, orc.SCRIPT), lm_head_int4=False)
    gm = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg, max_batch=rows, lm_head=gpt2.LM_HEAD_F32), qz)
    om = build_oracle_model(cfg, qz, lm_head_int4=False)
    prompts = np.stack([workloads.random_prompt(cfg, 50 + b, 5) for b in range(rows)])
    got = np.asarray(gm.forward_cached(prompts, all_rows=False)).reshape(rows, vocab)
    err = []
    for b in range(rows):
        om.reset_cache()
        ref = om.forward(prompts[b], all_rows=False)[0]
        err.append([((got[b] - ref) ** 2).sum(), (ref ** 2).sum()])
    err = np.sum(err, axis=0)
    assert np.sqrt(err[0] / err[1]) <= 4.2e-7
    tokens, _ = gm.generate_cached(prompts, 6, eos=-1)
    for b in range(rows):
        ref, margins = om.generate(prompts[b], 6, cached=True, eos=-1)
        assert np.array_equal(tokens[b], ref), (b, margins)


@pytest.mark.parametrize("last", [False, True])
@pytest.mark.parametrize("rows,heads,vocab", [(2, 4, 33), (4, 5, 2051), (5, 4, 7), (16, 32, 300), (9, 12, 513)])
def test_ties_of_several_rows_go_to_the_first_or_the_last(agpu, dev, rows, heads, vocab, last):
    """A block that adds nothing and a vocabulary whose tokens have a twin each, half of it away: every arg-max is a tie between two workgroups' candidates, and each
    step is fed the token that the step before has picked."""
    from async_gpu_amd import gpt2
    d, half = 64 * heads, vocab // 2
    rng = np.random.default_rng(rows)
    wte = rng.standard_normal((vocab, d)).astype(np.float32) * 0.02
    wte[half:2 * half] = wte[:half]
    zeros = lambda k, n: (np.zeros((k // 8, n), np.uint32), np.zeros((k // 32, n), np.float32), np.zeros(n, np.float32))
    layer = dict(qkv=zeros(d, 3 * d), proj=zeros(d, d), fc=zeros(d, 4 * d), fc_proj=zeros(4 * d, d))
    for name in ("ln1", "ln2"):
        layer[name + "_g"], layer[name + "_b"] = np.ones(d, np.float32), np.zeros(d, np.float32)
    qz = dict(wte=wte, wpe=rng.standard_normal((32, d)).astype(np.float32) * 0.02, lnf_g=np.ones(d, np.float32), lnf_b=0.1 * rng.standard_normal(d).astype(np.float32),
              layers=[layer], lm_head=None)
    cfg = dict(n_layer=1, n_embd=d, n_head=heads, vocab=vocab, n_positions=32)
    m = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg, max_batch=rows, lm_head=gpt2.LM_HEAD_F32, argmax_last=last), qz)
    start = rng.integers(0, vocab, (rows, 2)).astype(np.uint32)
    tokens = np.asarray(m.generate_cached(start, 4, eos=-1)[0]).reshape(rows, -1)[:, -4:]
    fed = start[:, -1]
    for step in range(4):
        x = (wte[fed] + qz["wpe"][1 + step]).astype(np.float64)
        x = (x - x.mean(1, keepdims=True)) / np.sqrt(x.var(1, keepdims=True) + 1e-5) + qz["lnf_b"]
        ref = x @ wte.T.astype(np.float64)
        best = ref.max(1, keepdims=True)
        close = ref >= best - 1e-12 * abs(best)
        want = vocab - 1 - close[:, ::-1].argmax(1) if last else close.argmax(1)
        sure = best[:, 0] - np.where(close, -np.inf, ref).max(1) > 1e-5 * abs(best[:, 0])
        assert sure.mean() >= 0.5 and np.array_equal(tokens[sure, step], want[sure]), step
        fed = tokens[:, step]
