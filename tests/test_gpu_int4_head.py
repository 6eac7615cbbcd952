"""The int4 LM head of two to sixteen rows with its arg-max and token feed (int4_head_rows_kernel): both layouts of the rows and their edges, widths whose groups
are no multiple of the ring's, scale groups of one to four units, vocabularies that leave workgroups and waves without columns."""
import numpy as np
import pytest

from conftest import gpu_config

pytestmark = pytest.mark.gpu


def _model(orc, rows, heads, vocab, group, last=False, nan_columns=()):
    """A model whose block adds nothing (its scales are zeros): the head sees the embedding rows.  Every token of the vocabulary has a twin, half of it away, of
    the same embedding, so every arg-max is a tie."""
    from async_gpu_amd import gpt2
    d = 64 * heads
    rng = np.random.default_rng(rows * 1000 + heads)
    wte = rng.standard_normal((vocab, d)).astype(np.float32) * 0.02
    wte[vocab // 2:2 * (vocab // 2)] = wte[:vocab // 2]
    zeros = lambda k, n: (np.zeros((k // 8, n), np.uint32), np.zeros((-(-k // group), n), np.float32), np.zeros(n, np.float32))
    layer = dict(qkv=zeros(d, 3 * d), proj=zeros(d, d), fc=zeros(d, 4 * d), fc_proj=zeros(4 * d, d))
    for name in ("ln1", "ln2"):
        layer[name + "_g"], layer[name + "_b"] = np.ones(d, np.float32), np.zeros(d, np.float32)
    packed, scales = orc.quantize_weight_int4(np.ascontiguousarray(wte.T), group, orc.SCRIPT)[:2]
    scales = np.array(scales, np.float32).reshape(-1, vocab)
    scales[:, list(nan_columns)] = np.nan
    qz = dict(wte=wte, wpe=rng.standard_normal((32, d)).astype(np.float32) * 0.02, lnf_g=1 + 0.1 * rng.standard_normal(d).astype(np.float32),
              lnf_b=0.1 * rng.standard_normal(d).astype(np.float32), layers=[layer], lm_head=(np.asarray(packed), scales))
    cfg = dict(n_layer=1, n_embd=d, n_head=heads, vocab=vocab, n_positions=32)
    return gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg, max_batch=rows, group_size=group, argmax_last=last), qz), qz


def _reference(qz, group, tokens, position):
    packed, scales = qz["lm_head"]
    packed = packed.reshape(-1, scales.shape[1])
    q = np.stack([(packed >> (4 * i)) & 15 for i in range(8)], 1).reshape(-1, packed.shape[1]).astype(np.float64) - 8
    x = (qz["wte"][tokens] + qz["wpe"][position]).astype(np.float64)
    x = (x - x.mean(1, keepdims=True)) / np.sqrt(x.var(1, keepdims=True) + 1e-5) * qz["lnf_g"] + qz["lnf_b"]
    return x @ (q * np.repeat(scales.astype(np.float64), group, 0)[:q.shape[0]])


CASES = [(2, 4, 1000, 32), (3, 16, 2049, 64), (4, 5, 64, 32), (5, 12, 515, 128), (8, 25, 1027, 32), (9, 25, 778, 64), (16, 13, 9000, 32), (12, 2, 35, 32),
         (16, 26, 300, 128), (16, 27, 300, 32), (8, 32, 300, 32), (2, 3, 300, 96)]


@pytest.mark.parametrize("rows,heads,vocab,group", CASES)
def test_logits_of_the_int4_head(orc, agpu, dev, rows, heads, vocab, group):
    """Against float64.  LayerNorm rounds an element some four times, the head's sums at 2^-24 of a partial sum in a chain of up to 64 additions over groups of 32:
    0.29 x 2^-24 x sqrt(4 + 64 / 3 + 3 x 3) = 1.0e-7 of the logits in rms.  Twice that is allowed."""
    m, qz = _model(orc, rows, heads, vocab, group)
    tokens = np.random.default_rng(5).integers(0, vocab, (rows, 1)).astype(np.uint32)
    ref = _reference(qz, group, tokens[:, 0], 0)
    got = np.asarray(m.forward_cached(tokens, all_rows=False)).reshape(rows, vocab)
    err = np.sqrt(((got - ref) ** 2).mean() / (ref ** 2).mean())
    print(f"{rows} x {64 * heads}, {vocab} tokens: {err:.3g}")
    assert err <= 2.0e-7
    half = vocab // 2
    assert np.array_equal(got[:, :half], got[:, half:2 * half])


@pytest.mark.parametrize("last", [False, True])
@pytest.mark.parametrize("rows,heads,vocab,group", CASES)
def test_tokens_of_the_int4_head(orc, agpu, dev, rows, heads, vocab, group, last):
    """Ties go to the first or the last of the maximal tokens, NaN never wins; each step is fed the token that the step before has picked."""
    start = np.random.default_rng(6).integers(0, vocab, (rows, 2)).astype(np.uint32)
    for nan in ((), (1, vocab // 2), range(vocab)):
        m, qz = _model(orc, rows, heads, vocab, group, last, nan)
        tokens = np.asarray(m.generate_cached(start, 4, eos=-1)[0]).reshape(rows, -1)[:, -4:]
        fed = start[:, -1]
        for step in range(4):
            ref = _reference(qz, group, fed, 1 + step)
            ref[np.isnan(ref)] = -np.inf
            best = ref.max(1, keepdims=True)
            want = np.zeros(rows, np.int64)
            if len(nan) < vocab:
                # a token and its twin differ by a float64 sum's order at most
                close = ref >= best - 1e-12 * abs(best)
                want = vocab - 1 - close[:, ::-1].argmax(1) if last else close.argmax(1)
                second = np.where(close, -np.inf, ref).max(1)
                sure = (best[:, 0] - second) > 1e-5 * abs(best[:, 0])
                assert sure.mean() >= 0.5
            else:
                sure = np.ones(rows, bool)
            assert np.array_equal(tokens[sure, step], want[sure]), (step, nan)
            fed = tokens[:, step]


@pytest.mark.parametrize("heads,group,batches", [(27, 32, (4, 12, 4, 9)), (3, 96, (3, 2, 5))])
def test_batches_with_and_without_the_head_on_pieces(orc, agpu, dev, heads, group, batches):
    """One model, batches whose int4 head is int4_head_rows_kernel's and such whose head is one on pieces, behind a fold that is worked out when a batch first needs it:
    tokens and the last step's logits are, bit for bit, those of a model that has seen that batch alone."""
    from async_gpu_amd import gpt2, workloads
    cfg = dict(n_layer=2, n_embd=64 * heads, n_head=heads, vocab=301, n_positions=24)
    w = workloads.gpt2_fp32_weights(cfg, 2, std=0.05, nonzero_bias=True, random_ln=True)
    qz = workloads.quantize_gpt2(w, group, lambda wt, g: orc.quantize_weight_int4(wt, g, orc.SCRIPT))

    def model():
        m = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg, max_batch=max(batches), group_size=group), qz)
        m.set_decode_mode(m.DECODE_PER_STAGE)
        return m

    def run(m, batch):
        tokens = m.generate_cached(workloads.random_prompt(cfg, 5, 7, batch=batch), 6, eos=-1)[0]
        return np.asarray(tokens), np.array(m.last_logits(batch))

    one = model()
    for batch in batches:
        for got, alone in zip(run(one, batch), run(model(), batch)):
            assert np.array_equal(got, alone), batch
