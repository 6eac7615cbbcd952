"""Prompts and chunks of few rows whose LayerNorms are inside the Linears (RowsLn: statistics of 32 columns left by whatever writes the residual stream): tiles of 32, 64
and 96 columns, rows that fill the last tile of 32 or not, widths of an odd number of statistics, several prompts, chunks behind cached positions;
and prompts and chunks of at most sixteen rows, whose K and V rows the Linear of the few writes into the cache."""
import ctypes as C

import numpy as np
import pytest

from conftest import build_oracle_model, gpu_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,batch,lengths,group", [(12, 1, (97,), 32), (12, 1, (128, 100), 64), (16, 1, (65, 150), 32), (16, 3, (33,), 128),
                                                       (9, 1, (161,), 32), (13, 2, (64, 49), 32), (15, 1, (66,), 32), (17, 1, (120,), 32), (20, 1, (100,), 64),
                                                       (2, 1, (49, 17), 32), (4, 3, (11,), 64), (8, 1, (30, 64), 32), (16, 1, (33,), 32),
                                                       (12, 3, (5, 4), 32), (5, 1, (9, 16), 64), (16, 8, (2, 2), 32), (25, 1, (2, 3, 12), 32), (3, 5, (3, 2), 24)])
def test_logits_behind_chunks_of_few_rows(orc, agpu, dev, heads, batch, lengths, group):
    """All logits of two layers against the f64 oracle; rows of the residual stream with a mean of 3.5 standard deviations.  Each of the eight
    Linears and five LayerNorms rounds at some 1e-7 of its result's rms, the head on many rows at 5e-7: sqrt(13 x 1e-14 + 25e-14) = 6.2e-7.  Twice that is allowed."""
    from async_gpu_amd import gpt2, workloads
    cfg = dict(n_layer=2, n_embd=64 * heads, n_head=heads, vocab=300, n_positions=260)
    w = workloads.gpt2_fp32_weights(cfg, 7, std=0.02, nonzero_bias=True, random_ln=True)
    w["wpe"] = w["wpe"] + np.float32(0.1)
    qz = workloads.quantize_gpt2(w, group, lambda wt, g: orc.quantize_weight_int4(wt, g, orc.SCRIPT), lm_head_int4=False)
    gm = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg, max_batch=batch, group_size=group, lm_head=gpt2.LM_HEAD_F32), qz)
    om = build_oracle_model(cfg, qz, lm_head_int4=False)
    prompts = [np.stack([workloads.random_prompt(cfg, 50 + b + 10 * i, n) for b in range(batch)]) for i, n in enumerate(lengths)]
    got = [np.asarray(gm.forward_cached(p, all_rows=True)).reshape(batch, p.shape[1], -1) for p in prompts]
    for b in range(batch):
        om.reset_cache()
        for p, g in zip(prompts, got):
            ref = om.forward(p[b], all_rows=True)
            assert np.sqrt(((g[b] - ref) ** 2).sum() / (ref ** 2).sum()) <= 1.24e-6


@pytest.mark.parametrize("heads,n,group", [(2, 49, 32), (12, 97, 32), (15, 66, 64), (16, 65, 32), (16, 150, 32), (20, 100, 64)])
def test_rows_whose_variance_is_no_ordinary_number(orc, agpu, dev, heads, n, group):
    """A row of 1e20 normal numbers, whose variance overflows: 1 / sqrt of it is zero and the LayerNorms give their offsets, as they do in a launch of their own.  A row of 1e-20
    normal numbers without an epsilon: its variance is 1e-40, to 2^-150 / 1e-40 = 0.7e-5 of it, so that its rstd is off by 0.35e-5 at each of three roundings
    (mean of squares, merge, division); twice that is allowed of its logits, and three times the bound above, which is of all rows together, of any other row."""
    from async_gpu_amd import gpt2, workloads
    cfg = dict(n_layer=2, n_embd=64 * heads, n_head=heads, vocab=300, n_positions=160)
    w = workloads.gpt2_fp32_weights(cfg, 9, std=0.02, nonzero_bias=True, random_ln=True)
    tiny, rng = n // 2, np.random.default_rng(heads)
    w["wpe"][n - 1] = 1e20 * rng.standard_normal(64 * heads)
    w["wpe"][tiny], w["wte"][299] = 0.0, 1e-20 * rng.standard_normal(64 * heads)
    qz = workloads.quantize_gpt2(w, group, lambda wt, g: orc.quantize_weight_int4(wt, g, orc.SCRIPT), lm_head_int4=False)
    tokens = workloads.random_prompt(dict(cfg, vocab=299), 3, n)
    tokens[tiny] = 299
    gm = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg, group_size=group, lm_head=gpt2.LM_HEAD_F32, layer_norm_epsilon=0.0), qz)
    got = np.asarray(gm.forward_cached(tokens.reshape(1, -1), all_rows=True)).reshape(n, -1)
    om = build_oracle_model(dict(cfg, eps=0.0), qz, lm_head_int4=False)
    ref = om.forward(tokens, all_rows=True)
    ref[-1] = qz["lnf_b"].astype(np.float64) @ qz["wte"].astype(np.float64).T
    err = np.sqrt(((got - ref) ** 2).sum(1) / (ref ** 2).sum(1))
    assert err[tiny] <= 2.2e-5 and np.delete(err, tiny).max() <= 3.7e-6, err
    gm.reset_cache()
    assert np.array_equal(np.asarray(gm.forward_cached(tokens.reshape(1, -1), all_rows=True)).reshape(n, -1), got)


@pytest.mark.parametrize("heads,n", [(2, 49), (12, 128), (16, 150), (4, 300), (12, 9)])
def test_the_same_forward_stage_by_stage(orc, agpu, dev, heads, n):
    """forward_profiled, forward_diagnostic and forward_early_exit with every layer: the bits of the forward's logits, also where its blocks are of few rows (all but
    the last two lengths), and the cache that it leaves."""
    import io
    from async_gpu_amd import gpt2, workloads
    cfg = dict(n_layer=3, n_embd=64 * heads, n_head=heads, vocab=300, n_positions=310)
    w = workloads.gpt2_fp32_weights(cfg, 11, std=0.05, nonzero_bias=True, random_ln=True)
    qz = workloads.quantize_gpt2(w, 32, lambda wt, g: orc.quantize_weight_int4(wt, g, orc.SCRIPT))
    gm = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg), qz)
    tokens = workloads.random_prompt(cfg, 4, n + 1)
    prompt, more = tokens[:n], tokens[n:].reshape(1, 1)
    ref = gm.forward_cached(prompt.reshape(1, -1), all_rows=False)[0]
    step = np.array(gm.forward_cached(more, all_rows=False))
    for logits in (lambda: gm.forward_profiled(prompt)[0], lambda: gm.forward_diagnostic(prompt, out=io.StringIO())[0]):
        gm.reset_cache()
        assert np.array_equal(logits(), ref)
        assert np.array_equal(np.array(gm.forward_cached(more, all_rows=False)), step)
    gm.reset_cache()
    whole = np.array(gm.forward_cached(prompt.reshape(1, -1), all_rows=True)).reshape(n, -1)
    logits, used = gm.forward_early_exit(prompt, 1.1)
    assert used == cfg["n_layer"] and np.array_equal(np.asarray(logits).reshape(n, -1), whole)


@pytest.mark.parametrize("m,k,n,group", [(17, 3072, 64, 32), (33, 3104, 100, 32), (128, 3072, 768, 32), (200, 3072, 768, 64), (150, 4096, 1024, 128), (250, 4096, 1001, 32),
                                         (60, 5120, 1280, 32), (160, 6400, 1600, 32), (18, 9216, 37, 256)])
def test_linears_of_few_rows_and_long_k_in_slices(agpu, dev, m, k, n, group):
    """Two to eight slices of K a tile, widths that leave a tile partial, K that no number of slices divides: against float64, the same bits again from the counters
    that the first call has left, where the scratch has room for the sums of 64 slices of a tile only, and not in slices at all (calls that share their scratch).  Sums of up to 288 scale groups in eight waves round at 2^-24 of
    a partial sum each: 0.29 x 2^-24 x sqrt(288 / 8 + 8 + 8 + 32 / 3) = 1.4e-7 of the result in rms.  Twice that is allowed."""
    import torch
    from async_gpu_amd import _lib, ops
    g = torch.Generator(device="cuda").manual_seed(m)
    randn = lambda *shape: torch.randn(shape, generator=g, device="cuda")
    x, bias, residual = randn(m, k), randn(n), randn(m, n)
    packed, scales = ops.int4_quantize(randn(k, n) * 0.02, group, _lib.QUANT_SCRIPT)
    ref = x.double() @ ops.int4_dequantize(packed, scales, group).double() + bias.double() + residual.double()
    ctx = ops.context(0)
    first = ops.int4_linear(x, packed, scales, bias, residual=residual, group=group)
    assert torch.equal(first, ops.int4_linear(x, packed, scales, bias, residual=residual, group=group))
    small = torch.empty(1 << 20, dtype=torch.uint8, device="cuda")
    ctx.call("agpu_ctx_set_workspace", small.data_ptr(), small.numel())
    try:
        little_room = ops.int4_linear(x, packed, scales, bias, residual=residual, group=group)
        torch.cuda.synchronize()
    finally:
        ctx.call("agpu_ctx_set_workspace", None, 0)
    unsplit, err = torch.empty_like(first), C.create_string_buffer(256)
    assert _lib.cdll().agpu_int4_linear_static(0, torch.cuda.current_stream().cuda_stream, x.data_ptr(), packed.data_ptr(), scales.data_ptr(), bias.data_ptr(), residual.data_ptr(),
                                               unsplit.data_ptr(), m, n, k, group, 0, err, 256) == 0, err.value
    for y in (first, little_room, unsplit):
        assert ((y.double() - ref).norm() / ref.norm()).item() <= 2.8e-7
