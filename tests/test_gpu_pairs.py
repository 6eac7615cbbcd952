"""The Linear of many rows on f16 pairs (csrc/int4_gemm_pairs.hip) against 64-bit products of the same inputs."""
import numpy as np
import pytest
import torch

from conftest import build_oracle_model, gpu_config

pytestmark = pytest.mark.gpu


def _inputs(dev, M, K, N, g, seed=1):
    from async_gpu_amd import _lib, ops
    gen = torch.Generator(device=dev).manual_seed(seed + M + K + N)
    rn = lambda *s: torch.randn(s, generator=gen, device=dev)
    packed, scales = ops.int4_quantize(rn(K, N) * 0.02, g, _lib.QUANT_SCRIPT)
    return rn, rn(M, K), packed, scales, ops.int4_dequantize(packed, scales, g).double()


def _rounding(K):
    """Of the sum of |x| |w|: an x is split to 23 bits, the 32 k of a sum of their own take at most eight roundings (two 16-k steps of two pieces, each
    in two halves), and a value that comes first into an accumulator is rounded with each of the at most K / 64 sums that follow."""
    return (2 + 8 + K / 64) * 2.0**-24


# With a LayerNorm in front the rows are turned into pairs by its launch.  One tile more than needed in rows and columns, an odd number of columns,
# K not a multiple of 64 nor of the groups' turns, two groups of waves (more tiles than CUs) and four, tiles sliced along K (all of them,
# or those beyond a whole round), long K, wide scale groups, and a last column block of two columns.
@pytest.mark.parametrize("M,K,N,g", [(333, 768, 3072, 32), (520, 800, 2049, 32), (3713, 1600, 130, 64), (1601, 768, 1500, 128),
                                     (1300, 2080, 521, 32), (200, 6400, 1601, 32), (2000, 3104, 1280, 32), (130, 8192, 900, 256)])
def test_linear_on_pairs_matches_64_bits(agpu, dev, M, K, N, g):
    from async_gpu_amd import _lib, ops
    rn, x, packed, scales, w = _inputs(dev, M, K, N, g)
    gamma, beta, bias, res = 1 + 0.1 * rn(K), 0.1 * rn(K), rn(N), rn(M, N)
    x = 2 * x + 0.5
    x[1] *= torch.exp(8 * rn(K).clamp(-2, 2))  # values of very different size in a row
    y = ops.int4_linear(x, packed, scales, bias=bias, residual=res, group=g, ln=(gamma, beta, 1e-5), flags=_lib.EPI_GELU_TANH)
    xn = torch.nn.functional.layer_norm(x.double(), (K,), gamma.double(), beta.double(), 1e-5)
    lin = xn @ w + bias.double()
    ref = torch.nn.functional.gelu(lin, approximate="tanh") + res.double()
    # the normalised rows are off by up to four roundings more; GELU and the sums with bias and residual are done in fp32 (GELU's slope
    # stays below 1.2)
    bound = 1.2 * (_rounding(K) + 4 * 2.0**-24) * (xn.abs() @ w.abs()) + 4e-7 * (lin.abs() + ref.abs() + res.abs() + 1)
    assert bool(((y.double() - ref).abs() <= bound).all()), float(((y.double() - ref).abs() / bound).max())
    assert torch.equal(y, ops.int4_linear(x, packed, scales, bias=bias, residual=res, group=g, ln=(gamma, beta, 1e-5), flags=_lib.EPI_GELU_TANH))


@pytest.mark.parametrize("M,K,N,g", [(1000, 1280, 3840, 32), (1100, 6400, 1601, 64)])
def test_plain_linear_on_pairs_over_the_dynamic_range(agpu, dev, M, K, N, g):
    """Rows of very different magnitude side by side, zeros, a NaN, an infinity and tiny rows; what is below 2^-39 of a row's largest value may be lost."""
    from async_gpu_amd import ops
    rn, x, packed, scales, w = _inputs(dev, M, K, N, g)
    x[0:8] *= torch.exp(torch.linspace(-12, 4, K, device=dev))
    x[8:12] *= 1e-20
    x[12:16] *= 1e-33
    x[16:20] *= 1e30
    x[20] = torch.where(torch.arange(K, device=dev) == 5, torch.tensor(3e4, device=dev), x[20])
    x[21] = 0.0
    clean = ops.int4_linear(x, packed, scales, group=g)
    xd = x.double()
    bound = _rounding(K) * (xd.abs() @ w.abs()) + 2.0**-39 * xd.abs().amax(1, keepdim=True) * w.abs().sum(0) + 1e-42  # (the smallest results are denormal numbers)
    err = (clean.double() - xd @ w).abs()
    assert bool((err <= bound).all()), float((err / bound).max())
    assert bool((clean[21] == 0).all())
    x[3, K // 2] = float("nan")
    x[33, K - 1] = float("inf")
    y = ops.int4_linear(x, packed, scales, group=g)
    assert bool(y[3].isnan().all()) and not bool(y[33].isfinite().any())
    keep = [m for m in range(M) if m not in (3, 33)]
    assert torch.equal(y[keep], clean[keep])


@pytest.mark.parametrize("size", [2.0 ** 116, 2.0 ** -110])  # of scales of about 2^-7
def test_scales_of_extreme_size(agpu, dev, size):
    """Rows and weights times powers of two: the same bits times that power."""
    from async_gpu_amd import ops
    _, x, packed, scales, _ = _inputs(dev, 1000, 1280, 3840, 32)
    y = ops.int4_linear(x, packed, scales, group=32)
    assert torch.equal(ops.int4_linear(x, packed, scales * size, group=32), y * size)
    part = min(max(size, 2.0 ** -90), 2.0 ** 90)  # (x has elements of 2^-20, which are to stay what they are)
    assert torch.equal(ops.int4_linear(x / part, packed, scales * size, group=32), y * (size / part))
    assert torch.isfinite(y * size).all()


def test_sliced_tiles_hand_over_the_same_bits(agpu, dev):
    """Partial sums through memory with the fast hand-over and with release and acquire fences."""
    from async_gpu_amd import ops
    rn, x, packed, scales, _ = _inputs(dev, 200, 6400, 1600, 32)
    ln = (1 + 0.1 * rn(6400), 0.1 * rn(6400), 1e-5)
    fast = ops.int4_linear(x, packed, scales, group=32, ln=ln)
    ctx = ops.context(0)
    ctx.call("agpu_ctx_set_strict_sync", 1)
    try:
        assert torch.equal(fast, ops.int4_linear(x, packed, scales, group=32, ln=ln))
    finally:
        ctx.call("agpu_ctx_set_strict_sync", 0)


# Elements 2^26 above the rest of their row meet weights of zero in every other column: what such a column is made of has its 24 bits all the same.  Some rows of
# a tile, and none of some tiles; two groups of waves and four, tiles sliced along K, a last column that stands alone; a LayerNorm whose gains do it to all rows.
@pytest.mark.parametrize("M,K,N,g,ln", [(1000, 1280, 3840, 32, False), (2048, 1600, 4801, 64, False), (1000, 5120, 1280, 32, False), (3000, 3104, 1601, 32, False),
                                        (333, 768, 3072, 128, True), (1601, 768, 1500, 32, True), (200, 6400, 1601, 32, True)])
def test_rows_with_elements_of_very_different_size(agpu, dev, M, K, N, g, ln):
    from async_gpu_amd import _lib, ops
    rn, x, packed, scales, _ = _inputs(dev, M, K, N, g)
    large = torch.arange(K, device=dev) // 8 % 2 == 0
    packed[::2, ::2] = -0x77777778  # 0x88888888: eight weights of zero
    w = ops.int4_dequantize(packed, scales, g).double()
    assert not w[large][:, ::2].any()
    bias, res = rn(N), rn(M, N)
    norm, rows = None, x.double()
    if ln:
        gamma, beta = torch.where(large, 2.0 ** 26, 1.0) * (1 + 0.1 * rn(K)), 0.1 * rn(K)
        norm, rows = (gamma, beta, 1e-5), torch.nn.functional.layer_norm(rows, (K,), gamma.double(), beta.double(), 1e-5)
    else:
        m = torch.arange(M, device=dev)
        x[:, large] *= torch.where((m % 3 == 0) & (m // 64 % 2 == 0), 2.0 ** 26, 1.0)[:, None]
        rows = x.double()
    y = ops.int4_linear(x, packed, scales, bias=bias, residual=res, group=g, ln=norm)
    ref = rows @ w + bias.double() + res.double()
    # on three pieces a 32 k's sum takes twelve roundings, and there are K / 32 of them; normalised rows four more; bias and residual one each
    bound = (12 + K / 32 + 4 * ln) * 2.0**-24 * (rows.abs() @ w.abs()) + 2.0**-23 * (ref.abs() + bias.abs() + res.abs())
    assert bool(((y.double() - ref).abs() <= bound).all())


def test_scratch_that_holds_no_pairs_takes_the_other_kernel(agpu, dev):
    """A caller's small scratch: the same Linear on three bf16 pieces, which needs none."""
    from async_gpu_amd import ops
    _, x, packed, scales, w = _inputs(dev, 1000, 1280, 3840, 32)
    y = ops.int4_linear(x, packed, scales, group=32)
    ctx = ops.context(0)
    small = torch.empty(1 << 20, dtype=torch.uint8, device=dev)
    ctx.call("agpu_ctx_set_workspace", small.data_ptr(), small.numel())
    try:
        z = ops.int4_linear(x, packed, scales, group=32)
        torch.cuda.synchronize()
    finally:
        ctx.call("agpu_ctx_set_workspace", None, 0)
    ref = x.double() @ w
    bound = 4e-7 * (x.double().abs() @ w.abs())
    assert bool(((y.double() - ref).abs() <= bound).all()) and bool(((z.double() - ref).abs() <= bound).all())


def _model_pair(orc, cfg, seed, max_batch, change=None):
    from async_gpu_amd import gpt2, workloads
    w = workloads.gpt2_fp32_weights(cfg, seed, std=0.08, nonzero_bias=True, random_ln=True)
    if change:
        change(w)
    qz = workloads.quantize_gpt2(w, 32, lambda wt, g: orc.quantize_weight_int4(wt, g, orc.SCRIPT))
    return qz, build_oracle_model(cfg, qz), gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg, max_batch=max_batch), qz)


@pytest.mark.parametrize("batch,prompt_len,d", [(4, 320, 768), (1, 777, 1280), (3, 420, 768)])
def test_model_with_gains_of_very_different_size(orc, agpu, dev, batch, prompt_len, d):
    """LayerNorms with gains of 2^34 where the Linear behind them has no weights: K and V, their fragments, and the FFN's rows, of rows that are not for pairs."""
    from async_gpu_amd import workloads
    cfg = dict(n_layer=1, n_embd=d, n_head=d // 64, vocab=331, n_positions=1024)
    large = np.arange(d) // 8 % 2 == 0

    def change(w):
        L = w["layers"][0]
        for norm, linear in (("ln1_g", "qkv_w"), ("ln2_g", "fc_w")):
            L[norm][large] = 2.0 ** 34
            L[linear][large] = 0.0

    _, om, gm = _model_pair(orc, cfg, 43, batch, change)
    prompts = workloads.random_prompt(cfg, 5, prompt_len, batch=batch).reshape(batch, prompt_len)
    got = gm.forward_cached(prompts)
    for b in sorted({0, batch - 1}):
        om.reset_cache()
        ref = om.forward(prompts[b], all_rows=True)
        assert np.abs(got[b] - ref).max() <= 2e-4 * max(1.0, np.abs(ref).max()), b


# The rows' size in channels that the Linears ignore (whose sums are zero, so that LayerNorm gives the others all their bits), or in the others gains that make
# up for it: V and the FFN's rows are far below what their weights allow.  Every attention kernel of prompts, QKV on pairs, on three pieces and on few rows;
# the chunks are of V and rows in the cache.
@pytest.mark.parametrize("batch,prompt_len,d,chunks,ffn", [(41, 31, 768, 1, True), (4, 320, 768, 1, True), (16, 256, 768, 1, True), (1, 777, 1280, 1, True),
                                                           (1, 288, 768, 1, False), (1, 489, 1024, 1, False), (1, 777, 1280, 1, False), (3, 150, 768, 3, False)])
def test_model_far_below_the_bounds_of_its_weights(orc, agpu, dev, batch, prompt_len, d, chunks, ffn):
    from async_gpu_amd import gpt2, workloads
    cfg = dict(n_layer=1, n_embd=d, n_head=d // 64, vocab=331, n_positions=1024)
    w = workloads.gpt2_fp32_weights(cfg, 43, std=0.08, nonzero_bias=False, random_ln=False)
    layer, ignored = w["layers"][0], np.arange(d) // 32 % 2 == 0
    pairs = np.flatnonzero(ignored).reshape(-1, 2)
    for rows in (w["wte"], w["wpe"]):
        rows[:, ~ignored] *= 2.0 ** -20
        rows[:, pairs[:, 1]] = -rows[:, pairs[:, 0]]
    for norm in ("ln1_g", "ln2_g"):
        layer[norm][~ignored] *= 2.0 ** 20
    for name in ("qkv_w", "fc_w"):
        layer[name][ignored] = 0.0
    for name in ("proj_w", "fc_proj_w"):
        layer[name][:, ignored] = 0.0
        layer[name][:, ~ignored] *= 2.0 ** -20
    if not ffn:  # what the attention gives, alone, and K within its bound (far below it the scores alone would have the block worked out on fp32 operands)
        layer["qkv_w"][:, d:2 * d] *= 2.0 ** -20
        layer["fc_proj_w"][:] = 0.0
        layer["proj_w"] *= 64.0
    w["lnf_g"][ignored] = 0.0
    w["lnf_g"][~ignored] *= 2.0 ** 40
    qz = workloads.quantize_gpt2(w, 32, lambda wt, g: orc.quantize_weight_int4(wt, g, orc.SCRIPT))
    om, gm = build_oracle_model(cfg, qz), gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg, max_batch=batch), qz)
    prompts = workloads.random_prompt(cfg, 5, prompt_len * chunks, batch=batch).reshape(batch, prompt_len * chunks)
    got = np.concatenate([gm.forward_cached(prompts[:, i * prompt_len:(i + 1) * prompt_len]) for i in range(chunks)], axis=1)
    for b in sorted({0, batch - 1}):
        om.reset_cache()
        ref = om.forward(prompts[b], all_rows=True)
        # on floats 7e-7 (2-norm, of the logits), on pairs under the bounds' scales 2e-5
        assert np.linalg.norm(got[b] - ref) <= 2e-6 * np.linalg.norm(ref), b


# The attention and the first FFN Linear leave their outputs as the pairs of the Linear behind them: every attention kernel of prompts (one key tile;
# rows of K and V; fragments, with one block of queries a workgroup and with two), rows that are no whole blocks, some heads.
@pytest.mark.parametrize("batch,prompt_len,d", [(41, 31, 768), (3, 420, 768), (1, 777, 1280), (4, 320, 768), (16, 256, 768)])
def test_prompts_whose_linears_hand_pairs_on(orc, agpu, dev, batch, prompt_len, d):
    from async_gpu_amd import workloads
    cfg = dict(n_layer=1, n_embd=d, n_head=d // 64, vocab=331, n_positions=1024)
    qz, om, gm = _model_pair(orc, cfg, 31, batch)
    prompts = workloads.random_prompt(cfg, 5, prompt_len, batch=batch).reshape(batch, prompt_len)
    got = gm.forward_cached(prompts)
    for b in sorted({0, batch - 1}):
        om.reset_cache()
        ref = om.forward(prompts[b], all_rows=True)
        # logits of one layer: 2e-4 of the largest, as in the other model tests
        assert np.abs(got[b] - ref).max() <= 2e-4 * max(1.0, np.abs(ref).max()), b


def test_rows_behind_a_prompt_leave_nothing_in_v(orc, agpu, dev):
    """A prompt of 260 rows ends four rows into a tile of keys.  Of the 28 behind it the QKV Linear's sums are the bias alone, here six times what V's columns
    can be in a row of the prompt (the bias takes back what LayerNorm's offset of 6 gives): as f16 that would be infinite, and NaN under a weight of zero."""
    from async_gpu_amd import gpt2, workloads
    d = 1024
    cfg = dict(n_layer=1, n_embd=d, n_head=16, vocab=331, n_positions=320)
    w = workloads.gpt2_fp32_weights(cfg, 41, std=0.08, nonzero_bias=True, random_ln=True)
    L = w["layers"][0]
    L["qkv_w"][:, 2 * d:] = np.abs(L["qkv_w"][:, 2 * d:]) + 0.05
    L["ln1_g"][:], L["ln1_b"][:] = 1.0, 6.0
    qz = workloads.quantize_gpt2(w, 32, lambda wt, g: orc.quantize_weight_int4(wt, g, orc.SCRIPT))
    packed, scales, bias = qz["layers"][0]["qkv"]
    q = ((packed.reshape(d // 8, 1, 3 * d) >> (4 * np.arange(8, dtype=np.uint32)).reshape(1, 8, 1)) & 15).reshape(d, 3 * d).astype(np.float64) - 8
    weights = q * np.repeat(scales.reshape(d // 32, 3 * d), 32, axis=0)
    bias = (bias - 6.0 * weights.sum(0)).astype(np.float32)
    qz["layers"][0]["qkv"] = (packed, scales, bias)
    # beyond f16 in every column of V, where the largest bound comes to 2^15 at most (and 2^14 at least)
    bound = np.sqrt(d * (weights[:, 2 * d:] ** 2).sum(0)).max()
    assert np.abs(bias[2 * d:]).min() > 4 * bound
    om, gm = build_oracle_model(cfg, qz), gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg, max_batch=1), qz)
    prompt = workloads.random_prompt(cfg, 5, 260)
    got, ref = gm.forward_cached(prompt.reshape(1, -1))[0], om.forward(prompt, all_rows=True)
    # V is a difference of numbers some hundred times as large, fp32 sums of 1024 terms: 2^-24 sqrt(1024) 400 = 8e-4 of it
    assert np.abs(got - ref).max() <= 2e-3 * np.abs(ref).max()


def test_columns_far_out_are_not_handed_on_as_pairs(orc, agpu, dev):
    """A V column and an FFN column 10^9 times the others: a scale that holds them would leave the others too few bits."""
    from async_gpu_amd import workloads
    cfg = dict(n_layer=1, n_embd=768, n_head=12, vocab=331, n_positions=1024)

    def change(w):
        w["layers"][0]["qkv_w"][:, 2 * 768 + 5] *= 1e9
        w["layers"][0]["proj_w"][5, :] = 0.0  # nothing of it comes through
        w["layers"][0]["fc_w"][:, 7] *= 1e9
        w["layers"][0]["fc_proj_w"][7, :] = 0.0

    qz, om, gm = _model_pair(orc, cfg, 33, 3, change)
    prompts = workloads.random_prompt(cfg, 5, 420, batch=3)
    got = gm.forward_cached(prompts)
    ref = om.forward(prompts[0], all_rows=True)
    assert np.abs(got[0] - ref).max() <= 2e-4 * max(1.0, np.abs(ref).max())


def test_columns_of_very_different_size_keep_their_bits(orc, agpu, dev):
    """Half of V's columns 2^-15 of the others, the rows of the projection that take them up 2^15 times: the same model, power by power of two."""
    from async_gpu_amd import gpt2, workloads
    cfg = dict(n_layer=1, n_embd=768, n_head=12, vocab=331, n_positions=1024)
    qz, _, gm = _model_pair(orc, cfg, 37, 3)
    prompts = workloads.random_prompt(cfg, 5, 420, batch=3)
    plain = gm.forward_cached(prompts)
    L = qz["layers"][0]
    small = 2 * 768 + np.flatnonzero(np.arange(768) // 32 % 2 == 0)  # the first 32 dimensions of every head: a scale group of the projection each
    (qp, qs, qb), (pp, ps, pb) = L["qkv"], L["proj"]
    qs, qb, ps = qs.copy(), qb.copy(), ps.copy()
    qs[:, small] *= 2.0 ** -15
    qb[small] *= 2.0 ** -15
    ps[::2] *= 2.0 ** 15
    L["qkv"], L["proj"] = (qp, qs, qb), (pp, ps, pb)
    scaled = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg, max_batch=3), qz).forward_cached(prompts)
    # both are within a few 1e-7 (rms, of the logits') of the exact ones
    assert np.sqrt(((scaled - plain).astype(np.float64) ** 2).mean() / (plain.astype(np.float64) ** 2).mean()) < 1e-6


def test_rows_that_are_handed_on_have_no_second_place(orc, agpu, dev):
    """What a prompt takes of device memory: its FFN rows stand there as pairs or as floats, not both, and come as floats once weights are not for pairs."""
    cfg = dict(n_layer=1, n_embd=1280, n_head=20, vocab=331, n_positions=1024)
    from async_gpu_amd import gpt2, workloads
    qz, _, gm = _model_pair(orc, cfg, 39, 8)
    prompts = workloads.random_prompt(cfg, 5, 1024, batch=8)
    rows, d = prompts.size, cfg["n_embd"]
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    first = gm.forward_cached(prompts, all_rows=False)
    torch.cuda.synchronize()
    # hidden rows, QKV, normalised rows, K and V fragments, pairs of d and of 4 d (4 bytes a number each), and 5 MB a buffer for their granularity
    assert before - torch.cuda.mem_get_info()[0] < 4 * rows * d * (1 + 3 + 1 + 2 + 4 + 4) + 50e6
    packed, scales, bias = qz["layers"][0]["fc"]
    far_out = scales.copy()
    far_out[:, 7] *= 1e9
    gm.set_int4_linear(0, "fc", packed, far_out, bias)
    gm.reset_cache()
    qz["layers"][0]["fc"] = (packed, far_out, bias)
    fresh = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg, max_batch=8), qz)
    assert np.array_equal(gm.forward_cached(prompts, all_rows=False), fresh.forward_cached(prompts, all_rows=False))
    gm.set_int4_linear(0, "fc", packed, scales, bias)
    gm.reset_cache()
    assert np.array_equal(gm.forward_cached(prompts, all_rows=False), first)


def test_cached_rows_of_replaced_weights_stay_within_range(orc, agpu, dev):
    """The attention's range follows from the weights; V rows in the cache may be of weights that have been replaced since."""
    from async_gpu_amd import gpt2, workloads
    cfg = dict(n_layer=1, n_embd=768, n_head=12, vocab=331, n_positions=128)
    qz, _, gm = _model_pair(orc, cfg, 35, 41)
    one = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg, max_batch=1), qz)
    prompts = workloads.random_prompt(cfg, 5, 62, batch=41)
    L = qz["layers"][0]
    out = []
    for m, p in ((gm, prompts), (one, prompts[:1])):
        m.forward_cached(p[:, :31], all_rows=False)
        m.set_layer_norms(0, L["ln1_g"] * 1e-6, L["ln1_b"] * 1e-6, L["ln2_g"], L["ln2_b"])
        out.append(m.forward_cached(p[:, 31:], all_rows=False)[0])
    assert np.isfinite(out[0]).all() and np.abs(out[0] - out[1]).max() <= 2e-4 * max(1.0, np.abs(out[1]).max())
