"""Tiles of 16 columns of the Linear on pieces (int4_skinny_px_kernel<.., 1>): the edges of the rule that takes them, K in one and two splits, fewer trips than
waves, outputs left as pieces without statistics; and, inside a decode step, with statistics of 16 columns at both ends of the widths that use them."""
import numpy as np
import pytest

from conftest import to_dev
from test_gpu_model import test_batched_decode_on_pieces_in_the_model as decode_on_pieces  # not collected under this name

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [5, 16])
@pytest.mark.parametrize("K,N,g", [(32, 16, 32), (64, 48, 64), (768, 2304, 32), (768, 4096, 128), (768, 4128, 32), (1280, 3840, 64), (2048, 2048, 32),
                                   (2048, 2080, 32), (512, 100, 32)])
def test_tiles_of_sixteen_columns(agpu, orc, dev, M, K, N, g):
    import torch
    from async_gpu_amd import ops, workloads
    rng = np.random.default_rng(M * 7 + K + N)
    packed, scales, bias = workloads.random_int4_linear(rng, K, N, g, bias=True)
    x = (rng.standard_normal((M, K)) * np.exp(rng.uniform(-2, 2, (M, 1)))).astype(np.float32)
    gamma, beta = (1 + 0.2 * rng.standard_normal(K)).astype(np.float32), (0.2 * rng.standard_normal(K)).astype(np.float32)
    og = (1 + 0.3 * rng.standard_normal(N)).astype(np.float32)
    d = [to_dev(v, dev) for v in (x, gamma, beta, packed, scales, bias, og)]
    y = ops.int4_linear_pieces(d[0], d[3], d[4], bias=d[5], group=g, ln=(d[1], d[2], 1e-5))
    ref = orc.int4_gemm_f64(orc.layer_norm(x, gamma, beta, 1e-5), packed, scales, g, bias=bias)
    # every product carries the rounding of its normalised input (a few 2^-24 of |x| gamma + |mean| gamma + |beta|), the sum that of its accumulators
    bound = (np.abs(x - x.mean(1, keepdims=True)) / x.std(1, keepdims=True) * np.abs(gamma) + np.abs(beta)).astype(np.float64) @ \
        np.abs(orc.int4_dequantize(packed, scales, g)).astype(np.float64)
    assert np.all(np.abs(y.cpu().numpy() - ref) <= 3e-6 * bound + 1e-6)
    if N % 32:
        return
    # tiles of 32 columns or more, which leave statistics: the same sums, the same pieces
    y32, pieces32, _ = ops.int4_linear_pieces(d[0], d[3], d[4], bias=d[5], group=g, ln=(d[1], d[2], 1e-5), out_gamma=d[6], want_pieces=True)
    pieces = torch.zeros_like(pieces32)
    y16 = torch.empty_like(y)
    ops.context(0).call("agpu_int4_linear_pieces", d[0], d[1], d[2], 1e-5, d[3], d[4], d[5], None, y16, M, N, K, g, 0, d[6], pieces, None)
    assert torch.equal(y, y32) and torch.equal(y16, y32)
    assert torch.equal(pieces, pieces32)


@pytest.mark.parametrize("batch,group,d,heads", [(16, 32, 64, 1), (9, 64, 448, 7), (16, 32, 1024, 16), (13, 64, 1088, 17)])
def test_decode_step_with_statistics_of_sixteen_columns(orc, agpu, dev, batch, group, d, heads, monkeypatch):
    """The widest model whose rows' statistics are of 16 columns, and the first of 32, against the oracle and the kernels that split their inputs themselves."""
    decode_on_pieces(orc, agpu, dev, batch, group, d, heads, monkeypatch)


@pytest.mark.parametrize("batch,d,heads", [(9, 64, 1), (16, 1088, 17), (5, 1600, 25)])
def test_a_step_starts_from_its_embedding_rows(orc, agpu, dev, batch, d, heads):
    """px_embed_kernel: a step's rows, its pieces and statistics are those of a prompt of one token through the operators that split their inputs themselves: the logits
    of a prompt's last token, fed alone behind the others, against the same token inside the prompt."""
    from conftest import gpu_config
    from test_gpu_model import _quantized
    from async_gpu_amd import gpt2, workloads
    cfg = dict(n_layer=1, n_embd=d, n_head=heads, vocab=301, n_positions=16)
    _, qz = _quantized(orc, cfg, 5, std=0.05, nonzero_bias=True, random_ln=True)
    tokens = np.asarray(workloads.random_prompt(cfg, 3, 7, batch=batch)).reshape(batch, 7)
    tokens[0, 6], tokens[-1, 6] = 0, 300
    gm = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg, max_batch=batch), qz)
    gm.set_decode_mode(gm.DECODE_PER_STAGE)
    whole = np.asarray(gm.forward_cached(tokens, all_rows=False)).reshape(batch, -1)[:, :301]
    gm.reset_cache()
    gm.forward_cached(tokens[:, :6], all_rows=False)
    step = np.asarray(gm.forward_cached(tokens[:, 6:], all_rows=False)).reshape(batch, -1)[:, :301]
    # one layer, both sides with relative errors of a few 1e-7 of a row's size
    assert np.linalg.norm(step - whole) <= 2e-6 * np.linalg.norm(whole)


@pytest.mark.parametrize("M", [5, 16])
@pytest.mark.parametrize("K,N,g", [(1696, 16, 32), (3072, 768, 512), (3072, 768, 32), (3328, 1360, 64), (3360, 1024, 96), (6400, 1040, 128), (10240, 512, 32), (2208, 2048, 32)])
def test_long_k_in_four_splits(agpu, orc, dev, M, K, N, g):
    """K in splits of whole scale groups, up to four while CUs are idle: just above the longest unsplit K, N on both sides of the CUs, groups that leave a last split
    shorter."""
    import torch
    from async_gpu_amd import ops, workloads
    rng = np.random.default_rng(M + K + N)
    packed, scales, bias = workloads.random_int4_linear(rng, K, N, g, bias=True)
    x = (rng.standard_normal((M, K)) * np.exp(rng.uniform(-2, 2, (M, 1)))).astype(np.float32)
    d = [to_dev(v, dev) for v in (x, packed, scales, bias)]
    ref = orc.int4_gemm_f64(x, packed, scales, g, bias=bias)
    bound = np.abs(x).astype(np.float64) @ np.abs(orc.int4_dequantize(packed, scales, g)).astype(np.float64)
    # the bound of the same Linear's test in test_gpu_ops.py
    y = ops.int4_linear_pieces(d[0], d[1], d[2], bias=d[3], group=g)
    assert np.all(np.abs(y.cpu().numpy() - ref) <= 3e-6 * bound + 1e-6 * np.abs(ref) + 1e-6)
    assert torch.equal(y, ops.int4_linear_pieces(d[0], d[1], d[2], bias=d[3], group=g))
