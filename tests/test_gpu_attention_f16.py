"""Prefill attention on f16 pairs against float64: every shape of workgroup at the edges of its blocks and of the rule that picks it,
key tiles whose sizes differ, and queries that see (almost) nothing."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(ops, q, k, v, by_dimension=False):
    """A score is a sum of 64 products in fp32 and of operands good to 2^-24 of the largest of their tile: off by at most (64 + 3) roundings
    of |q| |k| / 8, which the weight is off by relatively, beside the exponential's 2^-22 and the sum of its n; a result, by
    twice that of the largest value its query's key tiles hold, and the roundings of its own sum.  by_dimension: of the largest value that the query itself
    sees in that dimension, and 2^-39 of its tiles'."""
    n = q.shape[1]
    o = ops.attention(q, k, v)
    seen = torch.ones(n, n, device=q.device, dtype=torch.bool).tril()
    for h in range(0, q.shape[0], max(1, q.shape[0] // 3)):
        s = (q[h].double() @ k[h].double().T / 8).masked_fill(~seen, -float("inf"))
        ref = torch.softmax(s, -1) @ v[h].double()
        tiles = torch.nn.functional.pad(v[h].abs().amax(1), (0, -n % 32)).view(-1, 32).amax(1)
        largest = torch.cummax(tiles, 0).values.repeat_interleave(32)[:n]
        norms = k[h].norm(dim=1)
        reach = q[h].norm(dim=1) * torch.cummax(torch.nn.functional.pad(norms, (0, -n % 32)).view(-1, 32).amax(1), 0).values.repeat_interleave(32)[:n] / 8
        bound = 2 * (2.0 ** -22 + 67 * 2.0 ** -24 * reach + n ** 0.5 * 2.0 ** -24) * largest
        err = (o[h].double() - ref).abs()
        if by_dimension:
            bound = (bound / largest)[:, None] * torch.cummax(v[h].abs(), 0).values + 2.0 ** -39 * largest[:, None]
        else:
            err = err.amax(1)
        assert torch.all(err <= bound.double() + 1e-38), (h, float((err / bound).max()))
    return o


@pytest.mark.parametrize("H,n", [(2, 9), (2, 32),                            # one tile
                                 (2, 33), (3, 127), (12, 300), (64, 287),    # rows of K and V: fewer tiles than waves, as many, more; two query blocks in turn
                                 (1, 512), (3, 513), (8, 1024), (1, 2049),  # a workgroup of eight waves per block (8 x 32 blocks: the last one)
                                 (9, 1000), (24, 1024),                      # of four waves (24 x 32 = 3 x 256)
                                 (25, 1024), (33, 769), (70, 415)])          # of four waves for two blocks; the second one missing or ragged
def test_shapes(agpu, dev, H, n):
    from async_gpu_amd import ops
    g = torch.Generator(device=dev).manual_seed(n)
    _check(ops, *(torch.randn((H, n, 64), generator=g, device=dev) for _ in range(3)), by_dimension=True)


@pytest.mark.parametrize("H,n", [(3, 320), (3, 520), (16, 640), (50, 600)])
def test_sizes_that_differ(agpu, dev, H, n):
    """Whole key tiles of V up to 10^20 apart (the outputs' unit moves both ways), tiles of zeros, tiny and large queries and keys; scores
    that grow along the keys, so that the reference of the weights moves."""
    from async_gpu_amd import ops
    g = torch.Generator(device=dev).manual_seed(n)
    q, k, v = (torch.randn((H, n, 64), generator=g, device=dev) for _ in range(3))
    tile = torch.arange(n, device=dev) // 32
    _check(ops, q, k, v * (10.0 ** ((tile * 7) % 21 - 10.0))[None, :, None])
    _check(ops, q, k, v * (tile % 3 != 0)[None, :, None])
    dims = 10.0 ** ((torch.arange(64, device=dev) * 3) % 10 - 5.0)
    o = ops.attention(q, k, v * dims)
    assert torch.all((o / dims - ops.attention(q, k, v)).abs() <= 2e-6)  # dimensions of V 10^9 apart: each to its own size
    other = torch.where((torch.arange(64, device=dev) < 32)[None, :] ^ (tile > 3)[:, None], 1e-6, 1.0)  # the first keys unlike the rest
    _check(ops, q, k, v * other)
    _check_to_its_own_size(ops, q, k, v * other)  # 10^-6 of the others or not, dimension by dimension
    _check(ops, q * 1e-12, k * (10.0 ** ((tile * 5) % 9 - 4.0))[None, :, None], v)
    _check(ops, q * 1e-20, k * 1e18, v * 1e-20)
    grow = torch.linspace(0, 3, n, device=dev)[None, :, None]
    _check(ops, q.abs(), k.abs() * grow, v)
    _check(ops, torch.zeros_like(q), k, v)  # (every weight the same)


@pytest.mark.parametrize("H,n", [(12, 800), (2, 300)])  # fragments, of four waves and one block each; rows of K and V
def test_a_bad_key_keeps_to_its_tile(agpu, dev, H, n):
    from async_gpu_amd import ops
    key = 100
    g = torch.Generator(device=dev).manual_seed(n)
    q, k, v = (torch.randn((H, n, 64), generator=g, device=dev) for _ in range(3))
    clean = ops.attention(q, k, v)
    for which, bad in ((v, float("nan")), (v, float("inf")), (k, float("nan"))):
        keep = which[1, key, 5].clone()
        which[1, key, 5] = bad
        o = ops.attention(q, k, v)
        which[1, key, 5] = keep
        assert torch.equal(o[0], clean[0]) and torch.equal(o[1, :96], clean[1, :96])
        assert not torch.isfinite(o[1, key:, 5]).any()


def _check_to_its_own_size(ops, q, k, v, q_offset=0):
    """Every result to the precision of an fp32 sum of its own terms: a weight is off by the roundings of its score (64 products) and its exponential, twice that
    with the sum of the weights, and the sum of the n terms by its own roundings."""
    m, n = q.shape[1], k.shape[1]
    o = ops.attention(q, k, v, kv_len=n, q_offset=q_offset)
    seen = torch.arange(n, device=q.device)[None, :] <= torch.arange(m, device=q.device)[:, None] + q_offset
    assert torch.isfinite(o).all()
    for h in range(0, q.shape[0], max(1, q.shape[0] // 3)):
        p = torch.softmax((q[h].double() @ k[h].double().T / 8).masked_fill(~seen, -float("inf")), -1)
        reach = (q[h].norm(dim=1)[:, None] * torch.cummax(k[h].norm(dim=1), 0).values[q_offset : q_offset + m, None] / 8).double()
        bound = (2 * (2.0 ** -22 + 67 * 2.0 ** -24 * reach) + n ** 0.5 * 2.0 ** -24) * (p @ v[h].double().abs()) + 1e-38
        err = (o[h].double() - p @ v[h].double()).abs()
        assert torch.all(err <= bound), (h, float((err / bound).max()))


# On fragments with a workgroup of eight waves, of four, of four for two blocks; on rows of K and V behind a long context, and alone.
@pytest.mark.parametrize("H,n,q_offset", [(2, 1024, 0), (12, 1024, 0), (25, 1024, 0), (3, 64, 1000), (12, 300, 0)])
def test_values_that_are_nothing_for_whole_tiles(agpu, dev, H, n, q_offset):
    """Tiles of V that are all zeros, or far smaller than those in front of them: results as small as what they are made of."""
    from async_gpu_amd import ops
    g = torch.Generator(device=dev).manual_seed(n)
    m, n = n, n + q_offset
    q, k, v = (torch.randn((H, r, 64), generator=g, device=dev) for r in (m, n, n))
    tile = (torch.arange(n, device=dev) // 32)[None, :, None]
    one_hot = torch.zeros_like(v)
    one_hot[:, 40 + (n - 41) * torch.arange(64, device=dev) // 64, torch.arange(64, device=dev)] = 1.0
    for values in (one_hot, (tile == 1) + 0.0 * v, (tile // 8 == 1) + 0.0 * v, (tile == 4) * v, (tile == 0) * v, v * ((tile == 0) + 1e7 * (tile == 1)), v * torch.where(tile > 1, 1e-20, 1.0)):
        _check_to_its_own_size(ops, q, k, values, q_offset)


@pytest.mark.parametrize("H,n,q_offset", [(12, 800, 0), (25, 1024, 0), (2, 300, 0), (3, 64, 1000)])
def test_an_infinite_key_may_weigh_nothing(agpu, dev, H, n, q_offset):
    """-inf in K times a query that is positive there: a score of -inf, a weight of zero, as on fp32 operands; an infinity in V gives one."""
    from async_gpu_amd import ops
    g = torch.Generator(device=dev).manual_seed(n)
    m, n = n, n + q_offset
    q, k, v = (torch.randn((H, r, 64), generator=g, device=dev) for r in (m, n, n))
    key = 70
    q[1, :, 5] = q[1, :, 5].abs() + 0.1
    k[1, key, 5] = -float("inf")
    o = ops.attention(q, k, v, kv_len=n, q_offset=q_offset)
    seen = torch.arange(n, device=dev)[None, :] <= torch.arange(m, device=dev)[:, None] + q_offset
    s = (q[1].double() @ torch.where(k[1].isfinite(), k[1], 0.0).double().T / 8).masked_fill(~seen, -float("inf"))
    s[:, key] = -float("inf")
    assert (o[1].double() - torch.softmax(s, -1) @ v[1].double()).abs().max() < 1e-5  # (scores of a few units: 1e-6 of them, times the largest value)
    v[1, 3, 7] = float("inf")
    o = ops.attention(q, k, v, kv_len=n, q_offset=q_offset)
    assert torch.all(o[1, 3:, 7] == float("inf")) and torch.isfinite(o[1, :, :7]).all() and torch.isfinite(o[0]).all()


@pytest.mark.parametrize("H,n,q_offset", [(12, 800, 0), (25, 1024, 0), (2, 300, 0), (3, 64, 1000)])
def test_a_key_whose_size_dwarfs_the_others(agpu, dev, H, n, q_offset):
    """One key of 10^9 in a single dimension, where the query is nothing: the scores of the other keys keep their bits."""
    from async_gpu_amd import ops
    g = torch.Generator(device=dev).manual_seed(n)
    m, n = n, n + q_offset
    q, k, v = (torch.randn((H, r, 64), generator=g, device=dev) for r in (m, n, n))
    q[:, :, 9] = 0.0
    clean = ops.attention(q, k, v, kv_len=n, q_offset=q_offset).double()
    k[:, 1, 9] = 1e9  # times zero: the same scores
    assert (ops.attention(q, k, v, kv_len=n, q_offset=q_offset).double() - clean).abs().max() < 1e-5


@pytest.mark.parametrize("H,n,q_offset", [(2, 1024, 0), (12, 1024, 0), (25, 1024, 0), (3, 64, 1000), (12, 300, 0)])
def test_dimensions_and_keys_of_very_different_size(agpu, dev, H, n, q_offset):
    """Within a key tile: dimensions of V that change places behind the first keys, a dimension that is small, values that are zero but for a
    few keys (in every tile, or none of them in the first ones), and a last key far larger than those that most of its tile's queries see."""
    from async_gpu_amd import ops
    g = torch.Generator(device=dev).manual_seed(n)
    m, n = n, n + q_offset
    q, k, v = (torch.randn((H, r, 64), generator=g, device=dev) for r in (m, n, n))
    key, dim = torch.arange(n, device=dev)[None, :, None], torch.arange(64, device=dev)
    swapped = v * torch.where((dim < 32) ^ (key >= 32), 2.0 ** -14, 1.0)
    small = v * torch.where(dim == 17, 1e-6, 1.0)
    few = v * (key % 32 == dim // 2)
    later = v * ((dim < 60) | (key > 96))
    last = v * torch.where(key % 32 == 31, 1e8, 1.0)
    for values in (swapped, small, few, later, last):
        _check_to_its_own_size(ops, q, k, values, q_offset)


@pytest.mark.parametrize("lengths", [(777,), (200, 90)])  # on fragments; on the rows of the cache, from position 0 and behind others
def test_model_whose_scores_are_too_large_for_pairs(orc, agpu, dev, lengths):
    """Scores of some hundreds: products of elements of q and k beyond 2^13, bounds of K from the weights."""
    import numpy as np
    from async_gpu_amd import gpt2, workloads
    from conftest import build_oracle_model, gpu_config
    cfg = dict(n_layer=1, n_embd=768, n_head=12, vocab=331, n_positions=1024)
    w = workloads.gpt2_fp32_weights(cfg, 41, std=0.08, nonzero_bias=True, random_ln=True)
    w["layers"][0]["qkv_w"][:, : 2 * 768] *= 6.0
    qz = workloads.quantize_gpt2(w, 32, lambda wt, g: orc.quantize_weight_int4(wt, g, orc.SCRIPT))
    om, gm = build_oracle_model(cfg, qz), gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg, max_batch=1), qz)
    tokens = workloads.random_prompt(cfg, 5, sum(lengths)).reshape(1, -1)
    ref, at = om.forward(tokens[0], all_rows=True), 0
    for n in lengths:
        got = gm.forward_cached(tokens[:, at : at + n])[0]
        # a score of 500 is off by 500 (64 + 3) 2^-24 at most, a weight by twice that
        assert np.abs(got - ref[at : at + n]).max() <= 4e-3 * np.abs(ref).max()
        rms = np.sqrt(((got - ref[at : at + n]).astype(np.float64) ** 2).mean() / (ref.astype(np.float64) ** 2).mean())
        assert rms < 4e-5, rms  # (hundreds of them, of either sign)
        at += n
