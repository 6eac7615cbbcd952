"""The Linear of many rows on f16 pairs (csrc/int4_gemm_pairs.hip) against 64-bit products of the same inputs."""
import numpy as np
import pytest
import torch

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
