"""Attention of one new token for many heads and sequences, against float64, on both sides of the numbers of workgroups and of keys where the launch changes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [64, 65, 256, 257])
@pytest.mark.parametrize("kv", [1, 15, 17, 100, 192, 193, 700])
def test_one_token(agpu, dev, rows, kv):
    """Scores are sums of 64 fp32 products (64 roundings of |q| |k| / 8 at most), weights exponentials good to 2^-23, the result a mean
    of values: off by twice what a weight is off by, relatively, times the largest value, and by the roundings of its own sum."""
    from async_gpu_amd import ops
    g = torch.Generator(device=dev).manual_seed(rows * kv)
    q = torch.randn((rows, 1, 64), generator=g, device=dev)
    k, v = (torch.randn((rows, kv + 3, 64), generator=g, device=dev) for _ in range(2))
    k[:, kv:], v[:, kv:] = float("nan"), float("nan")  # behind the context
    o = ops.attention(q, k, v, kv, kv - 1)[:, 0]
    s = (q.double() * k[:, :kv].double()).sum(-1) / 8
    ref = (torch.softmax(s, -1)[..., None] * v[:, :kv].double()).sum(1)
    reach = q[:, 0].norm(dim=1) * k[:, :kv].norm(dim=2).amax(1) / 8
    bound = 2 * (2.0 ** -23 + 64 * 2.0 ** -24 * reach + kv ** 0.5 * 2.0 ** -24) * v[:, :kv].abs().amax((1, 2))
    assert torch.all((o.double() - ref).abs().amax(1) <= bound)
