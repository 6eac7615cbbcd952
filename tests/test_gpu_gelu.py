"""GELU from the hardware's exponential and reciprocal (gelu_tanh_dev, gelu_quick_dev): errors against float64 where the result is a normal number, and what is no number."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,factor,cubic,least", [(0, 2 * np.sqrt(2 / np.pi), 0.044715, -10.05), (1, 1.702, 0.0, -52.1)])
def test_errors_and_special_values(agpu, dev, mode, factor, cubic, least):
    """From the last x whose 2^e is below 2^128 on (results of 3e-38; behind it the divisor overflows and they are zero).  The exponent e of 2^e (2^e beside 1: e counts at
    2^e / (1 + 2^e)) is three roundings of up to 2^-24 and two constants of up to 2^-25, which share the sum, away: 7 x 2^-25 |e| ln 2 of 2^e at most; the exponential 2^-23, the
    sum 2^-24, the quotient 2^-24 + 2^-44, the product with its own: 2.5 x 2^-24 together at most."""
    import torch
    from async_gpu_amd import ops
    x = torch.cat([torch.linspace(least, -6, 1 << 18, device=dev), torch.linspace(-6, 30, 1 << 20, device=dev), torch.randn(1 << 20, device=dev, generator=torch.Generator(device=dev).manual_seed(1)),
                   torch.logspace(-30, 0, 4096, device=dev), -torch.logspace(-30, 0, 4096, device=dev)])
    y, z = ops.gelu(x, mode).double(), x.double()
    e = factor * (z + cubic * z ** 3)
    ref = z / (1 + torch.exp(-e))
    weight = 1 / (1 + torch.exp(e))  # 2^e / (1 + 2^e) of the exponent -e / ln 2
    bound = (7 * 2.0**-25 * e.abs() * weight + (1 + 2 * weight + 1.5) * 2.0**-24) * ref.abs() + 1e-44
    assert bool(((y - ref).abs() <= bound).all())
    special = ops.gelu(torch.tensor([np.inf, -np.inf, np.nan, 0.0, 1e30, -1e30, -100.0], device=dev), mode).cpu().numpy()
    assert special[0] == np.inf and np.isnan(special[2]) and special[4] == np.float32(1e30)
    assert np.all(special[[3, 5, 6]] == 0.0)
