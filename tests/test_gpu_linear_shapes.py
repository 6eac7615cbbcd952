"""Int4 Linears of shapes that only int4_gemm_rows_kernel takes beside the kernels on fp32 operands: K a multiple of 8 but not of 32, and few rows with any number
of columns."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,group", [(3, 8, 1, 32), (17, 16, 33, 32), (32, 24, 64, 64), (33, 40, 375, 32), (16, 1672, 375, 32), (100, 1000, 97, 256), (5, 1024, 31, 32),
                                         (333, 840, 3000, 128), (1000, 328, 2999, 32), (4, 5000, 1001, 32), (64, 4104, 130, 32), (16, 64, 4099, 32), (3, 4128, 33, 32)])
def test_against_float64(agpu, dev, m, k, n, group):
    """Every operand stands in a buffer with 256 bytes of NaN (0xffffffff for the words) on both sides, the output in one of a value that has to be there afterwards.
    Products are exact; a sum over 32 k on three pieces takes twelve roundings at 2^-24 of its terms' size, each scale group one more, the epilogue two."""
    import torch
    from async_gpu_amd import _lib, ops
    g = torch.Generator(device=dev).manual_seed(m + k)
    randn = lambda *shape: torch.randn(shape, generator=g, device=dev)

    def inside(t, around):
        whole = torch.full((t.numel() + 128,), around, dtype=t.dtype, device=dev)
        whole[64:-64] = t.reshape(-1)
        return whole[64:-64].view(t.shape)

    packed, scales = ops.int4_quantize(randn(k, n) * 0.02, group, _lib.QUANT_SCRIPT)
    packed, scales = inside(packed, -1), inside(scales, float("nan"))
    x, bias, residual = (inside(t, float("nan")) for t in (randn(m, k), randn(n), randn(m, n)))
    w = ops.int4_dequantize(packed, scales, group).double()
    out = torch.full((m * n + 128,), 1234.5, device=dev)
    y = out[64:-64].view(m, n)
    ops.context(0).call("agpu_int4_linear", x, packed, scales, bias, residual, y, m, n, k, group, 0)
    ref = x.double() @ w + bias.double() + residual.double()
    bound = (12 + k / 32 + 2) * 2.0**-24 * (x.double().abs() @ w.abs()) + 2.0**-23 * (ref.abs() + bias.abs() + residual.abs())
    assert bool(((y.double() - ref).abs() <= bound).all())
    assert bool((out[:64] == 1234.5).all()) and bool((out[-64:] == 1234.5).all())
    assert torch.equal(y, ops.int4_linear(x, packed, scales, bias, residual=residual, group=group))
