"""Heads split from and concatenated into rows: whole numbers of rows a thread takes and remainders, one and four of them, heads that are no whole
float4s and pointers that are not aligned to them."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seq,H,dh", [(1, 1, 64), (5, 3, 64), (333, 12, 64), (2050, 25, 64), (4099, 11, 64), (7, 2, 36), (9, 3, 6)])
@pytest.mark.parametrize("offset", [0, 1])
def test_split_and_concat(agpu, dev, seq, H, dh, offset):
    from async_gpu_amd import ops
    g = torch.Generator(device=dev).manual_seed(seq)
    qkv = torch.randn(seq * 3 * H * dh + offset, generator=g, device=dev)[offset:].view(seq, 3 * H * dh)
    want = qkv.view(seq, 3, H, dh).permute(1, 2, 0, 3)
    parts = ops.split_qkv(qkv, H, dh)
    for got, ref in zip(parts, want):
        assert torch.equal(got.reshape(H, seq, dh), ref)
    heads = torch.empty(H * seq * dh + offset, device=dev)[offset:].view(H, seq, dh)
    heads.copy_(want[1])
    assert torch.equal(ops.concat_heads(heads), qkv[:, H * dh:2 * H * dh])
