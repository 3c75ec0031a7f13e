"""The additive key bias of a prompt mask in one kernel: bit for bit the stock operators'."""
import pytest
import torch

from sana_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bool, torch.uint8, torch.int8, torch.int16, torch.int32, torch.int64, torch.float32,
                                   torch.float16, torch.bfloat16, torch.float64])
@pytest.mark.parametrize("shape", [(1, 1), (3, 85), (1, 256), (2, 300), (3, 1, 1, 257)])
def test_key_bias(cuda, dtype, shape):
    mask = torch.randint(0, 2 if dtype == torch.bool else 3, shape, generator=torch.Generator().manual_seed(5)).to(cuda).to(dtype)
    assert mask.numel() < 8 or ((mask == 0).any() and (mask == 1).any())
    want = (1.0 - mask.to(torch.float32)) * -10000.0
    got = ops.key_bias(mask)
    assert got.dtype == torch.float32 and got.is_contiguous() and torch.equal(got, want)
    if dtype.is_floating_point:      # fractions as well
        mask = mask / 3
        want = (1.0 - mask.to(torch.float32)) * -10000.0
        assert torch.equal(ops.key_bias(mask), want)
    turned = mask.transpose(0, -1)
    got = ops.key_bias(turned)
    assert got.is_contiguous() and torch.equal(got, want.transpose(0, -1))
