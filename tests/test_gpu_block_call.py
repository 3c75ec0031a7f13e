"""The image block as one library call against the same block composed entry point by entry point: the same launches, so the
same bits; and what has to keep the composition does."""
import pytest
import torch

import sana_amd as S
from sana_amd import ops

pytestmark = pytest.mark.gpu


def _block(C, H, dtype, dev, seed, ffn="glumbconv", **kw):
    g = torch.Generator().manual_seed(seed)
    b = S.SanaMSBlock(C, H, mlp_ratio=2.5, attn_type="linear", ffn_type=ffn, **kw)
    with torch.no_grad():
        for p in b.parameters():
            p.copy_(torch.randn(p.shape, generator=g) * (0.3 if p.dim() == 2 and p.shape[0] == 6 else 0.03))
    return b.to(dtype).to(dev).eval()


def _inputs(B, N, C, Nk, dtype, dev, masked, seed=3):
    g = torch.Generator().manual_seed(seed)
    x, y = torch.randn(B, N, C, generator=g).to(dtype).to(dev), torch.randn(B, Nk, C, generator=g).to(dtype).to(dev)
    t = (0.3 * torch.randn(B, 6 * C, generator=g)).to(dtype).to(dev)
    mask = (torch.arange(Nk)[None] < torch.tensor([[max(1, Nk - 5 * b)] for b in range(B)])).to(torch.int16).to(dev)
    return x, y, t, mask if masked else None


def _count(monkeypatch):
    calls, real = [], ops.block
    monkeypatch.setattr(ops, "block", lambda *a, **k: (calls.append(1), real(*a, **k))[1])
    return calls


@pytest.mark.parametrize("C,H,B,HW,Nk,dtype,masked,shared,ffn", [
    (1152, 16, 1, (16, 16), 300, torch.bfloat16, False, True, "glumbconv"),
    (1152, 16, 2, (32, 32), 300, torch.float16, False, True, "glumbconv"),
    (1152, 16, 4, (32, 33), 77, torch.float16, True, False, "glumbconv_linear"),      # f16: any number of tokens
    (2240, 20, 3, (27, 36), 230, torch.bfloat16, True, True, "glumbconv"),
    (2240, 20, 1, (32, 32), 300, torch.bfloat16, False, False, "glumbconv"),          # the point convolution splits k
    (288, 4, 5, (1, 3), 1, torch.bfloat16, False, False, "glumbconv_linear"),         # a few rows, an odd number of heads
])
def test_one_call_gives_the_bits_of_the_composition(cuda, monkeypatch, C, H, B, HW, Nk, dtype, masked, shared, ffn):
    b = _block(C, H, dtype, cuda, C + B, ffn)
    x, y, t, mask = _inputs(B, HW[0] * HW[1], C, Nk, dtype, cuda, masked)
    calls = _count(monkeypatch)
    with torch.no_grad():
        kw = S.StepConditioning([b])(y, t)[0] if shared else {}
        one = b(x, y, t, mask, HW, **kw)
        assert calls == [1]
        monkeypatch.setattr(S.SanaMSBlock, "_one_call", lambda *a: None)
        assert torch.equal(one, b(x, y, t, mask, HW, **kw)) and calls == [1]


def test_what_keeps_the_composition(cuda, monkeypatch):
    """Hooks, replaced layers, q/k norm, int8 weights, many bf16 tokens and odd addresses: the block runs, not in one call."""
    C, H, HW = 1152, 16, (8, 8)
    x, y, t, _ = _inputs(1, 64, C, 20, torch.bfloat16, cuda, False)
    calls = _count(monkeypatch)

    def run(b, x=x, HW=HW):
        with torch.no_grad():
            return b(x, y, t, None, HW)

    b = _block(C, H, torch.bfloat16, cuda, 1)
    ref = run(b)
    assert calls == [1]
    seen = []
    handle = b.attn.proj.register_forward_hook(lambda m, i, o: seen.append(1))
    assert torch.equal(run(b), ref) and seen == [1] and calls == [1]
    handle.remove()

    class Scaled(S.modules.HipLinear):
        def forward(self, x, *a, **k):
            return super().forward(2 * x, *a, **k)

    own = b.attn.qkv
    b.attn.qkv = Scaled(C, 3 * C, bias=False).bfloat16().to(cuda)
    b.attn.qkv.load_state_dict(own.state_dict())
    run(b)
    b.attn.qkv = own
    odd = torch.empty(x.numel() + 8, dtype=x.dtype, device=cuda)[8:].view(x.shape).copy_(x)      # another address, still aligned
    assert calls == [1] and torch.equal(run(b, odd), ref) and calls == [1, 1]
    run(_block(C, H, torch.bfloat16, cuda, 2, qk_norm=True))
    run(_block(C, H, torch.bfloat16, cuda, 2).quantize_w8_())
    big = x.repeat(1, 64, 1)
    run(b, big, (64, 64))
    assert calls == [1, 1]
    with pytest.raises((ops.SanaHipError, RuntimeError)):       # a mask left on the host: refused, as the composition refuses it
        with torch.no_grad():
            b(x, y, t, torch.ones(1, 20), HW)
    assert calls == [1, 1]


@pytest.mark.parametrize("kw,int8", [({}, True), ({"qk_norm": True}, False)])
def test_a_composed_block_decides_the_route_of_its_cross_attention_once(cuda, monkeypatch, kw, int8):
    """The decision walks modules, hooks, strides and pointers on the host, which a small image waits for."""
    b = _block(288, 4, torch.bfloat16, cuda, 1, **kw)
    if int8:
        b.quantize_w8_()
    x, y, t, _ = _inputs(1, 64, 288, 20, torch.bfloat16, cuda, False)
    asked, real = [], S.modules.MultiHeadCrossAttention._on_hip_path
    monkeypatch.setattr(S.modules.MultiHeadCrossAttention, "_on_hip_path", lambda *a: (asked.append(1), real(*a))[1])
    calls = _count(monkeypatch)
    with torch.no_grad():
        b(x, y, t, None, (8, 8))
    assert asked == [1] and not calls
