"""The passes around a streamed chunk: the state's cache and the channel-major frame, bit for bit as the stock operators."""
import pytest
import torch

from sana_amd import ops

pytestmark = pytest.mark.gpu


def _stock(state, past, save):
    d = state.shape[-1]
    saved = (state[:, :, 0, :d].clone(), state[:, :, 0, d:].clone()) if save else None
    if past is not None:
        state[:, :, 0, :d] += past[0].to(state)
        state[:, :, 0, d:] += past[1].to(state)
    return saved


@pytest.mark.parametrize("B,h,d", [(1, 20, 112), (2, 1, 32), (3, 7, 32)])
@pytest.mark.parametrize("with_past,save", [(True, True), (True, False), (False, True), (False, False)])
@pytest.mark.parametrize("form", ["as saved", "double", "strided"])
def test_state_cache(cuda, B, h, d, with_past, save, form):
    state = torch.randn(B, h, 1, d + 1, d, device=cuda)
    past = None
    if with_past:
        past = [torch.randn(B, h, d, d, device=cuda), torch.randn(B, h, 1, d, device=cuda)]
        if form == "double":
            past = [t.double() for t in past]
        if form == "strided":
            past[0] = past[0].transpose(2, 3)
    want = state.clone()
    want_saved, got_saved = _stock(want, past, save), ops.state_cache_(state, past, save)
    assert torch.equal(state, want) and (got_saved is None) == (want_saved is None)
    for g, w in zip(got_saved or (), want_saved or ()):
        assert g.shape == w.shape and g.stride() == w.stride() and torch.equal(g, w)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,P,C,off", [(1, 1560, 2240, 0), (2, 63, 64, 1), (1, 65, 72, 3), (3, 1, 8, 0), (2, 130, 136, 0)])
def test_channel_major_frame(cuda, dtype, B, P, C, off):
    cache = torch.randn(B, C, 2, P + off, device=cuda).to(dtype)[..., off:]       # rows at any alignment, two frames
    buf = torch.zeros(B, 2 * P + 1, C, dtype=dtype, device=cuda)
    ops.copy_tokens_(buf[:, :P], cache[:, :, -1].transpose(1, 2))
    assert torch.equal(buf[:, :P], cache[:, :, -1].transpose(1, 2)) and not buf[:, P:].any()
