"""The depthwise kernel's bands of 2, 4 and 8 rows give the same bits: a small image alone (bands of 2 where those are at most
1536 workgroups) and as one of a batch whose launch is large enough for taller bands."""
import pytest
import torch

from sana_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,W,Ch", [(16, 16, 2880), (15, 17, 1440), (1, 5, 8), (2, 16, 136), (3, 33, 128), (22, 16, 2880),
                                    (23, 16, 2880), (12, 12, 5600), (64, 64, 256), (65, 64, 256)])
def test_bands_agree(cuda, dtype, H, W, Ch):
    gen = torch.Generator(device=cuda).manual_seed(H * W)
    rand = lambda *s: torch.randn(*s, generator=gen, device=cuda).to(dtype)  # noqa: E731
    batch = -(-520 // (-(-Ch // 128) * -(-W // 16) * -(-H // 8)))            # 512 workgroups of 8 rows and more
    u, w, b = rand(batch, H, W, 2 * Ch), 0.3 * rand(2 * Ch, 1, 3, 3), rand(2 * Ch)
    many = ops.dwconv3x3_silu_gate(u, w, b)
    for i in (0, batch - 1):
        assert torch.equal(ops.dwconv3x3_silu_gate(u[i:i + 1].contiguous(), w, b)[0], many[i])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("batch,H,W,Ch", [(800, 16, 9, 8), (1600, 13, 16, 8), (420, 27, 17, 136)])
def test_tall_bands_agree(cuda, dtype, batch, H, W, Ch):
    """Bands of 8 rows and whole images (launches of 1536 workgroups and more) against bands of 2."""
    gen = torch.Generator(device=cuda).manual_seed(H * W)
    rand = lambda *s: torch.randn(*s, generator=gen, device=cuda).to(dtype)  # noqa: E731
    u, w, b = rand(batch, H, W, 2 * Ch), 0.3 * rand(2 * Ch, 1, 3, 3), rand(2 * Ch)
    many = ops.dwconv3x3_silu_gate(u, w, b)
    for i in (0, batch // 2, batch - 1):
        assert torch.equal(ops.dwconv3x3_silu_gate(u[i:i + 1].contiguous(), w, b)[0], many[i])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shift", [1, 3, 7])
@pytest.mark.parametrize("bias", [True, False])
def test_taps_on_any_boundary(cuda, dtype, shift, bias):
    """Taps and bias are read in 16- and 4-byte pieces wherever they stand."""
    gen = torch.Generator(device=cuda).manual_seed(shift)
    rand = lambda *s: torch.randn(*s, generator=gen, device=cuda).to(dtype)  # noqa: E731
    H, W, Ch = 6, 19, 200
    u, w, b = rand(2, H, W, 2 * Ch), 0.3 * rand(2 * Ch, 1, 3, 3), rand(2 * Ch)
    ws, bs = torch.zeros(18 * Ch + shift, dtype=dtype, device=cuda), torch.zeros(2 * Ch + shift, dtype=dtype, device=cuda)
    ws[shift:], bs[shift:] = w.flatten(), b
    got = ops.dwconv3x3_silu_gate(u, ws[shift:].view(2 * Ch, 1, 3, 3), bs[shift:] if bias else None)
    assert torch.equal(got, ops.dwconv3x3_silu_gate(u, w, b if bias else None))
