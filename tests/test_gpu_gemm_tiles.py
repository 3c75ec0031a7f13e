"""The tile kernels of the 16-bit GEMM at the edges of their tiles: integer operands (every product, sum and bias is exact
in fp32, so the result is bit for bit the rounded integer matrix product), ragged rows and channels, k tails, one and
several tiles per workgroup, gate rows that change inside a tile."""
import pytest
import torch

from sana_amd import ops

pytestmark = pytest.mark.gpu


def _ints(*shape, lo=-3, hi=3, seed=0, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(lo, hi + 1, shape, generator=g).to(dtype)


# (rows, channels, k): 256-token tiles of 256 / 192 / 128 channels, and the two-launch mix of 256 and 192; k of less
# than one k-tile, of whole ones, and with tails of 8, 32 and 56
MANY = [(1030, 8200, 8), (1030, 8200, 64), (1030, 8200, 72), (1030, 8200, 184), (1025, 8208, 160), (2563, 2240, 72),
        (4099, 2240, 136), (8200, 6720, 128), (4352, 4360, 192)]


# tiles of 64 x 64, 64 x 128, 128 x 128 and 128 x 160: one row and eight channels, ragged edges, fewer k-tiles than the
# ring has stages and more, k tails of 8, 32 and 56
FEW = [(1, 8, 8), (65, 72, 40), (200, 264, 184), (33, 16, 320), (206, 3456, 8), (700, 2240, 328), (1500, 1160, 1152),
       (3679, 536, 8), (999, 2248, 392), (2049, 1160, 120), (3671, 1120, 200), (2000, 2232, 1032), (2040, 2240, 2240)]


@pytest.mark.parametrize("M,N,K", MANY + FEW)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_many_token_tiles_are_exact_on_integers(cuda, M, N, K, dtype):
    a, w, bias = (_ints(M, K, seed=1, dtype=dtype).to(cuda), _ints(N, K, seed=2, dtype=dtype).to(cuda),
                  _ints(N, lo=-9, hi=9, seed=3, dtype=dtype).to(cuda))
    ref = a.float() @ w.float().T        # |sum| <= 9 k < 2^24: exact in any order
    assert torch.equal(ops.gemm_bf16(a, w), ref.to(dtype))
    ref = (ref + bias.float()).to(dtype)
    assert torch.equal(ops.gemm_bf16(a, w, bias, "bias"), ref)
    y = ops.gemm_bf16(a, w, bias, "bias_silu")
    want = torch.nn.functional.silu(ref.double())
    # the fp32 sigmoid is good to a few 2^-24, the rounding to the io dtype is half an ulp: at most one ulp apart
    ulp = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10
    assert ((y.double() - want).abs() <= ulp * want.abs() + 1e-7).all()


@pytest.mark.parametrize("B,Ntok,C,K", [(3, 1365, 2240, 72), (41, 100, 2240, 64), (2, 4100, 2240, 136), (1, 4096, 4360, 64),
                                           (7, 9, 72, 40), (5, 140, 2240, 328), (9, 111, 2248, 392), (3, 667, 2232, 1032)])
def test_many_token_gated_residual_across_batch_boundaries(cuda, B, Ntok, C, K):
    a, w, bias = _ints(B, Ntok, K, seed=1).to(cuda), _ints(C, K, seed=2).to(cuda), _ints(C, lo=-9, hi=9, seed=3).to(cuda)
    gate, res = _ints(B, 1, C, lo=-4, hi=4, seed=4).to(cuda), _ints(B, Ntok, C, lo=-99, hi=99, seed=5).to(cuda)
    y = (a.float() @ w.float().T + bias.float()).bfloat16()
    assert torch.equal(ops.gemm_gate_residual(a, w, bias, gate, res), res + gate * y)   # the stock pair's roundings
