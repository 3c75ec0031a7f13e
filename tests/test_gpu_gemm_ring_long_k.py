"""The ring tiles of the 16-bit GEMM at long k: rounds of the ring with and without a rest, k-tiles in odd and even number, k tails,
ragged rows and channels, gate rows that change inside a tile.  Integer operands: every product and sum is exact in fp32, so the
result is bit for bit the rounded integer one."""
import ctypes

import pytest
import torch

from sana_amd import _lib, ops

pytestmark = pytest.mark.gpu

# 17 .. 27 k-tiles (every remainder of the rings' rounds of 4, 6 and 10), the last one of 8, 56, 0, .. values
KS = [1032, 1080, 1152, 1216, 1288, 1344, 1408, 1472, 1536, 1600, 1664, 1720]
# (64 x 64: up to 128 tiles as two workgroups of 32 channels each: 4 x 17 tiles, 3 x 42; whole: 4 x 33)
# Dense weights: with the weights requested ahead, in the loop over whole k-tiles, where that pays (the second shape of a tile, and
# the only one of 64 x 128), else in the other loop, as rows of W apart always are.
TILES = [((64, 32), (195, 1048)), ((64, 64), (195, 2072)), ((64, 64), (465, 1048)), ((64, 32), (192, 2688)), ((64, 32), (129, 1048)),
         ((64, 128), (414, 2336)), ((96, 128), (1281, 2280)), ((96, 128), (1026, 2280)), ((128, 128), (1332, 2496)),
         ((128, 128), (2721, 1048)), ((128, 160), (2349, 1800)), ((192, 128), (1872, 2992)), ((192, 128), (3969, 1176)),
         ((256, 128), (1935, 2968))]


def _ints(*shape, hi=3, seed=0, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(-hi, hi + 1, shape, generator=g).to(dtype)


@pytest.mark.parametrize("tile,shape", TILES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_ring_tiles_are_exact_at_every_length_of_k(cuda, tile, shape, dtype):
    M, N = shape
    a_all, w_all = _ints(M, max(KS), seed=1, dtype=dtype).to(cuda), _ints(N, max(KS) + 8, seed=2, dtype=dtype).to(cuda)
    bias, gate = _ints(N, hi=9, seed=3, dtype=dtype).to(cuda), _ints(3, 1, N, hi=4, seed=4, dtype=dtype).to(cuda)
    res = _ints(3, M // 3, N, hi=99, seed=5, dtype=dtype).to(cuda)
    for K in KS:
        plan = (ctypes.c_int * 4)()
        _lib.check(_lib.load().sana_hip_gemm_plan(M, N, K, plan), "sana_hip_gemm_plan")
        assert tuple(plan) == (*tile, 0, 1), (tuple(plan), tile, K)
        a, dense, apart = a_all[:, :K].contiguous(), w_all[:, :K].contiguous(), w_all[:, :K]   # rows of W one after the other, and not
        y = (a.float() @ dense.float().T + bias.float()).to(dtype)      # |sum| <= 9 k < 2^24: exact in any order
        assert torch.equal(ops.gemm_bf16(a, dense, bias, "bias"), y), K
        assert torch.equal(ops.gemm_bf16(a, apart, bias, "bias"), y), K
        assert torch.equal(ops.gemm_gate_residual(a.view(3, M // 3, K), dense, bias, gate, res), res + gate * y.view(3, M // 3, N)), K


# tokens, channels, k, ranges: ranges of equal and of unequal length, k tails of half a k-tile, ragged rows and channels
RANGES = [((64, 32), (65, 2240, 5600, 8)), ((64, 32), (186, 2240, 5600, 8)), ((64, 32), (891, 448, 5984, 8)), ((64, 32), (2927, 8, 13504, 8)),
          ((64, 64), (390, 2240, 5600, 8)), ((64, 64), (447, 2240, 5600, 8)), ((64, 64), (1161, 720, 5664, 7)),
          ((96, 128), (1230, 2240, 5600, 4)), ((96, 128), (1311, 2296, 8032, 3)), ((96, 128), (804, 3240, 7328, 3)),
          ((192, 128), (2307, 2240, 5600, 2)), ((192, 128), (2559, 2240, 5600, 2)), ((192, 128), (1284, 3944, 5792, 2))]


@pytest.mark.parametrize("tile,shape", RANGES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_ranges_of_k_are_added_up_in_the_tile(cuda, tile, shape, dtype):
    """Long k in ranges: exact on integers, and on other values the bits of the split kernel, which the int8 weights of such shapes take."""
    M, N, K, ranges = shape
    plan = (ctypes.c_int * 4)()
    _lib.check(_lib.load().sana_hip_gemm_plan(M, N, K, plan), "sana_hip_gemm_plan")
    assert tuple(plan) == (*tile, 0, ranges)
    a, w_all = _ints(M, K, seed=1, dtype=dtype).to(cuda), _ints(N, K + 8, seed=2, dtype=dtype).to(cuda)
    dense, apart = w_all[:, :K].contiguous(), w_all[:, :K]
    bias, B = _ints(N, hi=9, seed=3, dtype=dtype).to(cuda), 3 if M % 3 == 0 else 1
    gate, res = _ints(B, 1, N, hi=4, seed=4, dtype=dtype).to(cuda), _ints(B, M // B, N, hi=99, seed=5, dtype=dtype).to(cuda)
    y = (a.float() @ dense.float().T + bias.float()).to(dtype)      # |sum| <= 9 k < 2^24: exact in any order
    assert torch.equal(ops.gemm_bf16(a, dense, bias, "bias"), y)
    assert torch.equal(ops.gemm_bf16(a, apart, bias, "bias"), y)
    assert torch.equal(ops.gemm_gate_residual(a.view(B, M // B, K), dense, bias, gate, res), res + gate * y.view(B, M // B, N))
    if dtype == torch.bfloat16:
        g = torch.Generator().manual_seed(K)
        x, wq = torch.randn(M, K, generator=g).to(dtype).to(cuda), torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8).to(cuda)
        scale = (torch.rand(N, generator=g) * 2e-4 + 1e-4).to(cuda)
        for epilogue in ("bias", "bias_silu"):
            assert torch.equal(ops.gemm_bf16(x, ops.dequant_w8(wq, scale), bias, epilogue),
                               ops.gemm_w8a16(x, wq, scale, bias, epilogue, expand=False))
