"""The tile kernels of the 16-bit GEMM at the edges of their tiles: integer operands (every product, sum and bias is exact
in fp32, so the result is bit for bit the rounded integer matrix product), ragged rows and channels, k tails, one and
several tiles per workgroup, gate rows that change inside a tile."""
import ctypes

import pytest
import torch

from sana_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _ints(*shape, lo=-3, hi=3, seed=0, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(lo, hi + 1, shape, generator=g).to(dtype)


# Tile (tokens, channels; "mix": the first channels in tiles of 256 x 256, the rest in 256 x 192, two launches) -> shapes
# (rows, channels, k) that run in it, asserted through the library's own plan: k of less than one k-tile (8, 40), of one (64),
# of an odd and an even number, with tails of 8, 32 and 56; ragged rows and channels; one row; more tiles than workgroups
# that are resident (persistent workgroups then take several).  128 x 160 is not chosen for short k or for many tiles.
TILES = {
    (64, 32): [(1, 8, 8), (65, 72, 40), (200, 264, 184), (33, 16, 320)],
    (64, 64): [(12300, 264, 72)],
    (64, 128): [(206, 3456, 8), (700, 2240, 328), (1500, 1160, 1152), (65, 6728, 40), (515, 6728, 64), (515, 6728, 136)],
    (128, 128): [(1030, 8200, 8), (1030, 8200, 64), (3679, 536, 8), (999, 2248, 392), (2049, 1160, 120), (1030, 6728, 40),
                 (1030, 6728, 184), (4100, 2240, 64)],
    (128, 160): [(3671, 1120, 200), (2000, 2232, 1032), (2040, 2240, 2240), (5121, 776, 136), (5121, 776, 192)],
    (256, 128): [(2563, 2240, 72), (4352, 4360, 192), (2563, 1544, 8), (9999, 1160, 40), (9999, 1160, 64), (16390, 776, 136),
                 (8200, 2240, 136)],
    (256, 192): [(1030, 8200, 72), (1030, 8200, 184), (1025, 8208, 160), (4099, 2240, 136), (6150, 5128, 40), (6150, 5128, 64),
                 (12300, 1288, 192)],
    (256, 256): [(8200, 6720, 128), (4613, 5128, 40), (4613, 5128, 64), (4613, 5128, 184), (1290, 8200, 136), (9999, 1160, 72)],
    "mix": [(8200, 4432, 712), (2563, 8920, 1736)],
}
# the same for the gated residual, (batch entries, tokens of each, channels, k): boundaries between them inside a tile
GATED = {
    (64, 32): [(7, 9, 72, 40), (3, 67, 264, 184)],
    (64, 128): [(5, 140, 2240, 328), (3, 172, 6728, 8)],
    (128, 128): [(9, 111, 2248, 392), (41, 100, 2240, 64), (5, 206, 6728, 40)],
    (128, 160): [(3, 667, 2232, 1032), (3, 1707, 776, 136)],
    (256, 128): [(2, 4100, 2240, 136), (1, 4096, 4360, 64), (3, 855, 1544, 8)],
    (256, 192): [(3, 1365, 2240, 72), (3, 2050, 5128, 40), (7, 147, 8200, 184)],
    (256, 256): [(3, 1538, 5128, 40), (6, 215, 8200, 136)],
    "mix": [(2, 4100, 4432, 712), (3, 855, 8920, 1736)],
}


def _runs_in(tile, M, N, K):
    plan = (ctypes.c_int * 4)()
    _lib.check(_lib.load().sana_hip_gemm_plan(M, N, K, plan), "sana_hip_gemm_plan")
    assert plan[3] == 1, "split over k: not these kernels"
    assert plan[2] > 0 if tile == "mix" else (tuple(plan[:2]) == tile and plan[2] == 0), (tuple(plan), tile)


@pytest.mark.parametrize("tile,M,N,K", [(t, *s) for t, shapes in TILES.items() for s in shapes])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_many_token_tiles_are_exact_on_integers(cuda, tile, M, N, K, dtype):
    _runs_in(tile, M, N, K)
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


@pytest.mark.parametrize("tile,B,Ntok,C,K", [(t, *s) for t, shapes in GATED.items() for s in shapes])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_many_token_gated_residual_across_batch_boundaries(cuda, tile, B, Ntok, C, K, dtype):
    _runs_in(tile, B * Ntok, C, K)
    ints = lambda *s, hi=3, seed: _ints(*s, lo=-hi, hi=hi, seed=seed, dtype=dtype).to(cuda)
    a, w, bias = ints(B, Ntok, K, seed=1), ints(C, K, seed=2), ints(C, hi=9, seed=3)
    gate, res = ints(B, 1, C, hi=4, seed=4), ints(B, Ntok, C, hi=99, seed=5)
    y = (a.float() @ w.float().T + bias.float()).to(dtype)
    assert torch.equal(ops.gemm_gate_residual(a, w, bias, gate, res), res + gate * y)   # the stock pair's roundings


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_two_widths_that_the_residual_keeps_in_288_channels(cuda, dtype):
    """Within 4 % of the estimate for 288 channels: two widths without a residual, one with (boundaries of entries inside its tiles)."""
    test_many_token_tiles_are_exact_on_integers(cuda, "mix", 9233, 5192, 1056, dtype)
    test_many_token_gated_residual_across_batch_boundaries(cuda, "mix", 7, 1319, 5192, 1056, dtype)


@pytest.mark.parametrize("M,N,K", [(257, 18440, 1152), (300, 17920, 2240), (320, 18376, 1208), (290, 20480, 1064)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_two_tiles_of_160_tokens_are_exact_on_integers(cuda, M, N, K, dtype):
    """160 x 192: a prompt's tokens by many channels, with ragged tokens and channels, k tails and gate rows that change inside a tile."""
    test_many_token_tiles_are_exact_on_integers(cuda, (160, 192), M, N, K, dtype)
    if M % 2 == 0:
        test_many_token_gated_residual_across_batch_boundaries(cuda, (160, 192), 2, M // 2, N, K, dtype)


@pytest.mark.parametrize("M,N,K", [(150, 33000, 1160), (129, 32808, 1096), (97, 41480, 1096), (560, 11400, 5608), (777, 8264, 3016),
                                   (790, 9208, 3080)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_one_four_and_five_tiles_of_160_tokens_are_exact_on_integers(cuda, M, N, K, dtype):
    """160 x 192 where its other rows of tiles fill one round: the same with a single row of tiles, with four and with five."""
    assert -(-M // 160) in (1, 4, 5)
    test_two_tiles_of_160_tokens_are_exact_on_integers(cuda, M, N, K, dtype)


@pytest.mark.parametrize("M,N,K", [(300, 264, 5664), (257, 200, 4128), (700, 1160, 6432), (130, 3000, 8192), (1025, 2232, 5600)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_split_over_k_is_exact_on_integers(cuda, M, N, K, dtype):
    """Partial planes of 256 x 192 tiles: ragged rows and channels, token halves without rows, ranges of unequal length, a k tail."""
    plan = (ctypes.c_int * 4)()
    _lib.check(_lib.load().sana_hip_gemm_plan(M, N, K, plan), "sana_hip_gemm_plan")
    assert tuple(plan[:2]) == (256, 192) and plan[3] > 1
    a, w, bias = (_ints(M, K, seed=1, dtype=dtype).to(cuda), _ints(N, K, seed=2, dtype=dtype).to(cuda),
                  _ints(N, lo=-9, hi=9, seed=3, dtype=dtype).to(cuda))
    ref = a.float() @ w.float().T        # |sum| <= 9 k < 2^24: exact in any order
    assert torch.equal(ops.gemm_bf16(a, w), ref.to(dtype))
    assert torch.equal(ops.gemm_bf16(a, w, bias, "bias"), (ref + bias.float()).to(dtype))


@pytest.mark.parametrize("N", [1, 5, 64])
@pytest.mark.parametrize("K", [16, 512, 3072, 3088, 5600])
def test_expanded_weights_are_the_rounded_products(cuda, N, K):
    """Pieces of 8 values, 64 lanes, six pieces a lane: one piece, whole passes, one more piece."""
    gen = torch.Generator().manual_seed(K + N)
    wq = torch.randint(-128, 128, (N, K + 16), generator=gen).to(torch.int8).to(cuda)[:, :K]
    scale = (0.001 + torch.rand(N, generator=gen)).to(cuda)
    assert torch.equal(ops.dequant_w8(wq, scale), (wq.float() * scale[:, None]).bfloat16())


@pytest.mark.parametrize("N,K,ld", [(131069, 16, 16), (131073, 48, 64), (262150, 16, 32), (7, 520 * 16, 521 * 16), (3, 496, 496)])
def test_int8_weights_of_many_rows_and_of_rows_apart_are_expanded(cuda, N, K, ld):
    """More rows than one grid plane takes (2^17), fewer and more than 512 values a row, the last wave's lanes past it, rows apart."""
    gen = torch.Generator().manual_seed(N)
    wq = torch.randint(-127, 128, (N, ld), generator=gen, dtype=torch.int8).to(cuda)[:, :K]
    scale = (0.001 + torch.rand(N, generator=gen)).to(cuda)
    assert torch.equal(ops.dequant_w8(wq, scale), (wq.float() * scale[:, None]).bfloat16())
