"""The 256 x 288 tile kernel of the 16-bit GEMM at the edges of its tiles: integer operands (every product, sum and bias is
exact in fp32, so the result is bit for bit the rounded integer matrix product), ragged rows and channels, k tails, one and
several tiles per workgroup, gate rows that change inside a tile, and the temporal convolution against narrower tiles."""
import ctypes

import pytest
import torch

from sana_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _ints(*shape, lo=-3, hi=3, seed=0, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(lo, hi + 1, shape, generator=g).to(dtype)


def _plan(M, N, K):
    plan = (ctypes.c_int * 4)()
    _lib.check(_lib.load().sana_hip_gemm_plan(M, N, K, plan), "sana_hip_gemm_plan")
    return tuple(plan)


def _runs_in_288(M, N, K):
    assert _plan(M, N, K) == (256, 288, 0, 1)


# k tails of 8, 56 and 0 in an odd and an even number of k-tiles; ragged rows; ragged channels in the first and the second
# wave column and one whole tile; the last two have more tiles than workgroups
@pytest.mark.parametrize("M,N,K", [(1413, 11016, 200), (3287, 5016, 248), (5257, 3400, 256), (4325, 4208, 320),
                                   (2907, 5528, 488), (8471, 4256, 200), (14040, 2592, 248)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_288_wide_tile_is_exact_on_integers(cuda, M, N, K, dtype):
    _runs_in_288(M, N, K)
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


# the last two have more tiles than workgroups, with one batch entry and with boundaries inside tiles
@pytest.mark.parametrize("B,Ntok,C,K", [(3, 1096, 5016, 248), (7, 202, 11016, 200), (5, 1052, 3400, 256), (1, 8471, 4256, 200),
                                        (3, 2824, 4256, 200)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_288_wide_gated_residual_across_batch_boundaries(cuda, B, Ntok, C, K, dtype):
    _runs_in_288(B * Ntok, C, K)
    ints = lambda *s, hi=3, seed: _ints(*s, lo=-hi, hi=hi, seed=seed, dtype=dtype).to(cuda)
    a, w, bias = ints(B, Ntok, K, seed=1), ints(C, K, seed=2), ints(C, hi=9, seed=3)
    gate, res = ints(B, 1, C, hi=4, seed=4), ints(B, Ntok, C, hi=99, seed=5)
    y = (a.float() @ w.float().T + bias.float()).to(dtype)
    assert torch.equal(ops.gemm_gate_residual(a, w, bias, gate, res), res + gate * y)   # the stock pair's roundings
    y = (a.float() @ w.float().T).to(dtype)
    assert torch.equal(ops.gemm_gate_residual(a, w, None, gate, res), res + gate * y)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("off", [1, 2, 4, 7])
def test_bias_at_any_alignment(cuda, off, dtype):
    """A bias that is a slice at an odd place gives what its aligned copy does (other tiles, the same sums)."""
    M, N, K = 8471, 4256, 200
    _runs_in_288(M, N, K)
    a, w, stored = (_ints(M, K, seed=1, dtype=dtype).to(cuda), _ints(N, K, seed=2, dtype=dtype).to(cuda),
                    _ints(N + 8, lo=-9, hi=9, seed=3, dtype=dtype).to(cuda))
    bias = stored[off:off + N]
    y = (a.float() @ w.float().T + bias.float()).to(dtype)
    assert torch.equal(ops.gemm_bf16(a, w, bias, "bias"), y)
    gate, res = _ints(1, 1, N, seed=4, dtype=dtype).to(cuda), _ints(1, M, N, hi=99, lo=-99, seed=5, dtype=dtype).to(cuda)
    assert torch.equal(ops.gemm_gate_residual(a[None], w, bias, gate, res), res + gate * y)


@pytest.mark.parametrize("ldw", [(1 << 21) - 8, 1 << 21])
def test_weight_rows_around_the_limit_of_its_offsets(cuda, ldw):
    M, N, K = 14040, 2592, 248
    _runs_in_288(M, N, K)
    w = torch.empty((N - 1) * ldw + K, dtype=torch.bfloat16, device=cuda).as_strided((N, K), (ldw, 1))
    dense = _ints(N, K, seed=2).to(cuda)
    w.copy_(dense)
    a = _ints(M, K, seed=1).to(cuda)
    assert torch.equal(ops.gemm_bf16(a, w), (a.float() @ dense.float().T).bfloat16())


# 248 and 256 tiles, one a workgroup; 1024, 1024 and 512: workgroups with several, frames (and flagged ones) inside a tile
@pytest.mark.parametrize("T,P,C,ends", [(5, 1560, 2240, [1, 3]), (6, 2700, 1152, []), (21, 1560, 2240, [4, 9, 17]),
                                        (21, 1560, 2240, []), (21, 1560, 1152, [0, 6])])
def test_288_wide_temporal_convolution_equals_one_launch_per_frame(cuda, T, P, C, ends):
    """The whole clip in 288-wide tiles, each frame by itself in narrower ones: the same products in the same order, so the
    same bits."""
    _runs_in_288(T * P, C, 3 * C)
    assert _plan(P, C, 3 * C)[:2] != (256, 288)
    g = torch.Generator().manual_seed(C + T)
    y = torch.randn((T + 1) * P, C, generator=g).bfloat16().to(cuda)          # a real frame in front (a cache's last one)
    w2 = (torch.randn(C, 3 * C, generator=g) * (1.0 / (3 * C)) ** 0.5).bfloat16().to(cuda)
    one = ops.tconv_residual(y, w2, T * P, P, zero_last_tap=ops.frame_flags(T, ends, cuda))
    for f in range(T):      # rows behind the last frame, or behind a flagged one, read as zeros
        frame = ops.tconv_residual(y[f * P:(f + (2 if f in ends else 3)) * P], w2, P, P)
        assert torch.equal(one[f * P:(f + 1) * P], frame), f
