"""Both phases of the linear attention in one kernel (short sequences): against the fp64 oracle, at the edges of its tiles
(16-token steps, 32-token tiles, the two calls' splits of 48 to 256 tokens, 256 heads, 1024 tokens) and just beyond them, and
bit for bit what the two calls give."""
import pytest
import torch

from oracle import sana_oracle as O
from sana_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return ((a.double() - b).norm() / b.norm()).item()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,N,C", [(1, 1, 64), (2, 15, 32), (1, 17, 96), (3, 33, 160), (1, 255, 1152), (1, 256, 1152),
                                   (2, 513, 64), (1, 972, 2240), (2, 1024, 1152), (3, 1023, 2240),
                                   (1, 1025, 96), (8, 100, 1056), (1, 65, 1152), (1, 128, 64), (2, 129, 1152), (1, 144, 2240),
                                   (1, 385, 2240), (1, 769, 1152), (256, 1024, 32), (85, 700, 96),
                                   (1, 257, 5088), (5, 257, 1024), (2, 1000, 2560)])
def test_matches_the_oracle_and_the_two_calls(cuda, B, N, C, dtype):
    eps = 1e-8
    gen = torch.Generator().manual_seed(N + C)
    wide = torch.randn(B, N, 3 * C + 32, generator=gen).to(dtype)      # rows with something between them
    q, k, v = (wide[:, :, i * C:(i + 1) * C] for i in range(3))
    heads = [t.double().reshape(B, N, C // 32, 32).permute(0, 2, 3, 1) for t in (q, k, v)]
    ref = O.relu_linear_attention(heads[0], heads[1].transpose(-1, -2), heads[2], eps).permute(0, 3, 1, 2).reshape(B, N, C)
    d = wide.to(cuda)
    q, k, v = (d[:, :, i * C:(i + 1) * C] for i in range(3))
    got = ops.relu_linear_attention(q, k, v, eps).cpu()
    two = ops.linattn_apply(q, ops.linattn_state(k, v), eps).cpu()
    assert bool(torch.isfinite(got).all())
    # fp32: a sum of N products, rounded at 6e-8 each in random directions; 16 bits: one rounding of the result (2^-9, 2^-12)
    bound = {torch.float32: 1e-6, torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}[dtype]
    assert _rel(got, ref) <= bound
    assert torch.equal(got, two)
    one = _lib.load().sana_hip_linattn_scratch_bytes(B, N, C // 32, 32, ops._dt(q)) == 0
    assert one == (N <= 1024 and B * C // 32 <= 256 and (dtype != torch.float32 or N <= 256 or B * C // 32 >= 160))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_zeros_and_infinities_as_the_two_calls(cuda, dtype):
    """Tokens without a positive key or query (0 / eps), a head of zeros, and an infinity in one head."""
    gen = torch.Generator().manual_seed(3)
    qkv = torch.randn(2, 70, 3, 128, generator=gen)
    qkv[0, :, 1, :32] = -1.0
    qkv[0, 5, 0] = -2.0
    qkv[1, 9, 1, 40], qkv[1, 11, 2, 70] = float("inf"), float("-inf")
    q, k, v = (qkv.to(dtype).to(cuda)[:, :, i] for i in range(3))
    got, two = ops.relu_linear_attention(q, k, v, 1e-8), ops.linattn_apply(q, ops.linattn_state(k, v), 1e-8)
    assert torch.isnan(two).any() and torch.allclose(got, two, rtol=0, atol=0, equal_nan=True)


def test_what_it_does_not_take_goes_to_the_two_calls(cuda):
    x = torch.randn(1, 64, 3, 64, device=cuda)
    q, k, v = x[:, :, 0], x[:, :, 1], x[:, :, 2]
    assert ops._one_call(q, k, v, 32)
    assert not ops._one_call(q, k.contiguous(), v, 32)                       # k and v of different strides: refused
    assert not ops._one_call(q, k.bfloat16(), v.bfloat16(), 32)
    with pytest.raises(_lib.SanaHipError):
        ops.relu_linear_attention(q, k.contiguous(), v, 1e-8)
    out32 = ops.relu_linear_attention(q.bfloat16(), k.bfloat16(), v.bfloat16(), 1e-8, out_dtype=torch.float32)
    assert out32.dtype == torch.float32


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_graphs_captured_on_one_stream_keep_a_state_each(cuda, monkeypatch, dtype):
    """Beyond one launch the state is in memory: nothing of it in the stream's scratch buffer, which graphs of one capture
    stream would share, and two such graphs replayed on two streams give the eager results."""
    stream, graphs, wants = torch.cuda.Stream(), [], []
    monkeypatch.setattr(ops, "_workspaces", {})      # (stream handles come from a pool: not those of other tests)
    for seed in (1, 2):
        gen = torch.Generator().manual_seed(seed)
        q, k, v = (t.to(cuda) for t in torch.randn(3, 2, 1500, 1152, generator=gen).to(dtype))
        wants.append(ops.relu_linear_attention(q, k, v, 1e-8))
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out = ops.relu_linear_attention(q, k, v, 1e-8)
        graphs.append((graph, out, (q, k, v)))
    assert (q.device.index, stream.cuda_stream) not in ops._workspaces
    sides = [torch.cuda.Stream(), torch.cuda.Stream()]
    for _ in range(5):
        for _, out, _ in graphs:
            out.zero_()
        torch.cuda.synchronize()
        for side, (graph, _, _) in zip(sides, graphs):
            with torch.cuda.stream(side):
                graph.replay()
        torch.cuda.synchronize()
        for (_, out, _), want in zip(graphs, wants):
            assert torch.equal(out, want)


def test_a_large_state_is_not_kept(cuda, monkeypatch):
    gen = torch.Generator().manual_seed(1)
    q, k, v = (t.to(cuda) for t in torch.randn(3, 1, 1100, 64, generator=gen))
    want = ops.linattn_apply(q, ops.linattn_state(k, v), 1e-8)
    need = _lib.load().sana_hip_linattn_scratch_bytes(1, 1100, 2, 32, ops._dt(q))
    torch.cuda.synchronize()
    for kept in (need - 1, need):
        monkeypatch.setattr(ops, "STATE_SCRATCH_KEPT", kept)
        stream = torch.cuda.Stream()
        monkeypatch.setattr(ops, "_workspaces", {})
        with torch.cuda.stream(stream):
            got = ops.relu_linear_attention(q, k, v, 1e-8)
        stream.synchronize()
        assert torch.equal(got, want)
        assert ((q.device.index, stream.cuda_stream) in ops._workspaces) == (kept == need)


@pytest.mark.parametrize("B,N,h", [(1, 257, 5), (1, 300, 1), (2, 383, 7), (1, 384, 6), (1, 385, 9), (3, 1000, 13), (1, 1024, 3),
                                   (1, 1008, 150), (53, 511, 3)])
def test_two_launches_on_partial_states(cuda, B, N, h):
    """fp32 between 257 and 1024 tokens: the sum over the splits inside phase 2, at the edges of its 128-token ranges, 32-token waves
    and head groups, with rows and batch entries apart, is that of the reduction kernel bit for bit."""
    C = 32 * h
    gen = torch.Generator().manual_seed(N + h)
    wide = torch.randn(B, N + 3, 3 * C + 4, generator=gen).to(cuda)[:, 1:N + 1]
    q, k, v = (wide[:, :, i * C:(i + 1) * C] for i in range(3))
    assert _lib.load().sana_hip_linattn_scratch_bytes(B, N, h, 32, ops._dt(q)) > 0
    assert torch.equal(ops.relu_linear_attention(q, k, v, 1e-15), ops.linattn_apply(q, ops.linattn_state(k, v), 1e-15))


@pytest.mark.parametrize("B,N,h,two", [(1, 257, 5, True), (1, 1024, 3, True), (4, 1024, 36, True), (1, 980, 150, True), (2, 300, 140, True),
                                       (1, 1025, 3, False), (1, 1008, 150, False), (5, 1024, 54, False)])
def test_which_launches_read_the_partial_states(cuda, B, N, h, two):
    """The two launches leave the front of the scratch, where the reduced state would be, as it was; the launches of the two calls
    write it.  Up to 1024 tokens and 147456 head-tokens it is two."""
    lib, C = _lib.load(), 32 * h
    gen = torch.Generator().manual_seed(N + h)
    q, k, v = (torch.randn(B, N, C, generator=gen).to(cuda) for _ in range(3))
    need = lib.sana_hip_linattn_scratch_bytes(B, N, h, 32, _lib.DT_F32)
    state = B * h * 33 * 32
    assert need > 4 * state                                    # a state and partial states
    scratch, out = torch.full((need // 4,), 7.25, device=cuda), torch.empty(B, N, C, device=cuda)
    _lib.check(lib.sana_hip_linattn(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), scratch.data_ptr(), need, B, N, h, 32,
                                    N * C, C, N * C, C, N * C, C, 1e-15, _lib.DT_F32, torch.cuda.current_stream().cuda_stream),
               "sana_hip_linattn")
    assert bool((scratch[:state] == 7.25).all()) == two
    assert not bool((scratch[-(need // 4 - state) // 2:] == 7.25).any())
    assert torch.equal(out, ops.linattn_apply(q, ops.linattn_state(k, v), 1e-15))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("far", ["q", "k and v", "out", "all"])
def test_rows_of_any_distance(cuda, dtype, far):
    """16-bit rows 2^20 values apart and more are addressed in 64 bits: the bits of dense rows, nothing written between the rows."""
    lib, N, h, ld = _lib.load(), 37, 3, 1 << 20
    C, gen = 32 * h, torch.Generator().manual_seed(7)
    dense = torch.randn(N, 3 * C, generator=gen).to(dtype).to(cuda)
    want = ops.relu_linear_attention(*(dense[None, :, i * C:(i + 1) * C] for i in range(3)), 1e-15)[0]
    wide = torch.full((N, ld), float("nan"), dtype=dtype, device=cuda)
    wide[:, :3 * C] = dense
    src = [wide if far == "all" or name in far else dense for name in "qkv"]
    out = torch.full((N, ld if far in ("out", "all") else C), 3.0, dtype=dtype, device=cuda)
    ptr = [s.data_ptr() + 2 * C * i for i, s in enumerate(src)]
    _lib.check(lib.sana_hip_linattn(*ptr, out.data_ptr(), None, 0, 1, N, h, 32, 0, src[0].stride(0), 0, src[1].stride(0), 0,
                                    out.stride(0), 1e-15, ops._dt(out), torch.cuda.current_stream().cuda_stream), "sana_hip_linattn")
    assert torch.equal(out[:, :C], want) and bool((out[:, C:] == 3.0).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,h", [(2, 32), (1, 65), (5, 17), (2, 43), (1, 128), (3, 43)])
@pytest.mark.parametrize("N", [16, 47, 49, 385, 1009])
def test_workgroups_that_share_a_head(cuda, B, h, N, dtype):
    """16 bits: four, three, two and one workgroup a head (64, 65 .. 85, 86 .. 128 and more heads), with steps of 16 queries that run out
    within one of them: every query is answered, with the bits of the two calls."""
    C, gen = 32 * h, torch.Generator().manual_seed(N + h)
    q, k, v = (torch.randn(B, N, C, generator=gen).to(dtype).to(cuda) for _ in range(3))
    out = torch.full((B, N + 1, C), float("nan"), dtype=dtype, device=cuda)       # (a row behind each batch entry's that stays)
    _lib.check(_lib.load().sana_hip_linattn(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), None, 0, B, N, h, 32, N * C, C,
                                            N * C, C, (N + 1) * C, C, 1e-8, ops._dt(q), torch.cuda.current_stream().cuda_stream),
               "sana_hip_linattn")
    assert torch.equal(out[:, :N], ops.linattn_apply(q, ops.linattn_state(k, v), 1e-8))
    assert bool(torch.isnan(out[:, N]).all())


@pytest.mark.parametrize("N", [1, 16, 17, 33, 64, 65, 81, 97, 130])
def test_fp32_splits_of_any_length_and_row_distance(cuda, N):
    """Phase 1 in passes of 64, 32 and 16 tokens with 32-bit offsets, and on rows too far apart for those, against 64 bits and each other;
    nothing between the rows or behind them (NaN) is read."""
    h, C, gen = 3, 96, torch.Generator().manual_seed(N)
    k, v = (torch.randn(1, N, C, generator=gen).to(cuda) for _ in range(2))
    want = torch.einsum("nhi,nhj->hij", v[0].double().view(N, h, 32), k[0].double().clamp(min=0).view(N, h, 32))
    near = ops.linattn_state(k, v)
    assert _rel(near.view(h, 33, 32)[:, :32], want) < 1e-6
    assert _rel(near.view(h, 33, 32)[:, 32], k[0].double().clamp(min=0).sum(0).view(h, 32)) < 1e-6
    for ld in [4 * C] + ([1 << 23] if N <= 17 else []):
        wide = torch.full(((N + 1) * ld,), float("nan"), device=cuda)[:N * ld].view(1, N, ld)
        wide[:, :, :C], wide[:, :, C:2 * C] = k, v
        assert torch.equal(ops.linattn_state(wide[:, :, :C], wide[:, :, C:2 * C]), near)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N,h", [(1, 3), (31, 2), (33, 5), (159, 3), (290, 1)])
def test_16_bit_splits_of_any_length_and_row_distance(cuda, N, h, dtype):
    """Phase 1 in 16 bits with 32-bit offsets, and on rows too far apart for those, against 64 bits and each other; nothing between the
    rows, behind the last channel of an odd head or behind the last token (NaN) is read."""
    C, gen = 32 * h, torch.Generator().manual_seed(N + h)
    k, v = (torch.randn(1, N, C, generator=gen).to(dtype).to(cuda) for _ in range(2))
    want = torch.einsum("nhi,nhj->hij", v[0].double().view(N, h, 32), k[0].double().clamp(min=0).view(N, h, 32))
    near = ops.linattn_state(k, v)
    assert _rel(near.view(h, 33, 32)[:, :32], want) < 1e-6
    assert _rel(near.view(h, 33, 32)[:, 32], k[0].double().clamp(min=0).sum(0).view(h, 32)) < 1e-6
    for ld in [2 * C + 8] + ([1 << 24] if N <= 33 else []):
        wide = torch.full(((N + 1) * ld,), float("nan"), dtype=dtype, device=cuda)[:N * ld].view(1, N, ld)
        wide[:, :, :C], wide[:, :, C:2 * C] = k, v
        assert torch.equal(ops.linattn_state(wide[:, :, :C], wide[:, :, C:2 * C]), near)
