"""Cross-attention to the text tokens: the short-key softmax attention kernel against the fp64 formula
(reference: diffusion/model/nets/sana_blocks.py:69-98, the scaled_dot_product_attention branch with its additive
padding mask), and the module built on it against the oracle module.  Tolerance: bf16 outputs, max-abs <= 2e-2 and
rel-L2 <= 1e-2 (the probabilities are rounded to bf16 before they multiply v, as fused attention kernels do)."""
import pytest
import torch

import sana_amd as S
from sana_amd import ops
from oracle import sana_oracle as O

pytestmark = pytest.mark.gpu


def rel_l2(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm()).item()


def formula(q, kv, H, bias=None):
    """softmax(q k^T / sqrt(d) + bias) v per head in fp64, token-major in and out."""
    B, N, C = q.shape
    d = C // H
    qh = q.double().view(B, N, H, d).transpose(1, 2)
    k = kv.double()[:, :, :C].reshape(B, -1, H, d).transpose(1, 2)
    v = kv.double()[:, :, C:].reshape(B, -1, H, d).transpose(1, 2)
    s = qh @ k.transpose(-1, -2) * d ** -0.5
    if bias is not None:
        s = s + bias.double()[:, None, None, :]
    return (torch.softmax(s, -1) @ v).transpose(1, 2).reshape(B, N, C)


@pytest.mark.parametrize("B,N,Nk,H,d,masked", [(1, 16384, 300, 20, 112, False),   # the 4096 px latent, Sana-1.6B
                                              (2, 1024, 300, 20, 112, True),
                                              (3, 200, 77, 16, 72, True),        # Sana-600M heads, ragged query blocks
                                              (1, 37, 1, 2, 112, False),         # a single key: the output is v
                                              (2, 130, 320, 4, 104, True),       # the largest key set, another head_dim
                                              (1, 64, 33, 3, 80, False)])
def test_cross_attention_matches_the_formula(cuda, B, N, Nk, H, d, masked):
    g = torch.Generator().manual_seed(B * 1000 + N + Nk + d)
    C = H * d
    q = (torch.randn(B, N, C, generator=g) * 1.5).bfloat16()
    kv = torch.randn(B, Nk, 2 * C, generator=g).bfloat16()
    bias = None
    if masked:   # the reference's padding mask: the tail of every text is padding, of another length per batch entry
        keep = torch.ones(B, Nk)
        for b in range(B):
            keep[b, max(1, Nk - 7 * (b + 1)):] = 0
        bias = (1 - keep) * -10000.0
    out = ops.cross_attention(q.to(cuda), kv.to(cuda), H, None if bias is None else bias.to(cuda))
    ref = formula(q, kv, H, bias)
    mx = (out.cpu().double() - ref).abs().max().item()
    assert mx <= 2e-2 and rel_l2(out.cpu(), ref) <= 1e-2, (mx, rel_l2(out.cpu(), ref))
    if Nk == 1:
        assert torch.equal(out.cpu().view(B, N, H, d), kv[:, :1, C:].view(B, 1, H, d).expand(B, N, H, d))


def test_cross_attention_on_strided_rows_and_masked_keys_contribute_nothing(cuda):
    """q as a column slice of a wider buffer (row stride > C); what keys under the -10000 bias hold does not matter
    (as long as their scores stay small against 10000: the mask is additive, as in the reference)."""
    g = torch.Generator().manual_seed(5)
    B, N, Nk, H, d = 2, 300, 40, 2, 112
    C = H * d
    wide = torch.randn(B, N, C + 64, generator=g).bfloat16().to(cuda)
    kv = torch.randn(B, Nk, 2 * C, generator=g).bfloat16()
    keep = torch.ones(B, Nk)
    keep[:, 25:] = 0
    bias = ((1 - keep) * -10000.0).to(cuda)
    a = ops.cross_attention(wide[:, :, :C], kv.to(cuda), H, bias)
    kv2 = kv.clone()
    kv2[:, 25:] = 3.0
    b = ops.cross_attention(wide[:, :, :C], kv2.to(cuda), H, bias)
    assert torch.equal(a, b)
    ref = formula(wide[:, :, :C].cpu(), kv, H, bias.cpu())
    assert (a.cpu().double() - ref).abs().max().item() <= 2e-2


def test_cross_attention_rejects_what_it_cannot_hold(cuda):
    q = torch.zeros(1, 16, 256, dtype=torch.bfloat16, device=cuda)
    with pytest.raises(S.SanaHipError):
        ops.cross_attention(q, torch.zeros(1, 321, 512, dtype=torch.bfloat16, device=cuda), 2)     # 128-wide heads, 321 keys
    with pytest.raises(S.SanaHipError):
        ops.cross_attention(q, torch.zeros(1, 10, 512, dtype=torch.bfloat16, device=cuda), 8)      # head_dim 32
    with pytest.raises(S.SanaHipError):
        ops.cross_attention(q.float(), torch.zeros(1, 10, 512, device=cuda), 2)


@pytest.mark.parametrize("C,H,B,N,Nk,masked", [(2240, 20, 1, 1024, 300, False), (1152, 16, 2, 256, 120, True)])
def test_cross_attention_module_matches_oracle(cuda, C, H, B, N, Nk, masked):
    g = torch.Generator().manual_seed(C + N)
    om = O.MultiHeadCrossAttention(C, H)
    with torch.no_grad():
        for p in om.parameters():
            p.copy_(torch.nn.init.trunc_normal_(torch.empty(p.shape), std=0.02, generator=g))
    om = om.bfloat16()
    hm = S.modules.MultiHeadCrossAttention(C, H).bfloat16()
    hm.load_state_dict(om.state_dict())
    hm = hm.to(cuda)
    x = torch.randn(B, N, C, generator=g).bfloat16()
    y = torch.randn(B, Nk, C, generator=g).bfloat16()
    mask = None
    if masked:
        mask = torch.ones(B, Nk, dtype=torch.int64)
        mask[0, Nk // 2:] = 0
    with torch.no_grad():
        out = hm(x.to(cuda), y.to(cuda), None if mask is None else mask.to(cuda))
        ref = om.float()(x.float(), y.float(), mask)
    mx = (out.cpu().double() - ref.double()).abs().max().item()
    assert mx <= 2e-2 and rel_l2(out.cpu(), ref) <= 1e-2, (mx, rel_l2(out.cpu(), ref))


def test_residual_add_inside_the_projection_gemm(cuda):
    """x + cross_attn(x, y): the add is the projection GEMM's epilogue at every row count (two roundings, as the stock
    linear + add); against the oracle module's output plus x, and against the unfused composition of this module (same
    products, another fp32 summation order inside the two GEMMs: at most one bf16 ulp of the sum apart)."""
    C, H, B, N, Nk = 2240, 20, 2, 2048, 300
    g = torch.Generator().manual_seed(3)
    om = O.MultiHeadCrossAttention(C, H)
    with torch.no_grad():
        for p in om.parameters():
            p.copy_(torch.nn.init.trunc_normal_(torch.empty(p.shape), std=0.02, generator=g))
    om = om.bfloat16()
    hm = S.modules.MultiHeadCrossAttention(C, H).bfloat16()
    hm.load_state_dict(om.state_dict())
    hm = hm.to(cuda)
    assert B * N >= hm.RESIDUAL_GEMM_MIN_ROWS
    x = torch.randn(B, N, C, generator=g).bfloat16()
    y = torch.randn(B, Nk, C, generator=g).bfloat16()
    with torch.no_grad():
        fused = hm.forward_residual(x.to(cuda), y.to(cuda))
        plain = x.to(cuda) + hm(x.to(cuda), y.to(cuda))
        ref = x.float() + om.float()(x.float(), y.float())
    assert (fused.float() - plain.float()).abs().max().item() <= 2 ** -7 * plain.float().abs().max().item()
    mx = (fused.cpu().double() - ref.double()).abs()
    assert (mx > 2e-2 + 2.0 ** -7 * ref.double().abs()).sum().item() == 0 and rel_l2(fused.cpu(), ref) <= 1e-2
    small = hm.forward_residual(x[:, :64].to(cuda), y.to(cuda))       # few rows: the same tile kernel either way
    assert torch.equal(small, x[:, :64].to(cuda) + hm(x[:, :64].to(cuda), y.to(cuda)))


@pytest.mark.parametrize("B,N,Nk,H,d,masked", [(2, 1024, 300, 16, 72, True), (1, 37, 1, 2, 112, False),
                                              (3, 130, 159, 4, 112, True), (1, 129, 161, 3, 96, False),
                                              (2, 17, 320, 2, 104, True)])
def test_cross_attention_fp16_matches_the_formula(cuda, B, N, Nk, H, d, masked):
    """The same kernel on f16 operands, around the two key-tile counts (160 keys) and the padded head dims.  Probabilities
    and outputs carry a relative 2^-11 each, the probabilities' errors average over the keys: 2e-3 in norm."""
    g = torch.Generator().manual_seed(B * 1000 + N + Nk + d)
    C = H * d
    q = (torch.randn(B, N, C, generator=g) * 1.5).half()
    kv = torch.randn(B, Nk, 2 * C, generator=g).half()
    keep = torch.ones(B, Nk)
    if masked:
        for b in range(B):
            keep[b, max(1, Nk - 7 * (b + 1)):] = 0
    bias = (1 - keep) * -10000.0
    out = ops.cross_attention16(q.to(cuda), kv.to(cuda), H, bias.to(cuda) if masked else None)
    ref = formula(q, kv, H, bias if masked else None)
    assert out.dtype == torch.float16
    assert (out.cpu().double() - ref).abs().max().item() <= 5e-3 and rel_l2(out.cpu(), ref) <= 2e-3


@pytest.mark.parametrize("C,H,B,N,Nk,dtype", [(1152, 16, 2, 100, 300, torch.float16), (2240, 20, 1, 7, 40, torch.bfloat16),
                                             (1152, 16, 1, 1000, 77, torch.bfloat16)])
def test_residual_projection_of_few_rows(cuda, C, H, B, N, Nk, dtype):
    """x + cross_attn(x, y) on this library's GEMMs at row counts below a tile and above, against the oracle in fp32; an x
    at an odd address takes the stock linears and gives the same up to the sums' order."""
    g = torch.Generator().manual_seed(N)
    om = O.MultiHeadCrossAttention(C, H)
    with torch.no_grad():
        for p in om.parameters():
            p.copy_(torch.nn.init.trunc_normal_(torch.empty(p.shape), std=0.02, generator=g))
    om = om.to(dtype)
    hm = S.modules.MultiHeadCrossAttention(C, H).to(dtype)
    hm.load_state_dict(om.state_dict())
    hm = hm.to(cuda)
    x, y = torch.randn(B, N, C, generator=g).to(dtype), torch.randn(B, Nk, C, generator=g).to(dtype)
    with torch.no_grad():
        out = hm.forward_residual(x.to(cuda), y.to(cuda))
        odd = torch.empty(x.numel() + 1, dtype=dtype, device=cuda)[1:].view(x.shape).copy_(x)
        assert odd.data_ptr() % 16
        stock = hm._linear(hm.q_linear, odd)
        ref = x.float() + om.float()(x.float(), y.float())
    tol = 1e-2 if dtype == torch.bfloat16 else 2e-3
    assert rel_l2(out.cpu(), ref) <= tol
    assert rel_l2(stock.cpu(), torch.nn.functional.linear(x.float(), om.q_linear.weight, om.q_linear.bias)) <= tol


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_hooks_and_patches_on_the_cross_attention_of_a_block_run(cuda, dtype):
    """A hook on, or another forward put over, a block's cross-attention is called at few rows too; a fp16 model's replaced
    or hooked linears are called, not read past."""
    C, H = 288, 4
    torch.manual_seed(0)
    b = S.SanaMSBlock(C, H, mlp_ratio=2.5, attn_type="linear", ffn_type="glumbconv").to(dtype).to(cuda).eval()
    x, y = torch.randn(1, 64, C, dtype=dtype, device=cuda), torch.randn(1, 20, C, dtype=dtype, device=cuda)
    t = torch.randn(1, 6 * C, dtype=dtype, device=cuda)
    ca = b.cross_attn
    with torch.no_grad():
        ref, seen = b(x, y, t, None, (8, 8)), []
        handle = ca.register_forward_hook(lambda m, i, o: seen.append(1))
        b(x, y, t, None, (8, 8))
        handle.remove()
        assert seen == [1]
        ca.forward = lambda x, *a, **k: torch.zeros_like(x)
        patched = b(x, y, t, None, (8, 8))
        del ca.forward
        assert not torch.equal(patched, ref) and torch.equal(b(x, y, t, None, (8, 8)), ref)
        if dtype == torch.float16:
            class Doubled(torch.nn.Linear):
                def forward(self, x):
                    return 2 * super().forward(x)

            for name in ("q_linear", "kv_linear", "proj"):
                own = getattr(ca, name)
                new = Doubled(own.in_features, own.out_features).to(dtype).to(cuda)
                new.load_state_dict(own.state_dict())
                setattr(ca, name, new)
                assert not torch.equal(b(x, y, t, None, (8, 8), **S.StepConditioning([b])(y, t)[0]), ref), name
                setattr(ca, name, own)
            assert torch.equal(b(x, y, t, None, (8, 8)), ref)


@pytest.mark.parametrize("Nk,lo,hi", [(1, 0, 1), (95, 0, 95), (96, 0, 96), (97, 0, 97), (97, 96, 97), (160, 96, 160), (160, 0, 96),
                                      (161, 160, 161), (300, 0, 160), (300, 160, 300), (320, 0, 320), (320, 159, 161)])
def test_cross_attention_fp16_groups_of_keys(cuda, Nk, lo, hi):
    """f16 keeps a maximum per group of keys (96 + 64 of up to 160, 160 + 160 of up to 320): groups without a key, groups that
    are masked throughout (only keys lo .. hi - 1 count) and both at work.  Probabilities and outputs are rounded to f16 once
    each, 2^-11 / sqrt(3) of their norm at most: 4e-4 together."""
    g = torch.Generator(device="cuda").manual_seed(Nk + lo)
    B, N, H, d = 2, 70, 4, 72
    q = torch.randn(B, N, H * d, device=cuda, generator=g).half()
    kv = torch.randn(B, Nk, 2 * H * d, device=cuda, generator=g).half()
    bias = torch.full((B, Nk), -10000.0, device=cuda)
    bias[:, lo:hi] = 0
    heads = lambda t: t.double().view(B, -1, H, d).transpose(1, 2)
    k, v = heads(kv[:, :, :H * d].contiguous()), heads(kv[:, :, H * d:].contiguous())
    p = (torch.matmul(heads(q), k.transpose(-1, -2).contiguous()) * d ** -0.5 + bias[:, None, None].double()).softmax(-1)
    ref = torch.matmul(p, v.contiguous()).transpose(1, 2).reshape(B, N, H * d)
    assert rel_l2(ops.cross_attention16(q, kv, H, bias), ref) <= 4e-4


def test_cross_attention_fp16_is_as_exact_as_the_stock_kernel(cuda):
    """Against 64 bits at 300 keys: no further off than the stock fused attention that it stands for (with one maximum for all
    keys it was 2.5 % further; a ratio over 2.4 M values varies by about 0.2 %)."""
    g = torch.Generator(device="cuda").manual_seed(1)
    B, N, Nk, H, d = 2, 1024, 300, 16, 72
    q = torch.randn(B, N, H * d, device=cuda, generator=g).half()
    kv = torch.randn(B, Nk, 2 * H * d, device=cuda, generator=g).half()
    heads = lambda t: t.contiguous().view(B, -1, H, d).transpose(1, 2)
    qh, k, v = heads(q), heads(kv[:, :, :H * d]), heads(kv[:, :, H * d:])
    flat = lambda t: t.transpose(1, 2).reshape(B, N, H * d)
    p = (torch.matmul(qh.double(), k.double().transpose(-1, -2).contiguous()) * d ** -0.5).softmax(-1)
    ref = flat(torch.matmul(p, v.double().contiguous()))
    stock = flat(torch.nn.functional.scaled_dot_product_attention(qh, k, v))
    assert rel_l2(ops.cross_attention16(q, kv, H), ref) <= 1.012 * rel_l2(stock, ref)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_residual_projection_first_called_inside_a_capture(cuda, dtype):
    """A caller's own graph captures the call before anything ran eagerly, and is not replayed yet: eager calls must not
    meet memory that only a replay fills, and replays (eager work between them) give the eager bits."""
    C, H = (352 if dtype == torch.bfloat16 else 416), 4      # widths of no other test: nothing is kept for them yet
    torch.manual_seed(1)
    ca = S.modules.MultiHeadCrossAttention(C, H).to(dtype).to(cuda)
    x, y = torch.randn(2, 24, C, dtype=dtype, device=cuda), torch.randn(2, 12, C, dtype=dtype, device=cuda)
    with torch.no_grad():
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            captured = ca.forward_residual(x, y)
        eager = ca.forward_residual(x, y)
        plain = x + ca(x, y)
        # the same products and roundings; the two GEMM calls may sum in another order
        assert (eager.float() - plain.float()).abs().max().item() <= 2 ** -7 * plain.float().abs().max().item()
        for _ in range(3):
            captured.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(captured, eager) and torch.equal(ca.forward_residual(x, y), eager)


def test_fp16_cross_attention_stays_visible_to_who_watches_its_ops(cuda):
    """vmap, torch.jit.trace and autocast to another dtype see stock ops (a call into the library is invisible to them: vmap
    raised, a trace recorded an unfilled buffer, autocast lost its dtype), and a kv in other rows than the kernel reads or a
    mask in other strides is taken as before."""
    C, H = 288, 4
    torch.manual_seed(2)
    ca = S.modules.MultiHeadCrossAttention(C, H).half().to(cuda)
    xs, y = torch.randn(3, 2, 16, C, dtype=torch.half, device=cuda), torch.randn(2, 12, C, dtype=torch.half, device=cuda)
    with torch.no_grad():
        refs = torch.stack([ca(x, y) for x in xs])
        assert rel_l2(torch.vmap(lambda x: ca(x, y))(xs), refs) <= 2e-3
        traced = torch.jit.trace(ca, (xs[0], y), check_trace=False)
        assert rel_l2(traced(xs[1], y), refs[1]) <= 2e-3
        with torch.autocast("cuda", torch.bfloat16):
            assert ca(xs[0], y).dtype == torch.bfloat16
        with torch.autocast("cuda", torch.float16):
            assert torch.equal(ca(xs[0], y), refs[0])
        kv = torch.nn.functional.linear(y, ca.kv_linear.weight, ca.kv_linear.bias)
        wide = torch.cat([kv, kv], 1)[:, :12]         # batch entries not back to back
        assert rel_l2(ca(xs[0], y, None, wide), refs[0]) <= 2e-3
        mask = torch.ones(12, 2, device=cuda).t()
        mask[1, 7:] = 0
        assert mask.stride() == (1, 2)
        assert torch.equal(ca(xs[0], y, mask), ca(xs[0], y, mask.contiguous()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_tensor_subclass_weights_of_the_cross_attention_are_dispatched(cuda, dtype):
    """A weight that is a tensor subclass (as quantisation libraries put in) sees its linear, alone and in a block."""
    C, H = 288, 4
    torch.manual_seed(3)
    b = S.SanaMSBlock(C, H, mlp_ratio=2.5, attn_type="linear", ffn_type="glumbconv").to(dtype).to(cuda).eval()
    x, y = torch.randn(1, 64, C, dtype=dtype, device=cuda), torch.randn(1, 20, C, dtype=dtype, device=cuda)
    t = torch.randn(1, 6 * C, dtype=dtype, device=cuda)
    seen = []

    class Doubled(torch.Tensor):
        """Stands for twice its memory."""
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            if func is torch.nn.functional.linear:
                seen.append(1)
                with torch._C.DisableTorchFunctionSubclass():
                    return torch.nn.functional.linear(args[0], 2 * args[1].as_subclass(torch.Tensor), args[2])
            return super().__torch_function__(func, types, args, kwargs or {})

    with torch.no_grad():
        ref = b(x, y, t, None, (8, 8))
        for name in ("q_linear", "kv_linear", "proj"):
            lin = getattr(b.cross_attn, name)
            own = lin.weight
            half = (own.detach() / 2).as_subclass(Doubled)
            lin.weight = torch.nn.Parameter(half, requires_grad=False)
            for f in (lambda: b(x, y, t, None, (8, 8)), lambda: x + b.cross_attn(x, y)):
                seen.clear()
                out = f()
                assert seen, name
            lin.weight = own
            assert rel_l2(out, x + b.cross_attn(x, y)) <= (1e-2 if dtype == torch.bfloat16 else 2e-3), name
        assert torch.equal(b(x, y, t, None, (8, 8)), ref)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Nk", [1, 160, 161, 320])
def test_few_queries_in_workgroups_of_four_waves_give_the_bits_of_eight(cuda, Nk, dtype):
    """16 heads of 72: up to 1024 queries are at most 256 blocks of 64, four waves each; a query's result is its own, so it is that
    of the call with more queries around it (eight waves)."""
    H, d = 16, 72
    g = torch.Generator().manual_seed(Nk)
    q = (torch.randn(1, 1025, H * d, generator=g) * 1.5).to(dtype)
    kv = torch.randn(1, Nk, 2 * H * d, generator=g).to(dtype)
    many = ops.cross_attention16(q.to(cuda), kv.to(cuda), H)
    assert rel_l2(many.cpu(), formula(q, kv, H)) <= 1e-2
    for N in (1, 63, 64, 65, 130, 1024):
        assert torch.equal(ops.cross_attention16(q[0, :N].clone()[None].to(cuda), kv.to(cuda), H), many[:, :N]), N


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N,Nk", [(64, 300), (65, 128), (256, 129), (200, 257)])
def test_few_queries_of_several_batch_entries(cuda, N, Nk, dtype):
    """Four entries of 16 heads: four waves a workgroup, or eight where each head's keys would be staged twice; either way the bits
    of the entries one by one."""
    H, d = 16, 72
    g = torch.Generator().manual_seed(N + Nk)
    q, kv = (torch.randn(4, n, c * H * d, generator=g).to(dtype).to(cuda) for n, c in ((N, 1), (Nk, 2)))
    out = ops.cross_attention16(q, kv, H)
    assert rel_l2(out.cpu(), formula(q.cpu(), kv.cpu(), H)) <= 1e-2
    for b in range(4):
        assert torch.equal(out[b:b + 1], ops.cross_attention16(q[b:b + 1].clone(), kv[b:b + 1].clone(), H)), b


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,d", [(2, 72), (3, 80), (2, 88), (1, 104), (2, 112)])
@pytest.mark.parametrize("Nk", [1, 31, 160, 161, 319])
def test_keys_of_any_distance_give_the_bits_of_dense_ones(cuda, dtype, H, d, Nk):
    """Rows of K and V that are 32-bit offsets apart go to LDS by direct loads, others through registers; neither reads what stands
    between the rows (NaN here)."""
    gen = torch.Generator(device=cuda).manual_seed(Nk)
    C = H * d
    q = torch.randn(1, 70, C, generator=gen, device=cuda).to(dtype)
    kv = torch.randn(1, Nk, 2 * C, generator=gen, device=cuda).to(dtype)
    dense = ops.cross_attention16(q, kv, H)
    assert (dense.double() - formula(q, kv, H)).norm() <= 1e-2 * dense.double().norm()
    for ld in [2 * C + 8] + ([1 << 21] if Nk <= 31 else []):
        rows = torch.full((Nk * ld,), float("nan"), dtype=dtype, device=cuda).view(1, Nk, ld)
        rows[:, :, :2 * C] = kv
        assert torch.equal(ops.cross_attention16(q, rows[:, :, :2 * C], H), dense)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,N,H,d", [(9, 130, 20, 112), (5, 1000, 16, 72), (3, 1, 150, 96), (2, 2300, 17, 104)])
@pytest.mark.parametrize("Nk", [33, 230])
def test_workgroups_of_several_heads(cuda, B, N, H, d, Nk, dtype):
    """Workgroups whose items run over query blocks, heads and batch entries, with waves that have no query in a head's last block and
    biases of each batch entry's own: queries requested an item ahead and K and V of the next head give the bits of one entry at a time."""
    g = torch.Generator().manual_seed(N + d + Nk)
    q, kv = (torch.randn(B, n, c * H * d, generator=g).to(dtype).to(cuda) for n, c in ((N, 1), (Nk, 2)))
    bias = torch.where(torch.rand(B, Nk, generator=g) < 0.3, -10000.0, 0.0).to(cuda)
    got = ops.cross_attention16(q, kv, H, bias)
    for b in range(B):
        assert torch.equal(got[b], ops.cross_attention16(q[b:b + 1], kv[b:b + 1], H, bias[b:b + 1])[0])
    ref = formula(q[-1:].cpu(), kv[-1:].cpu(), H, bias[-1:].cpu())
    assert rel_l2(got[-1:].cpu(), ref) <= 1e-2


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,N,H,d,Nk,masked", [(1, 70, 2, 112, 161, False), (1, 70, 2, 72, 161, True), (3, 600, 20, 112, 31, True),
                                               (3, 600, 20, 72, 31, False), (2, 1100, 15, 88, 165, True)])
def test_far_keys_of_many_heads(cuda, dtype, B, N, H, d, Nk, masked):
    """Rows of K and V too far apart for 32-bit offsets: both numbers of key tiles, biases, and workgroups of two items that stage the
    keys of a second head or batch entry over the first ones (from 257 items on): the bits of dense rows."""
    assert Nk > 160 or B * H * (-(-N // 128)) > 256
    gen = torch.Generator(device=cuda).manual_seed(Nk + d)
    C, ld = H * d, 1 << 21
    q = torch.randn(B, N, C, generator=gen, device=cuda).to(dtype)
    kv = torch.randn(B, Nk, 2 * C, generator=gen, device=cuda).to(dtype)
    bias = torch.where(torch.rand(B, Nk, generator=gen, device=cuda) < 0.3, -10000.0, 0.0) if masked else None
    rows = torch.full((B * Nk * ld,), float("nan"), dtype=dtype, device=cuda).view(B, Nk, ld)
    rows[:, :, :2 * C] = kv
    dense = ops.cross_attention16(q, kv, H, bias)
    assert bool(torch.isfinite(dense).all())
    assert torch.equal(ops.cross_attention16(q, rows[:, :, :2 * C], H, bias), dense)
