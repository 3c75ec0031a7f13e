"""CPU checks of the boundary: the library loads and exports every symbol the
header declares, argument validation works without touching a GPU."""
import ctypes
import os
import re

import pytest

from sana_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "sana_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(sana_hip_\w+)\s*\(", text)))


def test_library_is_built():
    assert os.path.exists(_lib.LIB_PATH), "run `python -m sana_amd.build` first"


def test_exports_every_declared_symbol():
    lib = ctypes.CDLL(_lib.LIB_PATH)
    declared = _declared_symbols()
    assert len(declared) >= 9
    for name in declared:
        assert hasattr(lib, name), f"{name} declared in include/sana_hip.h but not exported"
    assert sorted(_lib.SIGNATURES) == declared, "python signature table out of sync with the header"


def test_version_and_strerror():
    lib = _lib.load()
    assert lib.sana_hip_abi_version() == 8
    assert b"aligned" in lib.sana_hip_strerror(-3)
    assert b"unknown" in lib.sana_hip_strerror(-99)


def test_argument_validation_needs_no_gpu():
    lib = _lib.load()
    # null pointers / bad sizes are rejected before any launch
    assert lib.sana_hip_linattn_state(None, None, None, None, 0, 1, 16, 1, 32, 0, 32, None, 1, 16, 0, 1, None) == -1
    assert lib.sana_hip_linattn_state(16, 16, 16, None, 0, 1, 16, 1, 64, 0, 64, None, 1, 16, 0, 1, None) == -2  # d != 32
    assert lib.sana_hip_linattn_state(16, 16, 16, None, 0, 1, 16, 1, 32, 0, 32, None, 1, 16, 0, 7, None) == -6  # dtype
    assert lib.sana_hip_linattn_state(16, 18, 16, None, 0, 1, 16, 1, 32, 0, 32, None, 1, 16, 0, 1, None) == -3  # align
    assert lib.sana_hip_linattn_apply(16, 16, 16, 1, 16, 1, 32, 0, 32, 0, 32, None, 1, 16, 1e-8, 1, 2, None) == -6
    # head_dim 112: bf16 only (f16 for phase 1), needs its workspace, 32-bit byte offsets inside a batch entry
    F32, BF16, F16 = 0, 1, 2
    assert lib.sana_hip_linattn_state(16, 16, 16, 16, 1 << 30, 1, 16, 1, 112, 0, 112, None, 1, 16, 0, F32, None) == -6
    assert lib.sana_hip_linattn_state(16, 16, 16, None, 0, 1, 16, 1, 112, 0, 112, None, 1, 16, 0, BF16, None) == -4
    assert lib.sana_hip_linattn_state(16, 16, 16, 16, 1 << 30, 1, 1 << 20, 1, 112, 0, 1 << 12, None, 1, 1 << 20, 0,
                                      BF16, None) == -2
    assert lib.sana_hip_linattn_state(16, 16, 16, 16, 1 << 30, 1, 16, 1, 112, 0, 96, None, 1, 16, 0, BF16, None) == -1
    assert lib.sana_hip_linattn_apply(16, 16, 16, 1, 16, 1, 112, 0, 112, 0, 112, None, 1, 16, 1e-8, F16, F16, None) == -6
    assert lib.sana_hip_dwconv3x3_silu_gate(16, 16, None, 16, 1, 4, 4, 3, 1, 1, None) == -2  # odd Ch
    assert lib.sana_hip_gemm_bf16(16, 16, None, 16, 8, 8, 20, 24, 24, 8, 0, None, 0, None) == -2      # K % 8
    assert lib.sana_hip_gemm_bf16(16, 16, None, 16, 8, 8, 32, 32, 32, 8, 1, None, 0, None) == -1      # bias epilogue, no bias
    assert lib.sana_hip_gemm_w8a16(16, 16, None, None, 16, 8, 8, 32, 32, 32, 8, 0, None, 0, None) == -1  # no scale
    # temporal conv: C % 64, odd taps, the centre tap must exist for every output row
    assert lib.sana_hip_tconv_residual(16, 16, 32, 64, 96, 3, 16, 80, None, 96, 288, 96, None) == -2
    assert lib.sana_hip_tconv_residual(16, 16, 32, 64, 64, 2, 16, 80, None, 64, 128, 64, None) == -1
    assert lib.sana_hip_tconv_residual(16, 16, 32, 64, 64, 3, 16, 64, None, 64, 192, 64, None) == -1
    assert lib.sana_hip_tconv_residual(16, 16, 32, 64, 64, 3, 16, 80, None, 64, 128, 64, None) == -1   # ldw < taps * C
    assert lib.sana_hip_tconv_residual(16, 16, 32, 64, 64, 1, 16, 80, 16, 64, 64, 64, None) == -1   # chunk flags need >= 3 taps
    assert lib.sana_hip_tconv_residual(16, 16, 32, 64, 64, 3, 16, 80, None, 64, 192, 1 << 23, None) == -2   # 32-bit offsets


@pytest.mark.parametrize("dtype,N", [(0, 257), (0, 1024), (0, 1025), (1, 1025), (2, 4096)])
def test_one_call_attention_refuses_misaligned_scratch(dtype, N):
    """Nothing is launched on scratch that the kernels' 16-byte accesses do not fit, whichever launches the sizes select."""
    lib, h, C = _lib.load(), 5, 160
    need = lib.sana_hip_linattn_scratch_bytes(1, N, h, 32, dtype)
    assert need > 0
    call = lambda scratch, size: lib.sana_hip_linattn(16, 16, 16, 16, scratch, size, 1, N, h, 32, N * C, C, N * C, C, N * C, C,
                                                      1e-15, dtype, None)
    for off in (2, 4, 8, 12):
        assert call(4096 + off, need) == -3
    assert call(4096, need - 1) == -4 and call(None, need) == -4


def test_workspace_query():
    lib = _lib.load()
    # 1.6B @ 16384 tokens: 70 heads -> splits of the token axis need partial states
    n = lib.sana_hip_linattn_workspace_bytes(1, 70, 32, 1, 16384, 1)
    assert n > 0 and n % (33 * 32 * 4) == 0
    # short sequences are never split (a split is at least 256 tokens): no workspace
    assert lib.sana_hip_linattn_workspace_bytes(16, 70, 32, 1, 256, 1) == 0
    assert lib.sana_hip_linattn_workspace_bytes(64, 70, 32, 4, 300, 1) == 0
    # head_dim 112 always goes through records of token ranges: 20 heads at the video shape -> 256 // 20 = 12 ranges
    # of 2752 tokens (a multiple of 64) per head, one record per (range, chunk) pair that occurs, indexed range + chunk
    assert lib.sana_hip_linattn_workspace_bytes(1, 20, 112, 1, 32760, 1) == 20 * 12 * 113 * 112 * 4
    # 21 chunks of 1560 tokens: the same ranges, 12 + 21 - 1 records
    assert lib.sana_hip_linattn_workspace_bytes(1, 20, 112, 21, 1560, 1) == 20 * 32 * 113 * 112 * 4
    assert lib.sana_hip_linattn_workspace_bytes(1, 20, 64, 1, 32760, 1) == 0   # no kernel for this head dim


def test_gemm_split_k_workspace_query():
    """Shapes with few output tiles and a long K are split along K through fp32 partial planes where that is expected to
    be faster than the best unsplit tiling; the workspace is what the GEMM then uses, and nothing where it would not split."""
    lib = _lib.load()
    # one 1024 px image at Sana-1.6B: point conv 1024 x 2240 x 5600 -> 4 x 12 tiles of 256 x 192, 88 k-tiles, 5 ranges
    assert lib.sana_hip_gemm_workspace_bytes(1024, 2240, 5600) == 5 * 1024 * 2240 * 4
    # 256 tokens through it: at most 8 ranges
    assert lib.sana_hip_gemm_workspace_bytes(256, 2240, 5600) == 8 * 256 * 2240 * 4
    # not split: grids that fill the chip, wide N or short K (the partial planes would cost more than the loop saves), and
    # the shapes that the tiles for few tokens serve faster in one piece
    for M, N, K in ((16384, 2240, 5600), (16384, 11200, 2240), (1024, 11200, 2240), (1024, 6720, 2240),
                    (1024, 3456, 1152), (1024, 2240, 512), (0, 8, 64), (256, 2244, 5600), (1024, 2240, 2240),
                    (256, 2240, 2240), (1000, 1152, 2880), (2048, 2240, 5600)):
        assert lib.sana_hip_gemm_workspace_bytes(M, N, K) == 0, (M, N, K)


def test_gemm_plan_query():
    lib = _lib.load()
    plan = (ctypes.c_int * 4)()
    def of(*shape):
        assert lib.sana_hip_gemm_plan(*shape, plan) == 0
        return tuple(plan)
    assert of(256, 1152, 1152) == (64, 32, 0, 1)                   # 4 x 18 tiles of 64 x 64, two workgroups each
    assert of(512, 1152, 1152) == (64, 64, 0, 1)                   # 8 x 18
    assert of(16384, 11200, 2240) == (256, 256, 0, 1)
    assert of(4096, 6720, 2240) == (256, 256, 3840, 1)              # two widths, two launches
    assert of(1024, 2240, 5600) == (256, 192, 0, 5)                 # five ranges of k
    for M, N, K in ((1024, 2240, 5600), (256, 2240, 5600), (1024, 2240, 2240), (4096, 2240, 5600), (300, 264, 5664)):
        assert (of(M, N, K)[3] > 1) == (lib.sana_hip_gemm_workspace_bytes(M, N, K) > 0)
    assert lib.sana_hip_gemm_plan(256, 1152, 1152, None) == -1 and lib.sana_hip_gemm_plan(0, 8, 8, plan) == -1
    assert lib.sana_hip_gemm_plan(8, 12, 8, plan) == -2 and lib.sana_hip_gemm_plan(8, 8, 12, plan) == -2


@pytest.mark.parametrize("M,ranges", [(65, 8), (116, 8), (129, 8), (144, 8), (187, 8), (390, 8), (400, 8), (448, 8), (570, 7), (896, 5),
                                      (1226, 4), (1280, 4), (2305, 2), (2560, 2)])
def test_long_k_stays_split_where_a_small_tile_is_faster(M, ranges):
    """The point conv of the 2240-wide model, both kinds of weights: sums over ranges of k are closer to the 64-bit ones than one
    chain of 5600 products, and a faster tile is no reason to give that up."""
    lib, plan = _lib.load(), (ctypes.c_int * 4)()
    assert lib.sana_hip_gemm_plan(M, 2240, 5600, plan) == 0
    assert plan[3] == ranges and lib.sana_hip_gemm_workspace_bytes(M, 2240, 5600) == ranges * M * 2240 * 4
    assert lib.sana_hip_gemm_w8_expand(M, 2240, 5600) == 0


@pytest.mark.parametrize("B,N,C,hidden", [(16, 4096, 1152, 2880), (2, 16384, 2240, 5600), (1, 256, 288, 720)])
def test_block_scratch_is_no_more_than_the_calls_one_by_one_hold(B, N, C, hidden):
    """fp16 takes the block call at every size: its scratch stays within what the composition holds at its peak beside
    input and output (normalised rows, the second residual sum, hidden pairs, gated hidden values)."""
    lib = _lib.load()
    args = _lib.BlockArgs(B=B, N=N, C=C, hidden=hidden, cross_heads=C // 72, text_len=300, split_k=1, io_dtype=_lib.DT_F16)
    state = lib.sana_hip_linattn_workspace_bytes(B, C // 32, 32, 1, N, _lib.DT_F16) + B * (C // 32) * 33 * 32 * 4
    most = 2 * B * N * (2 * C + 3 * hidden) + state + 4096
    need = lib.sana_hip_block_scratch_bytes(ctypes.byref(args))
    assert 2 * B * N * (C + 3 * C + 2 * hidden) <= need <= most


def test_ops_refuse_cpu_tensors():
    import torch
    from sana_amd import ops
    x = torch.zeros(1, 32, 32)
    with pytest.raises(_lib.SanaHipError):
        ops.linattn_state(x, x)


def test_qkv_state_row_map_is_a_layout_of_the_qkv_weight():
    """sana_hip_qkv_state_rows (host code): q rows first, padded to whole 256-row tiles; then per tile of four heads
    [K h | V h | K h+1 | V h+1] twice; every row of the [3C, C] weight exactly once, the rest -1."""
    import ctypes
    lib = _lib.load()
    for heads in (1, 2, 5, 36, 70):
        C = 32 * heads
        n = lib.sana_hip_qkv_state_rows(C, heads, None, 0)
        q_pad = (C + 255) // 256 * 256
        assert n == q_pad + (heads + 3) // 4 * 256
        buf = (ctypes.c_int32 * n)()
        assert lib.sana_hip_qkv_state_rows(C, heads, ctypes.cast(buf, ctypes.c_void_p), n) == n
        rows = list(buf)
        assert rows[:C] == list(range(C)) and all(r == -1 for r in rows[C:q_pad])
        live = sorted(r for r in rows if r >= 0)
        assert live == list(range(3 * C))
        for i in range(q_pad, n):
            loc = (i - q_pad) % 256
            head = 4 * ((i - q_pad) // 256) + 2 * (loc // 128) + (loc // 64) % 2
            want = -1 if head >= heads else (1 + (loc // 32) % 2) * C + 32 * head + loc % 32
            assert rows[i] == want
    assert lib.sana_hip_qkv_state_rows(100, 3, None, 0) < 0          # C != 32 * heads
    assert lib.sana_hip_qkv_state_rows(64, 2, ctypes.cast((ctypes.c_int32 * 4)(), ctypes.c_void_p), 4) < 0
    assert lib.sana_hip_gemm_qkv_state_workspace_bytes(2, 512, 3) == 2 * 3 * 2 * 33 * 32 * 4
    assert lib.sana_hip_gemm_qkv_state_workspace_bytes(2, 500, 3) == 0
    assert lib.sana_hip_gemm_qkv_state_workspace_bytes(1, 500, 3) == 3 * 2 * 33 * 32 * 4   # one entry: a ragged last tile


def test_gemm_qkv_state_refuses_bad_arguments_before_any_launch():
    """The argument checks of sana_hip_gemm_qkv_state run on the host before anything is launched: wrong calls
    return their error code on a machine without a GPU too (the pointers below are never dereferenced)."""
    lib = _lib.load()
    P, ws = 0x10000, 1 << 30                      # a 16-byte aligned non-null "pointer", an ample workspace size
    call = lambda *a: lib.sana_hip_gemm_qkv_state(*a, None)
    good = [P, P, None, P, P, P, ws, 2, 512, 96, 3, 96, 96, 96]   # A W bias Q state ws bytes B N C heads lda ldw ldq
    bad = lambda i, v: good[:i] + [v] + good[i + 1:]
    assert call(*bad(0, None)) == -1 and call(*bad(3, None)) == -1 and call(*bad(7, 0)) == -1     # SANA_ERR_ARG
    assert call(*bad(8, 500)) == -2 and call(*bad(10, 4)) == -2                                    # SANA_ERR_SHAPE
    one = [P, P, P, P, P, P, ws, 1, 500, 96, 3, 96, 96, 96]      # one batch entry, ragged N: refused with a bias only
    assert call(*one) == -2
    assert call(*bad(11, 64)) == -1                                                                # lda < C
    assert call(*bad(0, P + 2)) == -3 and call(*bad(12, 100)) == -3                                # SANA_ERR_ALIGN
    assert call(*bad(6, 1024)) == -4 and call(*bad(5, None)) == -4                                 # SANA_ERR_WORKSPACE


@pytest.mark.parametrize("M,N,K,expand", [(4096, 3456, 1152, 1), (256, 1152, 2880, 1), (1024, 2240, 5600, 0), (0, 8, 16, 0),
                                          (1537, 6720, 2240, 1), (1536, 6720, 2240, 0), (3072, 3456, 1152, 0), (2048, 5760, 1152, 0),
                                          (1280, 11200, 2240, 0), (1281, 11200, 2240, 1), (2816, 5760, 1152, 0), (2817, 5760, 1152, 1)])
def test_which_int8_weights_are_expanded(M, N, K, expand):
    """Narrow outputs that are not split, a second round of int8 tiles, more than six token tiles on long rows of weights."""
    assert _lib.load().sana_hip_gemm_w8_expand(M, N, K) == expand


def test_packed_block_arguments_are_the_structure():
    """A value of its own for each field, packed in the fields' order, is read back under each field's name."""
    names = [n for n, _ in _lib.BlockArgs._fields_]
    values = [float(1 + i) if t is ctypes.c_float else 1 + i for i, (_, t) in enumerate(_lib.BlockArgs._fields_)]
    args = _lib.BlockArgs.from_buffer_copy(_lib.BLOCK_ARGS.pack(*values))
    assert [getattr(args, n) for n in names] == values


def test_the_block_call_fills_each_field(monkeypatch):
    """ops.block against the structure by name (a stand-in library: nothing is launched)."""
    import torch

    from sana_amd import ops

    seen = {}

    class Lib:
        def sana_hip_block_scratch_bytes(self, ref):
            return 64

        def sana_hip_block(self, ref, stream):
            a = ref._obj
            seen.update({n: getattr(a, n) for n, _ in _lib.BlockArgs._fields_})
            return 0

    monkeypatch.setattr(_lib, "load", lambda: Lib())
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    B, H, W, C, Nk, hid, heads = 2, 3, 5, 64, 7, 160, 4
    x, kv, mod = torch.zeros(B, H * W, C, dtype=torch.float16), torch.zeros(B, Nk, 3, 2 * C, dtype=torch.float16)[:, :, 1], \
        torch.zeros(B, 6, C, dtype=torch.float16)
    bias, ones, weights = torch.zeros(B, Nk), torch.ones(C), list(range(101, 115))
    weights[1] = 0                                # qkv without a bias
    out = ops.block(x, kv, bias, mod, weights, ones, hid, heads, (H, W), True, 1e-6, 2e-6, 1e-8)
    m = mod.data_ptr()
    want = dict(x=x.data_ptr(), text_kv=kv.data_ptr(), shift_msa=m, scale_msa=m + 2 * C, gate_msa=m + 4 * C, shift_mlp=m + 6 * C,
                scale_mlp=m + 8 * C, gate_mlp=m + 10 * C, ones=ones.data_ptr(), key_bias=bias.data_ptr(), out=out.data_ptr(),
                scratch_bytes=64, text_ld=6 * C, key_bias_ld=Nk, mod_stride=6 * C, B=B, N=H * W, C=C, hidden=hid, cross_heads=heads,
                text_len=Nk, H=H, W=W, round_like_reference=1, split_k=1 if ops.SPLIT_K else 0, io_dtype=_lib.DT_F16)
    want.update(zip(("qkv_w", "qkv_b", "proj_w", "proj_b", "q_w", "q_b", "o_w", "o_b", "inv_w", "inv_b", "dw_w", "dw_b", "point_w",
                     "point_b"), [w or None for w in weights]))
    floats = dict(eps_norm1=1e-6, eps_norm2=2e-6, eps_attn=1e-8, cross_scale=0.25)
    assert {n: seen[n] for n in want} == want and seen["scratch"]
    assert all(seen[n] == pytest.approx(v, rel=1e-6) for n, v in floats.items())
    assert set(want) | set(floats) | {"scratch"} == set(seen)


@pytest.mark.parametrize("M,N,K,straddling", [(6893, 4016, 2048, 2064), (12506, 5144, 4544, 4584), (13663, 1760, 1280, 1304),
                                              (17278, 3928, 1184, 1200)])
def test_rows_that_straddle_sectors_are_not_read_in_two_widths(M, N, K, straddling):
    """K % 32: one launch of 256 or 288 channels where k of whole sectors takes two widths."""
    plan = (ctypes.c_int * 4)()
    assert _lib.load().sana_hip_gemm_plan(M, N, K, plan) == 0 and plan[2] > 0
    assert _lib.load().sana_hip_gemm_plan(M, N, straddling, plan) == 0 and plan[1] in (256, 288) and plan[2:] == [0, 1]
