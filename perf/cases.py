"""The work that users of this framework have it do, as cases that can be timed and compared.

A case is a dict of plain values.  ``listed()`` names the ones that are always looked at, ``draw(rng)`` makes more
of the same ranges, ``prepare`` builds what a program holds before the call (weights, inputs, conditioning),
``run`` makes one pass through the public entry points, ``work`` says what the pass cannot do without and
``tolerance`` how far two correct implementations of the same precision may differ.

Four kinds of work:

* ``attn``    the ReLU linear attention alone on q, k, v (a program that keeps its own projections),
* ``image``   one denoising step through a run of SanaMSBlocks: the step's conditioning for all blocks, then the blocks,
              eagerly or replayed from a HIP graph, 16-bit or int8 weights, with or without q/k norm and padding mask,
* ``video``   one SanaVideoMSBlock on a whole latent clip: chunk-causal attention, chunked temporal Mix-FFN,
* ``stream``  the same block on one chunk of a clip that is generated chunk by chunk, with the cache of the chunks before.

Widths are those of the two image models (1152 with 16 cross-attention heads of 72, 2240 with 20 of 112) and the
video model (2240); Mix-FFN ratio 2.5, at most 300 text tokens.  ``depth`` is the number of blocks of the pass: fewer
than a model's 20 or 28, enough that the weights of one block have left the caches when it is called again.
"""
import math

import torch

import sana_amd
from sana_amd import ops

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
CROSS_HEADS = {1152: 16, 2240: 20}
IMAGE_DEPTH = {1152: 8, 2240: 4}


def _image(name, width, batch, h, w, *, dtype="bf16", text=300, int8=False, mask=False, qk_norm=False, graph=False):
    return {"name": name, "kind": "image", "width": width, "depth": IMAGE_DEPTH[width], "batch": batch, "h": h, "w": w,
            "dtype": dtype, "text": text, "int8": int8, "mask": mask, "qk_norm": qk_norm, "graph": graph}


def _video(name, kind, batch, frames, h, w, *, chunk=0, head_dim=112, text=300, per_frame=False):
    return {"name": name, "kind": kind, "width": 2240, "batch": batch, "frames": frames, "h": h, "w": w,
            "chunk": chunk, "head_dim": head_dim, "text": text, "per_frame": per_frame}


def listed():
    return [
        # the attention op alone at the 600M width, one 1024 px image, fp32: three launches of a few microseconds
        {"name": "attn_fp32_1024px", "kind": "attn", "heads": 36, "batch": 1, "tokens": 1024, "dtype": "fp32"},
        # a small preview image on the small model: latency of the launches and of the host
        _image("step_600m_512px", 1152, 1, 16, 16),
        # the released half-precision checkpoint with classifier-free guidance: a batch of two
        _image("step_600m_1024px_b2_fp16", 1152, 2, 32, 32, dtype="fp16"),
        # four images on the small model
        _image("step_600m_1024px_b4", 1152, 4, 32, 32),
        # a single image on the large model, as a serving loop replays it
        _image("step_1600m_1024px_graph", 2240, 1, 32, 32, graph=True),
        # int8 weights where memory is short: one prompt with guidance
        _image("step_1600m_1024px_b2_int8", 2240, 2, 32, 32, int8=True),
        # an aspect-ratio bucket: rows that are no multiple of any tile, padded prompts
        _image("step_1600m_27x36_b3_mask", 2240, 3, 27, 36, mask=True, text=230),
        # a 2048 px image on the variant with q/k norm
        _image("step_1600m_2048px_qknorm", 2240, 1, 64, 64, qk_norm=True),
        # throughput serving: sixteen 1024 px images
        _image("step_1600m_1024px_b16", 2240, 16, 32, 32),
        # one 4096 px image
        _image("step_1600m_4096px", 2240, 1, 128, 128),
        # a whole 480p clip of 21 latent frames in two causal chunks
        _video("video_480p_21f", "video", 1, 21, 30, 52, chunk=11),
        # the next three latent frames of a clip that is generated as a stream
        _video("stream_480p_3f", "stream", 1, 3, 30, 52),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_any(rng):
    kind = rng.choices(["attn", "image", "video", "stream"], [1, 6, 1.5, 1.5])[0]
    if kind == "attn":
        return {"kind": "attn", "heads": rng.choice([36, 70]), "batch": rng.randint(1, 4),
                "tokens": _log_int(rng, 64, 16384), "dtype": rng.choice(["fp32", "bf16"])}
    if kind == "image":
        width = rng.choice([1152, 2240, 2240])
        side = _log_int(rng, 12, 128)
        ratio = math.exp(rng.uniform(-math.log(2.0), math.log(2.0)))
        h, w = max(8, min(128, round(side * ratio))), max(8, min(128, round(side / ratio)))
        variant = rng.choices(["plain", "fp16", "int8", "qk_norm", "graph"], [4, 1.5, 1.5, 1, 1.5])[0]
        return _image("", width, _log_int(rng, 1, 16), h, w, dtype="fp16" if variant == "fp16" else "bf16",
                      text=rng.choice([300, 300, rng.randint(16, 300)]), int8=variant == "int8", mask=rng.random() < 0.3,
                      qk_norm=variant == "qk_norm", graph=variant == "graph")
    h, w = rng.randint(12, 45), rng.randint(12, 80)
    text = rng.choice([300, rng.randint(16, 300)])
    head_dim = rng.choice([112, 112, 32])
    if kind == "video":
        frames = rng.randint(5, 21)
        return _video("", "video", 1, frames, h, w, chunk=rng.choice([0, rng.randint(1, frames)]), head_dim=head_dim,
                      text=text, per_frame=rng.random() < 0.3)
    return _video("", "stream", rng.randint(1, 2), rng.randint(1, 5), h, w, head_dim=head_dim, text=text)


def draw(rng):
    most = max(work(c)["flops"] for c in listed())
    while True:
        case = _draw_any(rng)
        case.pop("name", None)
        if work(case)["flops"] <= most:
            return case


# ------------------------------------------------------------------ what a pass cannot do without


def work(case):
    kind = case["kind"]
    if kind == "attn":
        C, M = 32 * case["heads"], case["batch"] * case["tokens"]
        item = 4 if case["dtype"] == "fp32" else 2
        return {"bytes": 4 * M * C * item, "flops": 4 * M * C * 33}
    C, text, B = case["width"], case["text"], case["batch"]
    hid = int(C * 2.5)
    M = B * case["h"] * case["w"] * case.get("frames", 1)
    d = case.get("head_dim", 32)
    # per block: qkv, attention state and its application, proj; cross-attention's q, kv, products, proj; Mix-FFN
    flops = 2 * M * C * 3 * C + 4 * M * C * (d + 1) + 2 * M * C * C
    flops += 4 * M * C * C + 4 * B * text * C * C + 4 * M * text * C
    flops += 2 * M * C * 2 * hid + 18 * M * 2 * hid + 2 * M * hid * C
    main = 4 * C * C + 3 * C * hid              # the weights that int8 halves
    weights = main * (1 if case.get("int8") else 2) + 2 * (4 * C * C + 9 * 2 * hid + 20 * C + 2 * hid)
    io = 2 * (2 * M * C + B * text * C + 6 * B * C * (case["frames"] if case.get("per_frame") else 1))
    if kind == "image":
        return {"bytes": case["depth"] * weights + io, "flops": case["depth"] * flops}
    flops += 6 * M * C * C                      # the temporal convolution
    weights += 2 * 3 * C * C
    io += 8 * M * (d // 2)                      # rotary factors, complex64
    if kind == "stream":                        # the cache of the chunks before, read and written
        io += 2 * B * (4 * C * (d + 1) + 2 * case["h"] * case["w"] * C)
    return {"bytes": weights + io, "flops": flops}


def tolerance(case):
    if case["kind"] == "attn":
        # fp32: 1.2e-7 from the fp64 answer; bf16: sums in fp32 whose order tips a rounding of the result now and then
        return {"rel": 1e-6, "max": 1e-5} if case["dtype"] == "fp32" else {"rel": 2e-3, "max": 2e-2}
    # activations rounded a dozen times a block and carried over the blocks of the pass: against the same blocks on
    # stock operators at the same precision, bf16 is off by 3.8e-3 ... 4.6e-3 (largest value 4.2e-2), fp16 by 5.0e-4 (4.7e-3)
    return {"rel": 2e-3, "max": 2e-2} if case.get("dtype") == "fp16" else {"rel": 1.6e-2, "max": 0.17}


# ------------------------------------------------------------------ what a program holds before the call


def _fill(module, gen):
    """Weights of a trained model's scale: truncated normal of 0.02, biases and the modulation table not zero."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            r = torch.randn(p.shape, generator=gen, device="cuda")
            if name.endswith("scale_shift_table"):
                p.copy_(r * 0.3)
            elif name.endswith("norm.weight"):
                p.copy_(1 + 0.1 * r)
            elif name.endswith("depth_conv.conv.weight"):
                p.copy_(0.2 * r)
            elif name.endswith("t_conv.weight"):
                p.copy_(0.01 * r.clamp_(-2, 2))
            else:
                p.copy_(0.02 * r.clamp_(-2, 2))
    return module


def _prompt_mask(B, text, gen):
    """A 0 / 1 row per prompt: the first few dozen to all of its tokens count."""
    lengths = torch.randint(max(1, text // 8), text + 1, (B, 1), generator=gen, device="cuda")
    return (torch.arange(text, device="cuda")[None] < lengths).to(torch.int16)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    randn = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    kind, B = case["kind"], case["batch"]
    if kind == "attn":
        dtype, C, N = DTYPES[case["dtype"]], 32 * case["heads"], case["tokens"]
        qkv = randn(B, N, 3, C).to(dtype)     # as one projection writes it
        return {"kind": kind, "q": qkv[:, :, 0], "k": qkv[:, :, 1], "v": qkv[:, :, 2]}
    C, text = case["width"], case["text"]
    N = case["h"] * case["w"] * case.get("frames", 1)
    dtype = DTYPES[case.get("dtype", "bf16")]
    state = {"kind": kind, "x": randn(B, N, C).to(dtype), "y": randn(B, text, C).to(dtype)}
    if kind == "image":
        blocks = []
        for _ in range(case["depth"]):
            with torch.device("cuda"):
                block = sana_amd.SanaMSBlock(C, CROSS_HEADS[C], mlp_ratio=2.5, attn_type="linear", ffn_type="glumbconv",
                                             qk_norm=case["qk_norm"])
            block = _fill(block, gen).to(dtype).eval()
            if case["int8"]:
                block.quantize_w8_()
            blocks.append(block)
        state["t"] = (0.3 * randn(B, 6 * C)).to(dtype)
        state["mask"] = _prompt_mask(B, text, gen) if case["mask"] else None
        state["HW"] = (case["h"], case["w"])
        state["blocks"], state["cond"] = blocks, sana_amd.StepConditioning(blocks)
        if case["graph"]:
            state["replay"] = sana_amd.GraphedCall(lambda x, y, t: _step(state, x, y, t), [state["x"], state["y"], state["t"]])
        return state
    d = case["head_dim"]
    with torch.device("cuda"):
        block = sana_amd.SanaVideoMSBlock(
            C, CROSS_HEADS[C], mlp_ratio=2.5, qk_norm=True, linear_head_dim=d,
            attn_type="chunkcausal" if kind == "video" else "cachedcausal",
            ffn_type="ChunkGLUMBConvTemp" if kind == "video" else "CachedGLUMBConvTemp")
    state["block"] = _fill(block, gen).to(dtype).eval()
    frames = case["frames"]
    state["t"] = (0.3 * randn(*((B, 1, frames, 6 * C) if case["per_frame"] else (B, 6 * C)))).to(dtype)
    state["THW"] = (frames, case["h"], case["w"])
    angle = 6.2831853 * torch.rand(1, 1, N, d // 2, generator=gen, device="cuda")
    state["rotary"] = torch.polar(torch.ones_like(angle), angle)
    if kind == "video":
        state["chunks"] = list(range(0, frames, case["chunk"])) if case["chunk"] else None
    else:
        # what an earlier chunk left: sums over its tokens of relu(k) v and relu(k), and its last frame
        h = C // d
        state["cache"] = [3.0 * N ** 0.5 * randn(B, h, d, d), N * (0.4 + 0.02 * randn(B, h, 1, d)).abs(),
                          randn(B, C, 1, case["h"] * case["w"]).to(dtype)]
    return state


# ------------------------------------------------------------------ one pass


def _step(state, x, y, t):
    for block, shared in zip(state["blocks"], state["cond"](y, t)):
        x = block(x, y, t, state["mask"], state["HW"], **shared)
    return x


def run(state):
    kind = state["kind"]
    with torch.no_grad():
        if kind == "attn":
            return ops.relu_linear_attention(state["q"], state["k"], state["v"], 1e-15)
        x, y, t = state["x"], state["y"], state["t"]
        if kind == "image":
            return state["replay"](x, y, t) if "replay" in state else _step(state, x, y, t)
        if kind == "video":
            return state["block"](x, y, t, THW=state["THW"], rotary_emb=state["rotary"], chunk_index=state["chunks"])
        # the call replaces the slots of the list it is given; the state keeps its own
        out, cache = state["block"](x, y, t, THW=state["THW"], rotary_emb=state["rotary"], save_kv_cache=True,
                                    kv_cache=list(state["cache"]))
        return [out, *cache]
