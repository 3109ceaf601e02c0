"""The performance cases: what users of this framework have it compute, as layers, blocks and one
whole denoising step, with the float64 evaluation of each.

A case is a dict with a ``kind`` (one entry point) and its sizes. ``listed`` gives the fixed ones,
``draw`` others of the same ranges: video from a few hundred latent tokens to the 27 280 of a long
clip, stills from 256 to 4096 image tokens, text contexts of 64 to 1024 tokens, the audio stream's
few hundred rows, bf16 and fp16, dense and quantized weights, odd token counts among them.
Everything here is inference: the one direction that the framework has.
"""

from __future__ import annotations

import math

import torch

DEVICE = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


# ---- the cases -----------------------------------------------------------------------------------


def listed() -> list[dict]:
    return [
        # the modulation of one denoising step: one timestep through the AdaLN producer (every step
        # of every model runs it; a chain of one-row products over all of its weights)
        {"name": "adaln_1", "kind": "adaln", "dim": 4096, "rows": 9, "steps": 1},
        # the audio stream's self-attention layer: 5 s of audio latents, 64-wide heads, in the fp16
        # that the LTX-2 transformer runs in by default
        {"name": "audio_attention_127", "kind": "attention", "tokens": 127, "context": 0, "heads": 32,
         "head_dim": 64, "dtype": "fp16", "masked": False},
        # text cross-attention of a stage-2 clip (16 x 14 x 24 latents), the prompt padded to 256
        # tokens and masked
        {"name": "text_attention_5376", "kind": "attention", "tokens": 5376, "context": 256, "heads": 32,
         "head_dim": 128, "dtype": "fp16", "masked": True},
        # the feed-forward layer of a small clip with int8 weights, an odd number of rows
        {"name": "feed_forward_1111_int8", "kind": "feed_forward", "tokens": 1111, "dim": 4096, "weights": "int8"},
        # one whole denoising step (X0 model of two blocks, Euler update, finite check) of a
        # preview: 5 x 8 x 12 latents, where launches and host work count
        {"name": "denoise_480", "kind": "denoise", "frames": 5, "height": 8, "width": 12, "text": 128, "blocks": 2},
        # one LTX-2 block at the benchmark's size and, the largest, at its long-clip size with
        # int4 weights
        {"name": "ltx_block_9216", "kind": "ltx_block", "frames": 16, "height": 18, "width": 32, "text": 256,
         "weights": "bf16"},
        {"name": "ltx_block_27280_int4", "kind": "ltx_block", "frames": 31, "height": 22, "width": 40, "text": 256,
         "weights": "int4"},
        # a small still image: the benchmark's 32 x 32 + 128 GELU double block, 64-wide heads
        {"name": "image_block_1152", "kind": "flux_double", "height": 32, "width": 32, "text": 128, "dim": 1024,
         "heads": 16, "ff": 4096, "act": "gelu"},
        # FLUX.2 at 1024 x 1024 (64 x 64 + 512): the double block, and the single block on an
        # odd-sized still with a short prompt
        {"name": "flux_double_4608", "kind": "flux_double", "height": 64, "width": 64, "text": 512, "dim": 4096,
         "heads": 32, "ff": 12288, "act": "swiglu"},
        {"name": "flux_single_2628", "kind": "flux_single", "height": 45, "width": 51, "text": 333, "dim": 4096,
         "heads": 32, "ff": 12288},
        # the joint audio/video block of the stage-2 clip
        {"name": "av_block_5376", "kind": "av_block", "frames": 16, "height": 14, "width": 24, "text": 256,
         "audio": 127},
        # a Krea 2 block: grouped-query attention (24 query, 8 key/value heads), odd token count
        {"name": "krea_block_2305", "kind": "krea_block", "tokens": 2305, "heads": 24, "kv_heads": 8, "ff": 8192},
    ]


def _log(rng, low: float, high: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _video_grid(rng, low: int, high: int) -> dict:
    """A latent grid (frames, height, width) of about ``low`` to ``high`` tokens."""
    tokens = _log(rng, low, high)
    frames = max(1, min(31, _log(rng, 2, 31)))
    plane = max(12.0, tokens / frames)
    aspect = rng.uniform(0.5, 2.0)
    h = max(3, int(math.sqrt(plane / aspect)))
    w = max(3, int(plane / h))
    while frames * h * w > high:
        w -= 1
    return {"frames": frames, "height": h, "width": w}


def _image_grid(rng) -> dict:
    return {"height": rng.randint(16, 64), "width": rng.randint(16, 64)}


def draw(rng) -> dict:
    kind = rng.choice(["adaln", "audio_attention", "text_attention", "feed_forward", "denoise", "ltx_block",
                       "ltx_block", "image_block", "flux_double", "flux_single", "av_block", "krea_block"])
    if kind == "adaln":
        return {"kind": kind, "dim": rng.choice([2048, 4096]), "rows": rng.choice([1, 2, 4, 9]),
                "steps": _log(rng, 1, 8)}
    if kind == "audio_attention":
        return {"kind": "attention", "tokens": _log(rng, 50, 760), "context": 0, "heads": 32, "head_dim": 64,
                "dtype": rng.choice(["fp16", "bf16"]), "masked": False}
    if kind == "text_attention":
        return {"kind": "attention", "tokens": _log(rng, 384, 16384), "context": rng.randint(64, 1024), "heads": 32,
                "head_dim": 128, "dtype": rng.choice(["fp16", "bf16"]), "masked": rng.random() < 0.5}
    if kind == "feed_forward":
        return {"kind": kind, "tokens": _log(rng, 256, 9216), "dim": rng.choice([2048, 4096]),
                "weights": rng.choice(["bf16", "fp16", "int4", "int8", "mxfp8"])}
    if kind == "denoise":
        return {"kind": kind, **_video_grid(rng, 96, 3000), "text": rng.randint(64, 512), "blocks": 2}
    if kind == "ltx_block":
        return {"kind": kind, **_video_grid(rng, 384, 27280), "text": rng.randint(64, 256),
                "weights": rng.choice(["bf16", "fp16", "int4", "int8", "mxfp8"])}
    if kind == "image_block":
        return {"kind": "flux_double", **_image_grid(rng), "text": rng.randint(64, 512), "dim": 1024, "heads": 16,
                "ff": 4096, "act": "gelu"}
    if kind == "flux_double":
        return {"kind": kind, **_image_grid(rng), "text": rng.randint(64, 512), "dim": 4096, "heads": 32,
                "ff": 12288, "act": "swiglu"}
    if kind == "flux_single":
        return {"kind": kind, **_image_grid(rng), "text": rng.randint(64, 512), "dim": 4096, "heads": 32,
                "ff": 12288}
    if kind == "av_block":
        return {"kind": kind, **_video_grid(rng, 768, 9216), "text": rng.randint(64, 256),
                "audio": _log(rng, 50, 500)}
    return {"kind": "krea_block", "tokens": _log(rng, 320, 4608), "heads": 24, "kv_heads": 8, "ff": 8192}


# ---- inputs: everything drawn on the GPU from the seed ---------------------------------------------


class _Draw:
    """Named tensors N(mean, std^2), drawn in the order of the calls."""

    def __init__(self, seed: int, dtype: torch.dtype = torch.bfloat16) -> None:
        self.gen = torch.Generator(device=DEVICE).manual_seed(int(seed))
        self.dtype = dtype
        self.p: dict[str, torch.Tensor] = {}

    def normal(self, shape, std: float = 1.0, mean: float = 0.0, dtype: torch.dtype | None = None) -> torch.Tensor:
        t = torch.randn(tuple(shape), generator=self.gen, device=DEVICE, dtype=torch.float32) * std + mean
        return t.to(self.dtype if dtype is None else dtype)

    def linear(self, name: str, n: int, k: int, bias: bool = True) -> None:
        self.p[f"{name}.weight"] = self.normal((n, k), 0.02)
        if bias:
            self.p[f"{name}.bias"] = self.normal((n,), 0.02)

    def attention(self, name: str, qdim: int, cdim: int, heads: int, head_dim: int) -> None:
        inner = heads * head_dim
        for part, n, k in (("to_q", inner, qdim), ("to_k", inner, cdim), ("to_v", inner, cdim), ("to_out", qdim, inner),
                           ("to_gate_logits", heads, qdim)):
            self.linear(f"{name}.{part}", n, k)
        for part in ("q_norm", "k_norm"):
            self.p[f"{name}.{part}.weight"] = self.normal((inner,), 0.02, 1.0)

    def ltx(self, pre: str, dim: int, heads: int, head_dim: int) -> None:
        self.attention(f"{pre}attn1", dim, dim, heads, head_dim)
        self.attention(f"{pre}attn2", dim, dim, heads, head_dim)
        self.linear(f"{pre}ff.proj_in", 4 * dim, dim)
        self.linear(f"{pre}ff.proj_out", dim, 4 * dim)
        self.p[f"{pre}scale_shift_table"] = self.normal((9, dim), 0.02, dtype=torch.float32)
        self.p[f"{pre}prompt_scale_shift_table"] = self.normal((2, dim), 0.02, dtype=torch.float32)

    def modulation(self, rows: int, dim: int) -> torch.Tensor:
        """The AdaLN rows of one step: the spread that a 0.02-weight projection of a 1024-wide
        conditioning vector gives."""
        return self.normal((1, 1, rows, dim), 0.64)


def _quantize(weight: torch.Tensor, weights: str):
    """A packed weight in the checkpoint's format and the weight it stands for, in float64."""
    n, k = weight.shape
    if weights == "mxfp8":
        w = weight.double().view(n, k // 32, 32)
        exponent = (torch.floor(torch.log2(w.abs().amax(-1))) - 8).clamp(-127, 127)
        codes = (w * torch.exp2(-exponent)[..., None]).float().clamp(-448, 448).to(torch.float8_e4m3fn)
        dense = (codes.double() * torch.exp2(exponent)[..., None]).view(n, k)
        return codes.view(n, k).view(torch.int32), (exponent + 127).to(torch.uint8), None, dense
    bits = 4 if weights == "int4" else 8
    w = weight.float().view(n, k // 64, 64)
    low, high = w.amin(-1), w.amax(-1)
    scales = ((high - low) / (2 ** bits - 1)).bfloat16()
    biases = low.bfloat16()
    codes = ((w - biases.float()[..., None]) / scales.float()[..., None]).round().clamp(0, 2 ** bits - 1)
    # the format's value is bf16(scale * code + bias), the sum exact in float32
    dense = (codes * scales.float()[..., None] + biases.float()[..., None]).bfloat16().double().view(n, k)
    codes = codes.to(torch.uint8).view(n, k)
    if bits == 4:
        codes = codes[:, 0::2] | (codes[:, 1::2] << 4)
    return codes.contiguous().view(torch.int32), scales, biases, dense


def _ltx_names(pre: str = "") -> list[str]:
    parts = [f"{a}.{n}" for a in ("attn1", "attn2") for n in ("to_q", "to_k", "to_v", "to_out", "to_gate_logits")]
    return [f"{pre}{n}" for n in parts + ["ff.proj_in", "ff.proj_out"]]


def _video_tables(grid, dim: int, heads: int):
    """float64 split-RoPE angles' cosine and sine, ``(1, T, heads, dim / 2 heads)``, of a latent grid."""
    axes = torch.meshgrid(*(torch.arange(n, device=DEVICE, dtype=torch.float64) for n in grid), indexing="ij")
    return _axis_tables([a.reshape(-1) + 0.5 for a in axes], (20.0, 2048.0, 2048.0), dim, heads)


def _axis_tables(axes, max_pos, dim: int, heads: int):
    count = dim // (2 * len(axes))
    freqs = 10000.0 ** (torch.arange(count, device=DEVICE, dtype=torch.float64) / (count - 1)) * (math.pi / 2)
    angles = torch.stack([(a / m * 2 - 1)[:, None] * freqs for a, m in zip(axes, max_pos)], dim=-1)
    angles = angles.flatten(1)
    pad = torch.zeros((angles.shape[0], dim // 2 - angles.shape[1]), device=DEVICE, dtype=torch.float64)
    angles = torch.cat([pad, angles], dim=1)
    tables = angles.view(1, angles.shape[0], heads, -1)
    return tables.cos(), tables.sin()


def _head_major(tables):
    """The tables as the layers take them: float32, ``(1, heads, T, half)`` views of token-major rows."""
    return tuple(t.float().contiguous().transpose(1, 2) for t in tables)


def _pair_tables(grid, text: int, dims, theta: float):
    """Adjacent-pair tables ``(1, T, 1, Dh)`` in float32: text rows at the origin, then the image grid."""
    hh, ww = torch.meshgrid(*(torch.arange(n, device=DEVICE, dtype=torch.float64) for n in grid), indexing="ij")
    image = torch.stack([hh.reshape(-1), ww.reshape(-1)], dim=-1)
    positions = torch.cat([torch.zeros((text, 2), device=DEVICE, dtype=torch.float64), image])
    parts = []
    for axis, d in enumerate(dims):
        freqs = theta ** (-torch.arange(0, d, 2, device=DEVICE, dtype=torch.float64) / d)
        parts.append(torch.repeat_interleave(positions[:, axis, None] * freqs, 2, dim=-1))
    angles = torch.cat(parts, dim=-1)[None, :, None]
    return angles.cos().float(), angles.sin().float()


def _grid(case: dict) -> list[int]:
    return [case[axis] for axis in ("frames", "height", "width") if axis in case]


def _tokens(grid) -> int:
    return math.prod(grid)


def _inputs(case: dict, seed: int) -> dict:
    """Weights and inputs of a case, the same for ``prepare`` and ``exact``."""
    kind = case["kind"]
    dtype = DTYPES.get(case.get("dtype", case.get("weights", "bf16")), torch.bfloat16)
    d = _Draw(seed, dtype)
    p = d.p
    if kind == "adaln":
        dim = case["dim"]
        d.linear("linear_1", dim, 256)
        d.linear("linear_2", dim, dim)
        d.linear("linear", case["rows"] * dim, dim)
        p["timesteps"] = torch.rand(case["steps"], generator=d.gen, device=DEVICE)
    elif kind == "attention":
        dim = case["heads"] * case["head_dim"]
        d.attention("attn", dim, dim, case["heads"], case["head_dim"])
        p["x"] = d.normal((1, case["tokens"], dim))
        p["residual"] = d.normal((1, case["tokens"], dim), dtype=torch.float32)
        p["gate"] = d.normal((1, 1, dim), 0.64, dtype=torch.float32)
        if case["context"]:
            p["context"] = d.normal((1, case["context"], dim))
            if case["masked"]:
                # a prompt padded to the context's length: the additive mask of the padding
                keep = max(1, (2 * case["context"]) // 3)
                mask = torch.zeros((1, 1, 1, case["context"]), device=DEVICE)
                mask[..., keep:] = torch.finfo(dtype).min
                p["mask"] = mask.to(dtype)
    elif kind == "feed_forward":
        dim = case["dim"]
        d.linear("ff.proj_in", 4 * dim, dim)
        d.linear("ff.proj_out", dim, 4 * dim)
        p["x"] = d.normal((1, case["tokens"], dim))
        p["residual"] = d.normal((1, case["tokens"], dim), dtype=torch.float32)
        p["gate"] = d.normal((1, 1, dim), 0.64, dtype=torch.float32)
    elif kind == "ltx_block":
        d.ltx("", 4096, 32, 128)
        p["timesteps"] = d.modulation(9, 4096)
        p["x"] = d.normal((1, _tokens(_grid(case)), 4096))
        p["context"] = d.normal((1, case["text"], 4096))
    elif kind == "av_block":
        d.ltx("", 4096, 32, 128)
        d.ltx("audio_", 2048, 32, 64)
        d.attention("audio_to_video_attn", 4096, 2048, 32, 64)
        d.attention("video_to_audio_attn", 2048, 4096, 32, 64)
        p["scale_shift_table_a2v_ca_video"] = d.normal((5, 4096), 0.02, dtype=torch.float32)
        p["scale_shift_table_a2v_ca_audio"] = d.normal((5, 2048), 0.02, dtype=torch.float32)
        for pre, dim, tokens in (("", 4096, _tokens(_grid(case))), ("audio_", 2048, case["audio"])):
            p[f"{pre}timesteps"] = d.modulation(9, dim)
            p[f"{pre}cross_ss"] = d.modulation(4, dim)
            p[f"{pre}cross_gate"] = d.modulation(1, dim)
            p[f"{pre}x"] = d.normal((1, tokens, dim))
            p[f"{pre}context"] = d.normal((1, case["text"], dim))
    elif kind == "denoise":
        for i in range(case["blocks"]):
            block = _Draw(seed * 1000 + 1 + i)
            block.ltx("", 4096, 32, 128)
            p[f"block{i}"] = block.p
        d.linear("patchify_proj", 4096, 128)
        for name, rows in (("adaln_single", 9), ("prompt_adaln_single", 2)):
            d.linear(f"{name}.emb.timestep_embedder.linear_1", 4096, 256)
            d.linear(f"{name}.emb.timestep_embedder.linear_2", 4096, 4096)
            d.linear(f"{name}.linear", rows * 4096, 4096)
        p["scale_shift_table"] = d.normal((2, 4096), 0.02)
        d.linear("proj_out", 128, 4096)
        p["x"] = d.normal((1, _tokens(_grid(case)), 128))
        p["context"] = d.normal((1, case["text"], 4096))
    elif kind in ("flux_double", "flux_single"):
        dim, ff, heads = case["dim"], case["ff"], case["heads"]
        head_dim = dim // heads
        if kind == "flux_double":
            for n in ("to_q", "to_k", "to_v", "add_q_proj", "add_k_proj", "add_v_proj", "to_out", "to_add_out"):
                d.linear(f"attn.{n}", dim, dim, bias=False)
            for n in ("norm_q", "norm_k", "norm_added_q", "norm_added_k"):
                p[f"attn.{n}.weight"] = d.normal((head_dim,), 0.02, 1.0)
            for pre in ("ff", "ff_context"):
                if case["act"] == "swiglu":
                    d.linear(f"{pre}.linear_in", 2 * ff, dim, bias=False)
                    d.linear(f"{pre}.linear_out", dim, ff, bias=False)
                else:
                    d.linear(f"{pre}.proj_in", ff, dim)
                    d.linear(f"{pre}.proj_out", dim, ff)
            p["image"] = d.normal((1, _tokens(_grid(case)), dim))
            p["text"] = d.normal((1, case["text"], dim))
            p["image_mod"] = d.normal((1, 6 * dim), 0.64)
            p["text_mod"] = d.normal((1, 6 * dim), 0.64)
        else:
            d.linear("single.attn.to_qkv_mlp_proj", 3 * dim + 2 * ff, dim, bias=False)
            d.linear("single.attn.to_out", dim, dim + ff, bias=False)
            for n in ("norm_q", "norm_k"):
                p[f"single.attn.{n}.weight"] = d.normal((head_dim,), 0.02, 1.0)
            p["x"] = d.normal((1, _tokens(_grid(case)) + case["text"], dim))
            p["mod"] = d.normal((1, 3 * dim), 0.64)
        p["tables"] = _pair_tables(_grid(case), case["text"], (head_dim // 2, head_dim // 2), 10000.0)
    elif kind == "krea_block":
        heads, kv, ff = case["heads"], case["kv_heads"], case["ff"]
        dim = heads * 128
        for n, rows in (("to_q", dim), ("to_k", kv * 128), ("to_v", kv * 128), ("to_gate", dim), ("to_out", dim)):
            d.linear(f"attn.{n}", rows, dim, bias=False)
        d.linear("ff.gate", ff, dim, bias=False)
        d.linear("ff.up", ff, dim, bias=False)
        d.linear("ff.down", dim, ff, bias=False)
        for n, width in (("attn.norm_q", 128), ("attn.norm_k", 128), ("norm1", dim), ("norm2", dim)):
            p[f"{n}.weight"] = d.normal((width,), 0.1, dtype=torch.float32)
        p["scale_shift_table"] = d.normal((6, dim), 0.1, dtype=torch.float32)
        p["x"] = d.normal((1, case["tokens"], dim))
        p["mod"] = d.normal((1, 6 * dim), 0.3)
        ids = torch.randint(0, 64, (1, case["tokens"], 3), generator=d.gen, device=DEVICE)
        parts = []
        for axis, width in enumerate((32, 32, 64)):
            freqs = 1000.0 ** (-torch.arange(0, width, 2, device=DEVICE, dtype=torch.float64) / width)
            parts.append(torch.repeat_interleave(ids[..., axis, None].double() * freqs, 2, dim=-1))
        angles = torch.cat(parts, dim=-1)
        p["tables"] = (angles.cos().float(), angles.sin().float())
    else:
        raise ValueError(f"unknown kind {kind}")
    return p


def _quantized_names(case: dict) -> list[str]:
    if case.get("weights") not in ("int4", "int8", "mxfp8"):
        return []
    return _ltx_names() if case["kind"] == "ltx_block" else ["ff.proj_in", "ff.proj_out"]


# ---- prepare and run -------------------------------------------------------------------------------


def _layer(p: dict, name: str, quantized: str | None = None):
    from kinomlx_amd.kernels.quantized import QuantizedLinear
    from kinomlx_amd.ltx2.attention import Linear

    weight, bias = p[f"{name}.weight"], p.get(f"{name}.bias")
    if quantized is None:
        return Linear(weight, bias)
    words, scales, biases, _ = _quantize(weight, quantized)
    if quantized == "mxfp8":
        return QuantizedLinear(words, scales, None, bias, mode="mxfp8")
    return QuantizedLinear(words, scales, biases, bias, group_size=64, bits=4 if quantized == "int4" else 8)


def _fill_attention(attn, p: dict, name: str, quantized: str | None = None) -> None:
    for part in ("to_q", "to_k", "to_v", "to_out", "to_gate_logits"):
        setattr(attn, part, _layer(p, f"{name}.{part}", quantized))
    attn.q_norm.weight = p[f"{name}.q_norm.weight"]
    attn.k_norm.weight = p[f"{name}.k_norm.weight"]


def _fill_ltx(block, p: dict, pre: str, quantized: str | None = None) -> None:
    for a in ("attn1", "attn2"):
        _fill_attention(getattr(block, f"{pre}{a}"), p, f"{pre}{a}", quantized)
    ff = getattr(block, f"{pre}ff")
    ff.project_in.proj = _layer(p, f"{pre}ff.proj_in", quantized)
    ff.project_out = _layer(p, f"{pre}ff.proj_out", quantized)
    for table in ("scale_shift_table", "prompt_scale_shift_table"):
        setattr(block, f"{pre}{table}", p[f"{pre}{table}"])


def prepare(case: dict, seed: int) -> dict:
    p = _inputs(case, seed)
    kind = case["kind"]
    quantized = case["weights"] if _quantized_names(case) else None
    state: dict = {"kind": kind}
    if kind == "adaln":
        from kinomlx_amd.ltx2.timestep import AdaLayerNormSingle

        layer = AdaLayerNormSingle(case["dim"], case["rows"])
        layer.emb.timestep_embedder.linear_1 = _layer(p, "linear_1")
        layer.emb.timestep_embedder.linear_2 = _layer(p, "linear_2")
        layer.linear = _layer(p, "linear")
        state.update(layer=layer, timesteps=p["timesteps"])
    elif kind == "attention":
        from kinomlx_amd.ltx2.attention import Attention

        dim = case["heads"] * case["head_dim"]
        layer = Attention(dim, heads=case["heads"], dim_head=case["head_dim"], apply_gated_attention=True)
        _fill_attention(layer, p, "attn")
        layer.fuse_projections(self_attention=not case["context"])
        pe = None
        if not case["context"]:
            seconds = torch.arange(case["tokens"], device=DEVICE, dtype=torch.float64) / 25.0
            pe = _head_major(_axis_tables([seconds], (20.0,), dim, case["heads"]))
        state.update(layer=layer, x=p["x"], context=p.get("context"), mask=p.get("mask"), pe=pe,
                     residual=p["residual"], gate=p["gate"])
    elif kind == "feed_forward":
        from kinomlx_amd.ltx2.feed_forward import FeedForward

        layer = FeedForward(case["dim"])
        layer.project_in.proj = _layer(p, "ff.proj_in", quantized)
        layer.project_out = _layer(p, "ff.proj_out", quantized)
        state.update(layer=layer, x=p["x"], residual=p["residual"], gate=p["gate"])
    elif kind == "ltx_block":
        from kinomlx_amd.ltx2.transformer import BasicAVTransformerBlock, TransformerArgs, TransformerConfig

        block = BasicAVTransformerBlock(0, video_config=TransformerConfig(4096, 32, 128, 4096))
        _fill_ltx(block, p, "", quantized)
        block.fuse_projections()
        state.update(block=block, video=TransformerArgs(
            x=p["x"], context=p["context"], timesteps=p["timesteps"],
            positional_embeddings=_head_major(_video_tables(_grid(case), 4096, 32))))
    elif kind == "av_block":
        from kinomlx_amd.ltx2.transformer import BasicAVTransformerBlock, TransformerArgs, TransformerConfig

        block = BasicAVTransformerBlock(0, video_config=TransformerConfig(4096, 32, 128, 4096),
                                        audio_config=TransformerConfig(2048, 32, 64, 2048))
        for pre in ("", "audio_"):
            _fill_ltx(block, p, pre)
        for name in ("audio_to_video_attn", "video_to_audio_attn"):
            _fill_attention(getattr(block, name), p, name)
        block.scale_shift_table_a2v_ca_video = p["scale_shift_table_a2v_ca_video"]
        block.scale_shift_table_a2v_ca_audio = p["scale_shift_table_a2v_ca_audio"]
        block.fuse_projections()
        for stream, tables in _av_tables(case).items():
            pre = "" if stream == "video" else "audio_"
            state[stream] = TransformerArgs(
                x=p[f"{pre}x"], context=p[f"{pre}context"], timesteps=p[f"{pre}timesteps"],
                positional_embeddings=_head_major(tables[0]), cross_positional_embeddings=_head_major(tables[1]),
                cross_scale_shift_timestep=p[f"{pre}cross_ss"], cross_gate_timestep=p[f"{pre}cross_gate"])
        state["block"] = block
    elif kind == "denoise":
        from kinomlx_amd.ltx2.model import LTXAVModel
        from kinomlx_amd.ltx2.state import LatentState
        from kinomlx_amd.ltx2.wrappers import X0Model

        model = LTXAVModel(num_layers=case["blocks"])
        for i, block in enumerate(model.transformer_blocks):
            _fill_ltx(block, p[f"block{i}"], "")
            block.fuse_projections()
        model.patchify_proj = _layer(p, "patchify_proj")
        for name in ("adaln_single", "prompt_adaln_single"):
            adaln = getattr(model, name)
            adaln.emb.timestep_embedder.linear_1 = _layer(p, f"{name}.emb.timestep_embedder.linear_1")
            adaln.emb.timestep_embedder.linear_2 = _layer(p, f"{name}.emb.timestep_embedder.linear_2")
            adaln.linear = _layer(p, f"{name}.linear")
        model.scale_shift_table = p["scale_shift_table"]
        model.proj_out = _layer(p, "proj_out")
        axes = torch.meshgrid(*(torch.arange(n, device=DEVICE) for n in _grid(case)), indexing="ij")
        start = torch.stack([a.reshape(-1) for a in axes]).float()
        latent = LatentState(latent=p["x"], denoise_mask=torch.ones((1, start.shape[1], 1), device=DEVICE),
                             positions=torch.stack([start, start + 1.0], dim=-1)[None], clean_latent=p["x"])
        state.update(latent=latent, model=X0Model(model), context=p["context"])
    elif kind == "flux_double":
        from kinomlx_amd.flux2.transformer import DoubleBlock
        from kinomlx_amd.ltx2.feed_forward import FeedForward

        block = DoubleBlock(heads=case["heads"], head_dim=case["dim"] // case["heads"])
        for n in ("to_q", "to_k", "to_v", "add_q_proj", "add_k_proj", "add_v_proj", "to_add_out"):
            setattr(block.attn, n, _layer(p, f"attn.{n}"))
        block.attn.to_out = [_layer(p, "attn.to_out")]
        for n in ("norm_q", "norm_k", "norm_added_q", "norm_added_k"):
            getattr(block.attn, n).weight = p[f"attn.{n}.weight"]
        for pre in ("ff", "ff_context"):
            if case["act"] == "swiglu":
                getattr(block, pre).linear_in = _layer(p, f"{pre}.linear_in")
                getattr(block, pre).linear_out = _layer(p, f"{pre}.linear_out")
            else:
                ff = FeedForward(case["dim"], mult=case["ff"] // case["dim"])
                ff.project_in.proj = _layer(p, f"{pre}.proj_in")
                ff.project_out = _layer(p, f"{pre}.proj_out")
                setattr(block, pre, ff)
        block.fuse_projections()
        state.update(block=block, image=p["image"], text=p["text"], image_mod=p["image_mod"], text_mod=p["text_mod"],
                     tables=p["tables"])
    elif kind == "flux_single":
        from kinomlx_amd.flux2.transformer import SingleBlock

        block = SingleBlock(heads=case["heads"], head_dim=case["dim"] // case["heads"])
        block.attn.to_qkv_mlp_proj = _layer(p, "single.attn.to_qkv_mlp_proj")
        block.attn.to_out = _layer(p, "single.attn.to_out")
        block.attn.norm_q.weight = p["single.attn.norm_q.weight"]
        block.attn.norm_k.weight = p["single.attn.norm_k.weight"]
        state.update(block=block, x=p["x"], mod=p["mod"], tables=p["tables"], text=case["text"])
    else:
        from kinomlx_amd.krea2.transformer import Krea2BlockConfig, Krea2TransformerBlock

        block = Krea2TransformerBlock(Krea2BlockConfig(attention_head_dim=128, num_attention_heads=case["heads"],
                                                       num_key_value_heads=case["kv_heads"]))
        for n in ("to_q", "to_k", "to_v", "to_gate", "to_out"):
            setattr(block.attn, n, _layer(p, f"attn.{n}"))
        for n in ("gate", "up", "down"):
            setattr(block.ff, n, _layer(p, f"ff.{n}"))
        block.attn.norm_q.weight, block.attn.norm_k.weight = p["attn.norm_q.weight"], p["attn.norm_k.weight"]
        block.norm1.weight, block.norm2.weight = p["norm1.weight"], p["norm2.weight"]
        block.scale_shift_table = p["scale_shift_table"]
        block.fuse_projections()
        state.update(block=block, x=p["x"], mod=p["mod"], tables=p["tables"])
    return state


def _av_tables(case: dict) -> dict:
    """float64 (own, cross) tables of the video and the audio stream of a joint block."""
    frames, h, w = _grid(case)
    video_time = (torch.arange(frames, device=DEVICE, dtype=torch.float64) + 0.5).repeat_interleave(h * w)
    audio_time = (torch.arange(case["audio"], device=DEVICE, dtype=torch.float64) + 0.5) / 25.0
    return {
        "video": (_video_tables(_grid(case), 4096, 32), _axis_tables([video_time], (20.0,), 2048, 32)),
        "audio": (_axis_tables([audio_time], (20.0,), 2048, 32), _axis_tables([audio_time], (20.0,), 2048, 32)),
    }


SIGMAS = (0.909375, 0.725)


def run(state: dict):
    kind = state["kind"]
    if kind == "adaln":
        return state["layer"](state["timesteps"], torch.bfloat16, time_scale=1000.0)
    if kind == "attention":
        return state["layer"](state["x"], context=state["context"], mask=state["mask"], pe=state["pe"],
                              residual=state["residual"], gate=state["gate"], out_dtype=torch.float32)
    if kind == "feed_forward":
        return state["layer"](state["x"], residual=state["residual"], gate=state["gate"], out_dtype=torch.float32)
    if kind == "ltx_block":
        return state["block"](state["video"])[0].x
    if kind == "av_block":
        video, audio = state["block"](state["video"], state["audio"])
        return video.x, audio.x
    if kind == "denoise":
        from kinomlx_amd.ltx2.denoise import denoise_step

        return denoise_step(state["latent"], sigma=SIGMAS[0], sigma_next=SIGMAS[1], transformer=state["model"],
                            video_context=state["context"])[0].latent
    if kind == "flux_double":
        return state["block"](state["image"], state["text"], state["image_mod"], state["text_mod"], state["tables"])
    if kind == "flux_single":
        return state["block"](state["x"], state["mod"], state["tables"], text_tokens=state["text"])
    return state["block"](state["x"], time_modulation=state["mod"], rotary=state["tables"], attention_mask=None)


# ---- the float64 evaluation ------------------------------------------------------------------------


def _lin(p: dict, name: str, x: torch.Tensor) -> torch.Tensor:
    y = x @ p[f"{name}.weight"].double().t()
    bias = p.get(f"{name}.bias")
    return y if bias is None else y + bias.double()


def _rms(x: torch.Tensor, weight: torch.Tensor | None = None) -> torch.Tensor:
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6)
    return y if weight is None else y * weight


def _layer_norm(x: torch.Tensor) -> torch.Tensor:
    centred = x - x.mean(-1, keepdim=True)
    return centred * torch.rsqrt(centred.square().mean(-1, keepdim=True) + 1e-6)


def _gelu(x: torch.Tensor) -> torch.Tensor:
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _silu(x: torch.Tensor) -> torch.Tensor:
    return x * torch.sigmoid(x)


def _sdpa(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, heads: int, kv_heads: int | None = None,
          mask: torch.Tensor | None = None) -> torch.Tensor:
    """``(T, H D)`` flattened heads, a few thousand query rows of one head at a time."""
    dim = q.shape[-1] // heads
    group = heads // (kv_heads or heads)
    out = torch.empty_like(q)
    for h in range(heads):
        qs, g = slice(h * dim, (h + 1) * dim), h // group
        ks = slice(g * dim, (g + 1) * dim)
        kh, vh = k[:, ks].t().contiguous(), v[:, ks].contiguous()
        for start in range(0, q.shape[0], 8192):
            scores = q[start:start + 8192, qs].contiguous() @ kh
            scores *= dim ** -0.5
            if mask is not None:
                scores += mask
            out[start:start + 8192, qs] = torch.softmax(scores, dim=-1) @ vh
    return out


def _split_rope(x: torch.Tensor, tables, heads: int) -> torch.Tensor:
    cos, sin = (t.float().double()[0] for t in tables)
    half = x.view(x.shape[0], heads, 2, -1)
    a, b = half[:, :, 0], half[:, :, 1]
    return torch.stack([a * cos - b * sin, b * cos + a * sin], dim=2).flatten(1)


def _pair_rope(x: torch.Tensor, tables) -> torch.Tensor:
    """``x`` ``(T, H, Dh)``, tables ``(T, 1, Dh)``."""
    cos, sin = tables
    pairs = x.view(*x.shape[:-1], -1, 2)
    turned = torch.stack([-pairs[..., 1], pairs[..., 0]], dim=-1).view_as(x)
    return x * cos + turned * sin


def _attention64(p: dict, name: str, x, heads: int, context=None, pe=None, k_pe=None, mask=None):
    source = x if context is None else context
    q = _rms(_lin(p, f"{name}.to_q", x), p[f"{name}.q_norm.weight"].double())
    k = _rms(_lin(p, f"{name}.to_k", source), p[f"{name}.k_norm.weight"].double())
    if pe is not None:
        q = _split_rope(q, pe, heads)
        k = _split_rope(k, pe if k_pe is None else k_pe, heads)
    o = _sdpa(q, k, _lin(p, f"{name}.to_v", source), heads, mask=mask)
    gate = 2 * torch.sigmoid(_lin(p, f"{name}.to_gate_logits", x))
    return _lin(p, f"{name}.to_out", (o.view(*gate.shape, -1) * gate[..., None]).flatten(1))


def _first64(p: dict, pre: str, x, context, ada, prompt, tables, heads: int):
    """Self-attention and text cross-attention of one stream."""
    x = x + ada[2] * _attention64(p, f"{pre}attn1", _rms(x) * (1 + ada[1]) + ada[0], heads, pe=tables)
    return x + ada[8] * _attention64(p, f"{pre}attn2", _rms(x) * (1 + ada[7]) + ada[6], heads,
                                     context=context * (1 + prompt[1]) + prompt[0])


def _ff64(p: dict, pre: str, x, ada):
    h = _gelu(_lin(p, f"{pre}ff.proj_in", _rms(x) * (1 + ada[4]) + ada[3]))
    return x + ada[5] * _lin(p, f"{pre}ff.proj_out", h)


def _ltx64(p: dict, x, context, timesteps, tables, prompt_timesteps=None):
    ada = p["scale_shift_table"].double() + timesteps.double()
    prompt = p["prompt_scale_shift_table"].double()
    if prompt_timesteps is not None:
        prompt = prompt + prompt_timesteps
    return _ff64(p, "", _first64(p, "", x, context, ada, prompt, tables, 32), ada)


def _adaln64(p: dict, pre: str, linear: str, timesteps: torch.Tensor):
    freqs = torch.exp(-math.log(10000.0) * torch.arange(128, device=DEVICE, dtype=torch.float64) / 128)
    angles = timesteps.double()[:, None] * 1000.0 * freqs
    embedded = _lin(p, f"{pre}linear_2", _silu(_lin(p, f"{pre}linear_1", torch.cat([angles.cos(), angles.sin()], -1))))
    return _lin(p, linear, _silu(embedded)), embedded


def exact(case: dict, seed: int):
    p = _inputs(case, seed)
    kind = case["kind"]
    for name in _quantized_names(case):
        p[f"{name}.weight"] = _quantize(p[f"{name}.weight"], case["weights"])[3]
    if kind == "adaln":
        return _adaln64(p, "", "linear", p["timesteps"])
    if kind == "attention":
        pe = None
        heads = case["heads"]
        if not case["context"]:
            seconds = torch.arange(case["tokens"], device=DEVICE, dtype=torch.float64) / 25.0
            pe = _axis_tables([seconds], (20.0,), heads * case["head_dim"], heads)
        context = p["context"][0].double() if case["context"] else None
        mask = p["mask"].double()[0, 0] if "mask" in p else None
        y = _attention64(p, "attn", p["x"][0].double(), heads, context=context, pe=pe, mask=mask)
        return (p["residual"].double()[0] + p["gate"].double()[0] * y)[None]
    if kind == "feed_forward":
        y = _lin(p, "ff.proj_out", _gelu(_lin(p, "ff.proj_in", p["x"][0].double())))
        return (p["residual"].double()[0] + p["gate"].double()[0] * y)[None]
    if kind == "ltx_block":
        return _ltx64(p, p["x"][0].double(), p["context"][0].double(), p["timesteps"][0, 0],
                      _video_tables(_grid(case), 4096, 32))[None]
    if kind == "av_block":
        tables = _av_tables(case)
        base, ada, cross, gate = {}, {}, {}, {}
        for stream, pre in (("video", ""), ("audio", "audio_")):
            ada[stream] = p[f"{pre}scale_shift_table"].double() + p[f"{pre}timesteps"][0, 0].double()
            prompt = p[f"{pre}prompt_scale_shift_table"].double()
            base[stream] = _first64(p, pre, p[f"{pre}x"][0].double(), p[f"{pre}context"][0].double(), ada[stream],
                                    prompt, tables[stream][0], 32)
            table = p[f"scale_shift_table_a2v_ca_{stream}"].double()
            cross[stream] = table[:4] + p[f"{pre}cross_ss"][0, 0].double()
            gate[stream] = table[4] + p[f"{pre}cross_gate"][0, 0, 0].double()
        out = []
        for stream, other, name, row, pre in (("video", "audio", "audio_to_video_attn", 0, ""),
                                              ("audio", "video", "video_to_audio_attn", 2, "audio_")):
            def modulated(s):
                return _rms(base[s]) * (1 + cross[s][row]) + cross[s][row + 1]

            y = _attention64(p, name, modulated(stream), 32, context=modulated(other), pe=tables[stream][1],
                             k_pe=tables[other][1])
            out.append(_ff64(p, pre, base[stream] + gate[stream] * y, ada[stream])[None])
        return tuple(out)
    if kind == "denoise":
        sigma = torch.full((1,), SIGMAS[0], dtype=torch.float64, device=DEVICE)
        rows, embedded = _adaln64(p, "adaln_single.emb.timestep_embedder.", "adaln_single.linear", sigma)
        prompt, _ = _adaln64(p, "prompt_adaln_single.emb.timestep_embedder.", "prompt_adaln_single.linear", sigma)
        latent = p["x"][0].double()
        x = _lin(p, "patchify_proj", latent)
        tables = _video_tables(_grid(case), 4096, 32)
        for i in range(case["blocks"]):
            x = _ltx64(p[f"block{i}"], x, p["context"][0].double(), rows.view(9, 4096), tables, prompt.view(2, 4096))
        shift, scale = p["scale_shift_table"].double() + embedded
        velocity = _lin(p, "proj_out", _layer_norm(x) * (1 + scale) + shift)
        denoised = latent - SIGMAS[0] * velocity
        return (denoised + SIGMAS[1] / SIGMAS[0] * (latent - denoised))[None]
    if kind == "krea_block":
        return _krea64(p, case)[None]
    cos, sin = (t.double()[0] for t in p["tables"])
    dim, heads = case["dim"], case["heads"]

    def rows(name: str, q_norm: str, k_norm: str, x, at: slice):
        qkv = [_lin(p, f"attn.{n}", x) for n in name]
        for i, norm in enumerate((q_norm, k_norm)):
            h = _rms(qkv[i].view(x.shape[0], heads, -1), p[f"attn.{norm}.weight"].double())
            qkv[i] = _pair_rope(h, (cos[at], sin[at])).flatten(1)
        return qkv

    if kind == "flux_single":
        x = p["x"][0].double()
        shift, scale, gate = p["mod"].double()[0].chunk(3)
        fused = _lin(p, "single.attn.to_qkv_mlp_proj", _layer_norm(x) * (1 + scale) + shift)
        q, k, v, up, content = fused.split([dim, dim, dim, case["ff"], case["ff"]], dim=-1)
        q, k = (_pair_rope(_rms(t.reshape(x.shape[0], heads, -1), p[f"single.attn.{n}.weight"].double()),
                           (cos, sin)).flatten(1) for t, n in ((q, "norm_q"), (k, "norm_k")))
        joined = torch.cat([_sdpa(q, k, v.contiguous(), heads), _silu(up) * content], dim=-1)
        return (x + gate * _lin(p, "single.attn.to_out", joined))[None]
    text_rows = case["text"]
    image, text = p["image"][0].double(), p["text"][0].double()
    im, tm = p["image_mod"].double()[0].chunk(6), p["text_mod"].double()[0].chunk(6)
    ti = rows(("add_q_proj", "add_k_proj", "add_v_proj"), "norm_added_q", "norm_added_k",
              _layer_norm(text) * (1 + tm[1]) + tm[0], slice(0, text_rows))
    ii = rows(("to_q", "to_k", "to_v"), "norm_q", "norm_k", _layer_norm(image) * (1 + im[1]) + im[0],
              slice(text_rows, None))
    o = _sdpa(*(torch.cat(pair) for pair in zip(ti, ii)), heads)
    image = image + im[2] * _lin(p, "attn.to_out", o[text_rows:])
    text = text + tm[2] * _lin(p, "attn.to_add_out", o[:text_rows])

    def feed_forward(pre: str, x):
        if case["act"] == "swiglu":
            up, content = _lin(p, f"{pre}.linear_in", x).chunk(2, dim=-1)
            return _lin(p, f"{pre}.linear_out", _silu(up) * content)
        return _lin(p, f"{pre}.proj_out", _gelu(_lin(p, f"{pre}.proj_in", x)))

    image = image + im[5] * feed_forward("ff", _layer_norm(image) * (1 + im[4]) + im[3])
    text = text + tm[5] * feed_forward("ff_context", _layer_norm(text) * (1 + tm[4]) + tm[3])
    return image[None], text[None]


def _krea64(p: dict, case: dict) -> torch.Tensor:
    heads, kv = case["heads"], case["kv_heads"]
    x = p["x"][0].double()
    mod = p["mod"].double().view(6, -1) + p["scale_shift_table"].double()
    tables = tuple(t.double()[0][:, None] for t in p["tables"])
    h = _rms(x, p["norm1.weight"].double() + 1) * (1 + mod[0]) + mod[1]
    q, k = (_pair_rope(_rms(_lin(p, f"attn.to_{n}", h).view(x.shape[0], -1, 128),
                            p[f"attn.norm_{n}.weight"].double() + 1), tables).flatten(1) for n in ("q", "k"))
    o = _sdpa(q, k, _lin(p, "attn.to_v", h), heads, kv)
    x = x + mod[2] * _lin(p, "attn.to_out", o * torch.sigmoid(_lin(p, "attn.to_gate", h)))
    h = _rms(x, p["norm2.weight"].double() + 1) * (1 + mod[3]) + mod[4]
    return x + mod[5] * _lin(p, "ff.down", _silu(_lin(p, "ff.gate", h)) * _lin(p, "ff.up", h))


# ---- work and tolerance ----------------------------------------------------------------------------


def _weight_bytes(elements: float, weights: str) -> float:
    per_element = {"bf16": 2.0, "fp16": 2.0, "int4": 0.5 + 4 / 64, "int8": 1.0 + 4 / 64, "mxfp8": 1.0 + 1 / 32}
    return elements * per_element[weights]


def _ltx_work(t: int, tc: int, d: int, heads: int, weights: str = "bf16") -> tuple[float, float]:
    """(bytes, flops) of one stream's block without its A/V attention: weights, stream in and out,
    context and RoPE tables."""
    elements = 4 * d * d + 4 * d * d + 2 * heads * d + 8 * d * d
    flops = 2.0 * t * d * (4 * d + 2 * d + 2 * heads) + 2.0 * tc * d * 2 * d + 2.0 * 2 * t * d * 4 * d
    flops += 4.0 * d * t * (t + tc)
    return _weight_bytes(elements, weights) + 2 * t * d * 2 + tc * d * 2 + 2 * t * (d // 2) * 4, flops


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "adaln":
        d, n = case["dim"], case["steps"]
        elements = 256 * d + d * d + case["rows"] * d * d
        return {"bytes": 2.0 * elements + n * (4 + 2 * d * (1 + case["rows"])), "flops": 2.0 * n * elements}
    if kind == "attention":
        d, t, tc = case["heads"] * case["head_dim"], case["tokens"], case["context"]
        keys = tc or t
        flops = 2.0 * t * d * (2 * d + case["heads"]) + 2.0 * keys * d * 2 * d + 4.0 * d * t * keys
        tables = 0 if tc else 2 * t * (d // 2) * 4
        weights = 4 * d * d + case["heads"] * d
        return {"bytes": 2.0 * weights + t * d * (2 + 4 + 4) + tc * d * 2 + tables, "flops": flops}
    if kind == "feed_forward":
        d, t = case["dim"], case["tokens"]
        return {"bytes": _weight_bytes(8 * d * d, case["weights"]) + t * d * (2 + 4 + 4), "flops": 16.0 * t * d * d}
    if kind == "ltx_block":
        b, f = _ltx_work(_tokens(_grid(case)), case["text"], 4096, 32, case["weights"])
        return {"bytes": b, "flops": f}
    if kind == "av_block":
        t, a = _tokens(_grid(case)), case["audio"]
        bv, fv = _ltx_work(t, case["text"], 4096, 32)
        ba, fa = _ltx_work(a, case["text"], 2048, 32)
        cross = 2.0 * 2048 * ((t + a) * 4096 * 2 + (a + t) * 2048 * 2) + 2 * 4.0 * 2048 * t * a
        elements = 2 * 2048 * (4096 + 2048 + 2048 + 4096)
        return {"bytes": bv + ba + 2.0 * elements, "flops": fv + fa + cross}
    if kind == "denoise":
        t = _tokens(_grid(case))
        b, f = _ltx_work(t, case["text"], 4096, 32)
        producers = 2 * (256 * 4096 + 4096 * 4096) + 11 * 4096 * 4096
        ends = 2 * 128 * 4096
        return {"bytes": case["blocks"] * (b - 2 * t * 4096 * 2) + 2.0 * (producers + ends) + 2 * t * 128 * 2,
                "flops": case["blocks"] * f + 2.0 * producers + 2.0 * t * ends}
    if kind == "krea_block":
        t, d, kv, ff = case["tokens"], case["heads"] * 128, case["kv_heads"] * 128, case["ff"]
        elements = 3 * d * d + 2 * d * kv + 3 * d * ff
        return {"bytes": 2.0 * elements + 2 * t * d * 2 + 2 * t * 128 * 4,
                "flops": 2.0 * t * elements + 4.0 * t * t * d}
    d, ff = case["dim"], case["ff"]
    ti, tt = _tokens(_grid(case)), case["text"]
    t = ti + tt
    per_stream = 4 * d * d + (3 if case.get("act") != "gelu" else 2) * d * ff
    if kind == "flux_single":
        elements = weights = per_stream
    else:
        elements, weights = per_stream, 2 * per_stream
    return {"bytes": 2.0 * weights + 2 * t * d * 2 + 2 * t * (d // case["heads"]) * 4,
            "flops": 2.0 * t * elements + 4.0 * t * t * d}


def tolerance(case: dict) -> dict:
    """About four times the error against ``exact`` that was measured over seeds and sizes: the
    roundings of the 16-bit values that every implementation stores between the products (8 bits of
    bf16, 11 of fp16), next to the float32 residual where a layer returns one."""
    half = case.get("dtype", case.get("weights")) == "fp16"
    if case["kind"] == "attention":
        return {"rel": 4e-4 if half else 2.5e-3}
    if case["kind"] == "feed_forward":
        return {"rel": 1e-3 if half else 6e-3}
    if case["kind"] == "ltx_block":
        return {"rel": 2.5e-3 if half else 1.2e-2}
    return {"rel": 1.6e-2}
