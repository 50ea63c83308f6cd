"""The work that users of this framework have it do, as timed cases.

Every case goes through public entry points: the engine's whole call (``HipIris.__call__``), one
trunk block (``HipIris.block_forward``), the text adapter (``HipIris.encode_text``) and the single
layers of ``iris_mi355x.kernels`` (a SwiGLU MLP, joint attention, a modulated norm, the shared
adaLN core). Widths are Iris-3B's (2560 wide, 20 query and 5 K/V heads of 128, 16-pixel patches, a
pixel stage of 16 channels with 10 heads); whole calls run a model of full width and reduced depth
that keeps the full model's proportions, so that weights can be drawn quickly. Sizes span what
the model is run at: images from 256 x 256 to one megapixel, square and oblong, prompts of a few
to 300 tokens, batches of one (Turbo) and of two (classifier-free guidance).

Weights and inputs are random with the distributions of the parity tests; weight matrices are
rounded to BF16, the precision that checkpoints are served at, so the 64-bit results of ``exact``
are those of the very weights the engine multiplies.
"""

from __future__ import annotations

import math
import sys
from dataclasses import replace
from pathlib import Path

import torch
import torch.nn.functional as F

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "iris-3b-metal_amd"))

from iris_mi355x import kernels as K  # noqa: E402
from iris_mi355x.config import IRIS_3B  # noqa: E402
from iris_mi355x.engine import HipIris  # noqa: E402
from iris_mi355x.weights import synthetic_state_dict  # noqa: E402

D, HEADS, KV_HEADS, HD = 2560, 20, 5, 128
HIDDEN = IRIS_3B.mlp_hidden
HIDDEN_PAD = (HIDDEN + 63) // 64 * 64
EPS = IRIS_3B.norm_eps
PATCH = 16
LAYERS, LAYER_HEADS = IRIS_3B.text_lap_num_layers, IRIS_3B.text_lap_num_heads
LAYER_HIDDEN = int(D * IRIS_3B.text_lap_mlp_ratio)
PIXEL_D, PIXEL_HEADS = IRIS_3B.pixel.attn_hidden_size, IRIS_3B.pixel.num_heads

# one pixel block per six trunk blocks, one dual-stream block per two single-stream ones: 4, 8 and 16
# in the full model
FORWARD = replace(IRIS_3B, depth=6, dual_depth=2, pixel=replace(IRIS_3B.pixel, depth=1))
BLOCKS = replace(IRIS_3B, depth=2, dual_depth=1, pixel=replace(IRIS_3B.pixel, depth=1))  # block 0 dual, 1 single


def listed() -> list[dict]:
    return [
        # one denoise step of the smallest image, with a short prompt: a preview
        {"name": "forward-256", "kind": "forward", "batch": 1, "height": 256, "width": 256, "text": 77},
        # the step that users run most: one megapixel, one image, a full prompt
        {"name": "forward-1024", "kind": "forward", "batch": 1, "height": 1024, "width": 1024, "text": 256},
        # a dual-stream block under guidance (conditional and unconditional rows) on a small oblong image
        {"name": "dual-192x320-cfg", "kind": "dual", "batch": 2, "height": 192, "width": 320, "text": 77},
        # a dual-stream block at one megapixel with the longest prompt
        {"name": "dual-1024", "kind": "dual", "batch": 1, "height": 1024, "width": 1024, "text": 300},
        # a single-stream block at a middle size: a restoration tile, a draft
        {"name": "single-512", "kind": "single", "batch": 1, "height": 512, "width": 512, "text": 256},
        # a single-stream block of a guided portrait image: ragged row counts, two batch items
        {"name": "single-832x1216-cfg", "kind": "single", "batch": 2, "height": 832, "width": 1216, "text": 300},
        # a prompt through the text adapter, padded to the full length as the tokenizer does
        {"name": "text-300", "kind": "text", "batch": 1, "text": 300},
        # a short prompt and its negative
        {"name": "text-77-cfg", "kind": "text", "batch": 2, "text": 77},
        # the feed-forward layer over the rows of a small image and its prompt
        {"name": "mlp-333", "kind": "mlp", "rows": 333},
        # the pixel stage's attention at one megapixel
        {"name": "attention-pixel-4096", "kind": "attention", "batch": 1, "tokens": 4096, "heads": PIXEL_HEADS,
         "kv_heads": PIXEL_HEADS, "gate": False},
        # a block's input norm at one megapixel
        {"name": "norm-4352", "kind": "norm", "batch": 1, "tokens": 4352, "dtype": "float32"},
        # the shared adaLN core with every block's bias, once per step and image
        {"name": "modulation-1", "kind": "modulation", "batch": 1, "blocks": IRIS_3B.depth},
    ]


def _log_uniform(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _image(rng, patches: int) -> tuple[int, int]:
    """Height and width of an image of at most ``patches`` patches, down to 12 x 12 of them."""
    area = _log_uniform(rng, 192, patches)
    aspect = math.exp(rng.uniform(math.log(0.5), math.log(2.0)))
    rows = max(12, min(64, round(math.sqrt(area * aspect))))
    cols = max(12, min(64, area // rows))
    return rows * PATCH, cols * PATCH


def draw(rng) -> dict:
    kind = rng.choice(["forward", "dual", "single", "single", "text", "mlp", "attention", "norm", "modulation"])
    if kind in ("forward", "dual", "single"):
        batch = rng.choice([1, 1, 2])
        height, width = _image(rng, 4096 if batch == 1 or kind != "forward" else 1900)
        return {"kind": kind, "batch": batch, "height": height, "width": width, "text": _log_uniform(rng, 16, 256)}
    if kind == "text":
        return {"kind": kind, "batch": rng.choice([1, 2]), "text": _log_uniform(rng, 16, 300)}
    if kind == "mlp":
        return {"kind": kind, "rows": _log_uniform(rng, 64, 8704)}
    if kind == "attention":
        pixel = rng.random() < 0.4
        return {"kind": kind, "batch": rng.choice([1, 2]), "tokens": _log_uniform(rng, 208, 4352),
                "heads": PIXEL_HEADS if pixel else HEADS, "kv_heads": PIXEL_HEADS if pixel else KV_HEADS,
                "gate": not pixel}
    if kind == "norm":
        return {"kind": kind, "batch": rng.choice([1, 2]), "tokens": _log_uniform(rng, 208, 4352),
                "dtype": rng.choice(["float32", "bfloat16"])}
    return {"kind": "modulation", "batch": rng.choice([1, 2, 3, 4]), "blocks": rng.randint(2, 32)}


# -- inputs ---------------------------------------------------------------------------------
def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(gen, *shape, scale: float = 1.0, dtype=torch.float32) -> torch.Tensor:
    return (scale * torch.randn(*shape, generator=gen, device="cuda")).to(dtype)


def _weights(cfg, seed: int) -> dict[str, torch.Tensor]:
    state = synthetic_state_dict(cfg, seed=seed + 1, device="cuda")
    for name, value in state.items():
        if name.endswith(".weight") and value.dim() >= 2:
            state[name] = value.to(torch.bfloat16).float()
    return state


def _inputs(case: dict, seed: int) -> dict:
    """The tensors of one call, drawn in a fixed order."""
    gen = _generator(seed)
    kind = case["kind"]
    bf16 = torch.bfloat16
    if kind == "forward":
        return {"x": _randn(gen, case["batch"], 3, case["height"], case["width"]),
                "t": 50.0 + 950.0 * torch.rand(case["batch"], generator=gen, device="cuda"),
                "text": _randn(gen, case["batch"], case["text"], D)}
    if kind in ("dual", "single"):
        tokens = (case["height"] // PATCH) * (case["width"] // PATCH)
        return {"x": _randn(gen, case["batch"], tokens, D),
                "t": 50.0 + 950.0 * torch.rand(case["batch"], generator=gen, device="cuda"),
                "text": _randn(gen, case["batch"], case["text"], D)}
    if kind == "text":
        mask = torch.zeros(case["batch"], case["text"], dtype=torch.int64, device="cuda")
        for b in range(case["batch"]):  # about two thirds of the tokens are the prompt's, the rest padding
            mask[b, : max(1, case["text"] * (4 + seed % 3 - b) // 6)] = 1
        return {"states": _randn(gen, case["batch"], case["text"], LAYERS, D), "mask": mask}
    if kind == "mlp":
        return {"x": _randn(gen, case["rows"], D, dtype=bf16),
                "w1": _randn(gen, HIDDEN, D, scale=0.02, dtype=bf16),
                "w3": _randn(gen, HIDDEN, D, scale=0.02, dtype=bf16),
                "w2": _randn(gen, D, HIDDEN, scale=0.02, dtype=bf16)}
    if kind == "attention":
        b, n, h, hkv = case["batch"], case["tokens"], case["heads"], case["kv_heads"]
        return {"q": _randn(gen, b, h, n, HD, dtype=bf16), "k": _randn(gen, b, hkv, n, HD, dtype=bf16),
                "v": _randn(gen, b, hkv, n, HD, dtype=bf16), "gate": _randn(gen, b * n, h * HD, dtype=bf16)}
    if kind == "norm":
        return {"x": _randn(gen, case["batch"], case["tokens"], D, dtype=getattr(torch, case["dtype"])),
                "weight": 1 + _randn(gen, D, scale=0.02), "mods": _randn(gen, case["batch"], 1, 6 * D, scale=0.1)}
    return {"weight": _randn(gen, 6 * D, D, scale=0.02, dtype=bf16), "x": _randn(gen, case["batch"], D),
            "bias": _randn(gen, 6 * D, scale=0.02), "extra": _randn(gen, case["blocks"], 6 * D, scale=0.02)}


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    state = {"case": case, **_inputs(case, seed)}
    if kind == "forward":
        state["engine"] = HipIris(FORWARD, _weights(FORWARD, seed))
        state["out"] = torch.empty_like(state["x"])
    elif kind in ("dual", "single", "text"):
        state["engine"] = HipIris(BLOCKS, _weights(BLOCKS, seed))
    elif kind == "mlp":
        state["w13"] = K.pack_swiglu(state.pop("w1"), state.pop("w3"), HIDDEN_PAD)
        state["w2"] = F.pad(state["w2"], (0, HIDDEN_PAD - HIDDEN)).contiguous()
    elif kind == "attention":
        b, n, h, hkv = case["batch"], case["tokens"], case["heads"], case["kv_heads"]
        pad = (n + 63) // 64 * 64 - n
        state["q"], state["k"] = (F.pad(state[key], (0, 0, 0, pad)) for key in ("q", "k"))
        v = F.pad(state.pop("v"), (0, 0, 0, pad))
        state["vt"] = v[:, :, K.vt_positions(n + pad).to(v.device)].transpose(2, 3).contiguous()
        state["out"] = torch.empty(b * n, h * HD, device="cuda", dtype=torch.bfloat16)
    elif kind == "modulation":
        state["out"] = torch.empty(case["blocks"], case["batch"], 6 * D, device="cuda")
    return state


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "forward":
        return state["engine"](state["x"], state["t"], state["text"], out=state["out"])
    if kind in ("dual", "single"):
        grid = (case["height"] // PATCH, case["width"] // PATCH)
        return state["engine"].block_forward(0 if kind == "dual" else 1, state["x"], state["text"], state["t"], grid)
    if kind == "text":
        return state["engine"].encode_text(state["states"], state["mask"])
    if kind == "mlp":
        return K.linear(K.linear(state["x"], state["w13"], swiglu=True), state["w2"])
    if kind == "attention":
        K.flash_attention(state["q"], state["k"], state["vt"], case["tokens"], None, state["out"],
                          gate1=state["gate"] if case["gate"] else None)
        return state["out"]
    if kind == "norm":
        mods = state["mods"]
        return K.rms_norm_modulate(state["x"], state["weight"], mods[..., :D], mods[..., D:2 * D], EPS, torch.bfloat16)
    return K.gemv(state["weight"], state["x"], state["bias"], state["out"], extra_bias=state["extra"], in_silu=True)


# -- what a pass cannot do without ---------------------------------------------------------------
def _trunk(rows_by_weights: list[int], batch: int, tokens: int) -> tuple[float, float]:
    """(weight bytes, FLOPs) of a trunk block whose row groups each have projection weights of their own."""
    weights = (HEADS + 2 * KV_HEADS) * HD * D + 2 * D * D + 3 * HIDDEN * D
    flops = sum(2.0 * rows * weights for rows in rows_by_weights) + 4.0 * batch * tokens * tokens * HEADS * HD
    return 2.0 * weights * len(rows_by_weights), flops


def work(case: dict) -> dict:
    kind = case["kind"]
    b = case.get("batch", 1)
    core_bytes = 2.0 * 2 * 6 * D * D + 2.0 * (256 * D + D * D)
    if kind in ("forward", "dual", "single"):
        patches = (case["height"] // PATCH) * (case["width"] // PATCH)
        text = case["text"]
        n = patches + text
        dual = _trunk([b * patches, b * text], b, n)
        single = _trunk([b * n], b, n)
    if kind == "forward":
        pixels = 256 * 16
        pixel_weights = 4 * pixels * D + 2 * pixels * PIXEL_D + 4 * PIXEL_D * PIXEL_D
        pixel = (2.0 * b * patches * pixel_weights + 4.0 * b * patches * patches * PIXEL_D
                 + 2.0 * b * patches * 256 * 2 * 16 * 64)
        nbytes = (2 * dual[0] + 4 * single[0] + 2.0 * (pixel_weights + 768 * D) + core_bytes
                  + 4.0 * b * (2 * 3 * case["height"] * case["width"] + text * D))
        flops = 2 * dual[1] + 4 * single[1] + pixel + 2.0 * b * patches * 768 * D
        return {"bytes": nbytes, "flops": flops}
    if kind in ("dual", "single"):
        weight_bytes, flops = dual if kind == "dual" else single
        return {"bytes": weight_bytes + core_bytes + 2 * 4.0 * b * n * D, "flops": flops}
    if kind == "text":
        rows = b * case["text"]
        layer = 4 * D * D + 2 * LAYER_HIDDEN * D
        refiner = 4 * D * D + 3 * HIDDEN * D
        flops = (2 * (2.0 * rows * LAYERS * layer + 4.0 * rows * LAYERS * LAYERS * D)
                 + 2.0 * rows * D * D + 2 * (2.0 * rows * refiner + 4.0 * b * case["text"] ** 2 * D))
        return {"bytes": 2.0 * (2 * layer + D * D + 2 * refiner) + 4.0 * rows * D * (LAYERS + 1), "flops": flops}
    if kind == "mlp":
        return {"bytes": 2.0 * (3 * HIDDEN * D + 2 * case["rows"] * D), "flops": 2.0 * case["rows"] * 3 * HIDDEN * D}
    if kind == "attention":
        n, h, hkv = case["tokens"], case["heads"], case["kv_heads"]
        rows = 2 * h + 2 * hkv + (h if case["gate"] else 0)
        return {"bytes": 2.0 * b * n * HD * rows, "flops": 4.0 * b * n * n * h * HD}
    if kind == "norm":
        n = b * case["tokens"]
        return {"bytes": n * D * (2.0 + (4 if case["dtype"] == "float32" else 2)) + 4.0 * D * (1 + 2 * b),
                "flops": 6.0 * n * D}
    return {"bytes": 2.0 * 6 * D * D + 4.0 * (b * D + 6 * D * (1 + case["blocks"] * (1 + b))),
            "flops": 2.0 * b * 6 * D * D}


def tolerance(case: dict) -> dict:
    """Four times the measured distance from ``exact`` (BF16 operands with FP32 sums; a block's distance
    is small because its FP32 residual carries most of its output; the modulation is all FP32 sums)."""
    return {"rel": {"forward": 1e-2, "dual": 1.6e-3, "single": 1.6e-3, "text": 2.4e-2, "mlp": 1e-2, "attention": 1e-2,
                    "norm": 7e-3, "modulation": 1e-6}[case["kind"]]}


# -- the same in 64 bits -----------------------------------------------------------------------
def _linear(p: dict, name: str, x: torch.Tensor) -> torch.Tensor:
    bias = p.get(f"{name}.bias")
    return F.linear(x, p[f"{name}.weight"].double(), None if bias is None else bias.double())


def _rms(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * weight.double()


def _swiglu(p: dict, name: str, x: torch.Tensor) -> torch.Tensor:
    return _linear(p, f"{name}.w2", F.silu(_linear(p, f"{name}.w1", x)) * _linear(p, f"{name}.w3", x))


def _softmax_attention(q, k, v, keep=None) -> torch.Tensor:
    """``[B, N, heads, d]`` inputs with grouped K/V heads, one batch item and head at a time."""
    out = torch.empty(*q.shape[:3], v.shape[3], dtype=q.dtype, device=q.device)
    group = q.shape[2] // k.shape[2]
    for b in range(q.shape[0]):
        for h in range(q.shape[2]):
            s = q[b, :, h] @ k[b, :, h // group].T / math.sqrt(q.shape[3])
            if keep is not None:
                s = s.masked_fill(~keep[b], -math.inf)
            out[b, :, h] = torch.softmax(s, -1) @ v[b, :, h // group]
    return out


def _angles_1d(tokens: int) -> torch.Tensor:
    freqs = IRIS_3B.text_rope_theta ** (-torch.arange(0, HD, 2, dtype=torch.float64, device="cuda") / HD)
    return torch.outer(torch.arange(tokens, dtype=torch.float64, device="cuda"), freqs)


def _angles_2d(rows: int, cols: int) -> torch.Tensor:
    freqs = IRIS_3B.rope_theta ** (-torch.arange(0, HD, 4, dtype=torch.float64, device="cuda") / HD)
    step = IRIS_3B.rope_scale / max(max(rows, cols) - 1, 1)
    y, x = torch.meshgrid(torch.arange(rows, device="cuda"), torch.arange(cols, device="cuda"), indexing="ij")
    return torch.stack([x.reshape(-1, 1) * step * freqs, y.reshape(-1, 1) * step * freqs], -1).flatten(1)


def _rotate(x: torch.Tensor, angles: torch.Tensor) -> torch.Tensor:
    """Adjacent pairs of ``[B, N, heads, d]`` turned by ``angles`` ``[N, d / 2]``."""
    cos, sin = angles.cos()[:, None], angles.sin()[:, None]
    a, b = x[..., ::2], x[..., 1::2]
    return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)


def _time(p: dict, t: torch.Tensor) -> torch.Tensor:
    k = torch.arange(128, dtype=torch.float64, device="cuda")
    phase = torch.outer(t.double(), torch.exp(-math.log(IRIS_3B.timestep_max_period) * k / 128))
    h = _linear(p, "t_embedder.mlp.0", torch.cat([phase.cos(), phase.sin()], -1))
    return _linear(p, "t_embedder.mlp.2", F.silu(h))[:, None]


def _mods(p: dict, stream: str, name: str, temb: torch.Tensor) -> list[torch.Tensor]:
    mods = _linear(p, f"modulation_cores.adaln_{stream}", F.silu(temb)) + p[f"{name}.bias"].double()
    return list(mods.chunk(6, -1))


def _qkv(p: dict, prefix: str, suffix: str, h: torch.Tensor, angles: torch.Tensor):
    q, k, v = (_linear(p, f"{prefix}{n}_proj{suffix}", h).unflatten(-1, (-1, HD)) for n in "qkv")
    q, k = (_rms(a, p[f"{prefix}{n}_norm{suffix}.weight"]) for n, a in (("q", q), ("k", k)))
    return _rotate(q, angles), _rotate(k, angles), v


def _tail(p, x, attn, h, mods, gate, proj, post, norm2, mlp, mlp_post):
    """The rest of a block for one stream, from its rows of the attention output on."""
    attn = attn.flatten(-2) * torch.sigmoid(_linear(p, gate, h))
    x = x + mods[2] * _rms(_linear(p, proj, attn), p[f"{post}.weight"])
    h = _rms(x, p[f"{norm2}.weight"]) * (1 + mods[4]) + mods[3]
    return x + mods[5] * _rms(_swiglu(p, mlp, h), p[f"{mlp_post}.weight"])


def _block(p: dict, index: int, dual: bool, x, text, temb, angles_text, angles_image):
    b, n_text = f"blocks.{index}", text.shape[1]
    if dual:
        streams = []
        for st, rows, angles, core in (("y", text, angles_text, "txt"), ("x", x, angles_image, "img")):
            mods = _mods(p, core, f"{b}.adaln_{core}", temb)
            h = _rms(rows, p[f"{b}.norm_{st}1.weight"]) * (1 + mods[1]) + mods[0]
            streams.append((st, rows, mods, h, _qkv(p, f"{b}.attn.", f"_{st}", h, angles)))
        attn = _softmax_attention(*(torch.cat([s[4][i] for s in streams], 1) for i in range(3)))
        out = [_tail(p, rows, a, h, mods, f"{b}.attn_gate_{st}", f"{b}.attn.proj_{st}", f"{b}.attn_post_norm_{st}",
                     f"{b}.norm_{st}2", f"{b}.mlp_{st}", f"{b}.mlp_post_norm_{st}")
               for (st, rows, mods, h, _), a in zip(streams, (attn[:, :n_text], attn[:, n_text:]))]
        return out[1], out[0]
    rows = torch.cat([text, x], 1)
    mods = _mods(p, "img", f"{b}.adaln", temb)
    h = _rms(rows, p[f"{b}.norm1.weight"]) * (1 + mods[1]) + mods[0]
    attn = _softmax_attention(*_qkv(p, f"{b}.", "", h, torch.cat([angles_text, angles_image])))
    rows = _tail(p, rows, attn, h, mods, f"{b}.attn_gate", f"{b}.attn_proj", f"{b}.attn_post_norm", f"{b}.norm2",
                 f"{b}.mlp", f"{b}.mlp_post_norm")
    return rows[:, n_text:], rows[:, :n_text]


def _self_qkv(p: dict, name: str, x, heads: int, angles=None):
    q, k, v = _linear(p, f"{name}.qkv", x).unflatten(-1, (3, heads, -1)).unbind(-3)
    if f"{name}.q_norm.weight" in p:
        q, k = _rms(q, p[f"{name}.q_norm.weight"]), _rms(k, p[f"{name}.k_norm.weight"])
    if angles is not None:
        q, k = _rotate(q, angles), _rotate(k, angles)
    return q, k, v


def _pixel_positions(height: int, width: int) -> torch.Tensor:
    omega = 10000.0 ** (-torch.arange(4, dtype=torch.float64, device="cuda") / 4)
    x, y = (torch.outer(torch.arange(n, dtype=torch.float64, device="cuda"), omega) for n in (width, height))
    x, y = (torch.cat([a.sin(), a.cos()], -1) for a in (x, y))
    return torch.cat([x[None].expand(height, -1, -1), y[:, None].expand(-1, width, -1)], -1)


def _exact_forward(p: dict, cfg, inputs: dict) -> torch.Tensor:
    x, text = inputs["x"].double(), inputs["text"].double()
    batch, _, height, width = x.shape
    rows, cols = height // PATCH, width // PATCH
    temb = _time(p, inputs["t"])
    angles_text, angles_image = _angles_1d(text.shape[1]), _angles_2d(rows, cols)
    patches = x.unflatten(2, (rows, PATCH)).unflatten(4, (cols, PATCH)).permute(0, 2, 4, 1, 3, 5)
    s = _linear(p, "s_embedder.proj", patches.reshape(batch, rows * cols, -1))
    for i in range(cfg.depth):
        s, text = _block(p, i, i < cfg.dual_depth, s, text, temb, angles_text, angles_image)
    cond = F.silu(temb + s)
    pixels = _linear(p, "pixel_embedder.proj", x.permute(0, 2, 3, 1)) + _pixel_positions(height, width)
    pixels = pixels.unflatten(1, (rows, PATCH)).unflatten(3, (cols, PATCH)).permute(0, 1, 3, 2, 4, 5)
    pixels = pixels.reshape(batch, rows * cols, PATCH * PATCH, -1)
    for i in range(cfg.pixel.depth):
        b = f"pixel_blocks.{i}"
        scale1, shift1, scale2, shift2 = _linear(p, f"{b}.adaln", cond).unflatten(-1, (PATCH * PATCH, 4, -1)).unbind(-2)
        h = _linear(p, f"{b}.compress", _rms(pixels, p[f"{b}.norm1.weight"]).flatten(2))
        q, k, v = _self_qkv(p, f"{b}.attn", h, PIXEL_HEADS, angles_image)
        h = _linear(p, f"{b}.attn.proj", _softmax_attention(q, k, v).flatten(2))
        pixels = pixels + _linear(p, f"{b}.expand", h).view_as(pixels) * (1 + scale1) + shift1
        h = F.gelu(_linear(p, f"{b}.mlp.fc1", _rms(pixels, p[f"{b}.norm2.weight"])))
        pixels = pixels + _linear(p, f"{b}.mlp.fc2", h) * (1 + scale2) + shift2
    v = _linear(p, "final_layer.linear", _rms(pixels, p["final_layer.norm.weight"]))
    return v.unflatten(1, (rows, cols)).unflatten(3, (PATCH, PATCH)).permute(0, 5, 1, 3, 2, 4).reshape(x.shape)


def _exact_text(p: dict, inputs: dict) -> torch.Tensor:
    states, mask = inputs["states"].double(), inputs["mask"].bool()
    batch, n = mask.shape
    h = states.flatten(0, 1)
    for i in range(2):
        b = f"y_embedder.layer_blocks.{i}"
        q, k, v = _self_qkv(p, f"{b}.attn", _rms(h, p[f"{b}.norm1.weight"]), LAYER_HEADS)
        q, k, v = (a.transpose(1, 2) for a in (q, k, v))
        a = torch.softmax(q @ k.transpose(2, 3) / math.sqrt(q.shape[-1]), -1) @ v
        h = h + _linear(p, f"{b}.attn.proj", a.transpose(1, 2).flatten(2))
        m = F.silu(_linear(p, f"{b}.mlp.0", _rms(h, p[f"{b}.norm2.weight"])))
        h = h + _linear(p, f"{b}.mlp.2", m)
    y = _linear(p, "y_embedder.layer_pool", h.transpose(1, 2)).squeeze(-1).view(batch, n, -1)
    y = _linear(p, "y_embedder.refiner.proj", y)
    keep = mask[:, None, :] | torch.eye(n, dtype=torch.bool, device="cuda")
    for i in range(2):
        b = f"y_embedder.refiner.blocks.{i}"
        q, k, v = _self_qkv(p, f"{b}.attn", _rms(y, p[f"{b}.norm1.weight"]), HEADS)
        y = y + _linear(p, f"{b}.attn.proj", _softmax_attention(q, k, v, keep).flatten(2))
        y = y + _swiglu(p, f"{b}.mlp", _rms(y, p[f"{b}.norm2.weight"]))
    return _rms(y, p["y_embedder.refiner.norm.weight"]) + p["y_pos_embedding"][:, :n].double()


@torch.no_grad()
def exact(case: dict, seed: int):
    kind = case["kind"]
    inputs = _inputs(case, seed)
    if kind == "forward":
        return _exact_forward(_weights(FORWARD, seed), FORWARD, inputs)
    if kind in ("dual", "single"):
        p = _weights(BLOCKS, seed)
        rows, cols = case["height"] // PATCH, case["width"] // PATCH
        return _block(p, 0 if kind == "dual" else 1, kind == "dual", inputs["x"].double(), inputs["text"].double(),
                      _time(p, inputs["t"]), _angles_1d(case["text"]), _angles_2d(rows, cols))
    if kind == "text":
        return _exact_text(_weights(BLOCKS, seed), inputs)
    if kind == "mlp":
        p = {f"mlp.{k}.weight": inputs[k] for k in ("w1", "w2", "w3")}
        return _swiglu(p, "mlp", inputs["x"].double())
    if kind == "attention":
        q, k, v = (inputs[n].double().transpose(1, 2) for n in "qkv")
        out = _softmax_attention(q, k, v).flatten(2).flatten(0, 1)
        return out * torch.sigmoid(inputs["gate"].double()) if case["gate"] else out
    if kind == "norm":
        shift, scale = inputs["mods"].double()[..., :2 * D].chunk(2, -1)
        return _rms(inputs["x"].double(), inputs["weight"]) * (1 + scale) + shift
    x = F.linear(F.silu(inputs["x"].double()), inputs["weight"].double(), inputs["bias"].double())
    return x + inputs["extra"].double()[:, None]
