"""The work a program gives this library, as measured cases.

A diffusion transformer on 8-bit weights is, call by call: the modulation product on one row, the text
stream's products on tens to hundreds of rows, the image stream's on thousands, in each of the weight
formats that are published (int8 or fp8 per output channel, convrot int8 on quantized activations, GGUF
Q8_0 block scales), on packed weights or on a map's [K, N] codes in place, and the whole block around
them. `listed` holds one case of each kind at the sizes of this library's workloads; `draw` spreads the
rows, widths, types and options over the ranges those stand for.
"""
from __future__ import annotations

import math

import torch

import siliconed_amd as sq
from siliconed_amd.dit_block import DiTBlock

# The multiply-adds of the largest listed product (4096 x 3840 x 20480): no drawn product has more.
MOST_MACS = 4096 * 3840 * 20480
GLU = ("silu_glu", "situ_glu")


def listed():
    return [
        # The adaptive-norm modulation of a block: one timestep embedding, six vectors of 3072, fp32 out.
        {"name": "modulation_row", "kind": "linear", "m": 1, "k": 3072, "n": 18432, "weight": "int8",
         "epilogue": "none", "out": "f32"},
        # A prompt's tokens through an attention output projection: few rows, a square weight.
        {"name": "text_out_int8", "kind": "linear", "m": 77, "k": 3072, "n": 3072, "weight": "int8",
         "epilogue": "none", "out": "bf16"},
        # A longer, ragged prompt through the fused gate and up projection of an fp8 checkpoint.
        {"name": "text_gate_up_fp8", "kind": "linear", "m": 333, "k": 3840, "n": 20480, "weight": "fp8",
         "epilogue": "silu_glu", "out": "bf16"},
        # A prompt's tokens through an up projection of a GGUF Q8_0 file.
        {"name": "text_up_q8", "kind": "q8", "m": 77, "k": 3072, "n": 12288, "epilogue": "gelu_tanh",
         "out": "bf16"},
        # The text stream of a convrot int8 checkpoint: fp32 rows rotated, quantized, multiplied int8 by int8.
        {"name": "text_out_w8a8", "kind": "w8a8", "m": 512, "k": 3072, "n": 3072, "group": 256,
         "epilogue": "none", "out": "bf16"},
        # The library's operator as a host calls it by default on a map: an fp32 activation used whole.
        {"name": "image_out_fp32", "kind": "fp32", "m": 1531, "k": 3072, "n": 3072, "group": 0,
         "epilogue": "none", "out": "f32"},
        # The same operator on [K, N] codes as they lie in the map, the rows rounded already, a ragged count.
        {"name": "map_in_place_int8", "kind": "in_place", "m": 1021, "k": 3072, "n": 9216, "out": "f32"},
        # The image stream: up projection with GELU on 4096 rows in int8 (this library's headline) ...
        {"name": "image_up_int8", "kind": "linear", "m": 4096, "k": 3072, "n": 12288, "weight": "int8",
         "epilogue": "gelu_tanh", "out": "bf16"},
        # ... the fused gate and up projection of an fp8 checkpoint (the most work of one product) ...
        {"name": "image_gate_up_fp8", "kind": "linear", "m": 4096, "k": 3840, "n": 20480, "weight": "fp8",
         "epilogue": "silu_glu", "out": "bf16"},
        # ... the up projection on quantized activations ...
        {"name": "image_up_w8a8", "kind": "w8a8", "m": 4096, "k": 3072, "n": 12288, "group": 256,
         "epilogue": "gelu_tanh", "out": "bf16"},
        # ... and of a GGUF Q8_0 file.
        {"name": "image_up_q8", "kind": "q8", "m": 4096, "k": 3072, "n": 12288, "epilogue": "gelu_tanh",
         "out": "bf16"},
        # One whole single-stream block, 4096 image and 512 text tokens, its products on quantized activations.
        {"name": "block_w8a8", "kind": "block", "tokens": 4608, "d": 3072, "heads": 24, "route": "w8a8",
         "group": 256},
    ]


def draw(rng):
    """A case of the same kinds: 1 to 4608 rows, 768 to 12288 in, 64 to 20480 out, whole and ragged."""
    kind = rng.choice(["linear", "linear", "linear", "q8", "q8", "w8a8", "w8a8", "fp32", "in_place", "block"])

    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if kind == "block":
        heads = rng.choice([8, 12, 16, 24])
        route = rng.choice(["bf16", "w8a8"])
        return {"kind": "block", "tokens": log_int(256, 4608), "d": 128 * heads, "heads": heads, "route": route,
                "group": rng.choice([0, 64, 256]) if route == "w8a8" else 0}
    m = log_int(1, 4608)
    group = rng.choice([0, 16, 64, 256, 256]) if kind in ("w8a8", "fp32") else 0
    # Widths: whole steps of the kernels mostly, ragged ones among them (a block of 32 or a rotation group at least).
    step = {"q8": rng.choice([32, 64, 256]), "w8a8": max(group, 8), "fp32": max(group, 8)}.get(kind, rng.choice([8, 64, 256, 256]))
    k = max(1, round(log_int(768, 12288) / step)) * step
    n = log_int(64, 20480)
    ragged = rng.random() < 0.3
    n = max(64, n // 64 * 64) if not ragged else n
    epilogue = "none" if kind in ("fp32", "in_place") else rng.choice(["none", "none", "gelu_tanh", "silu_glu", "situ_glu"])
    if epilogue in GLU:
        n -= n % 2
    most = MOST_MACS // 3 if kind in ("fp32", "q8") else MOST_MACS
    while m * k * n > most:
        m = max(1, m // 2)
    c = {"kind": kind, "m": m, "k": k, "n": n, "out": rng.choice(["bf16", "bf16", "f32"])}
    if kind == "in_place":
        return c
    c["epilogue"] = epilogue
    if kind == "linear":
        c["weight"] = rng.choice(["int8", "int8", "fp8"])
    if kind in ("w8a8", "fp32"):
        c["group"] = group
    return c


# ---- inputs ----------------------------------------------------------------------------------------------------


def _normal(g, *shape):
    return torch.randn(*shape, device="cuda", generator=g)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _inputs(case, seed):
    """x [m, k], the codes [n, k], their scales and the bias: activations N(0, 1) (a normed or modulated row),
    weights N(0, 0.02) quantized per output channel to int8 or fp8 (Q8_0: per 32 of an output, fp16 scales)."""
    g = _generator(seed)
    m, k, n, kind = case["m"], case["k"], case["n"], case["kind"]
    x = _normal(g, m, k)
    if kind in ("linear", "in_place", "q8"):
        x = x.to(torch.bfloat16)
    w = _normal(g, n, k) * 0.02
    if kind == "q8":
        blocks = w.view(n, k // 32, 32)
        s = (blocks.abs().amax(dim=2) / 127.0).to(torch.float16)
        q = torch.round(blocks / s.float()[:, :, None]).clamp(-127, 127).to(torch.int8).view(n, k)
    elif case.get("weight") == "fp8":
        s = w.abs().amax(dim=1) / 448.0
        q = (w / s[:, None]).to(torch.float8_e4m3fn)
    else:
        s = w.abs().amax(dim=1) / 127.0
        q = torch.round(w / s[:, None]).clamp(-127, 127).to(torch.int8)
    bias = _normal(g, n) * 0.02
    return x, q, s, bias


def _block_inputs(case, seed):
    g = _generator(seed + 1)
    return _normal(g, case["tokens"], case["d"]), _normal(g, case["d"])


def prepare(case, seed):
    ctx = sq.context(0)
    if case["kind"] == "block":
        blk = DiTBlock(d=case["d"], heads=case["heads"], seed=seed, ctx=ctx, route=case["route"], group=case["group"])
        x, temb = _block_inputs(case, seed)
        return {"kind": "block", "block": blk, "x": x, "temb": temb}
    x, q, s, bias = _inputs(case, seed)
    m, k, n, kind = case["m"], case["k"], case["n"], case["kind"]
    epilogue = case.get("epilogue", "none")
    glu = epilogue in GLU
    out = torch.empty((m, n // 2 if glu else n), device="cuda",
                      dtype=torch.bfloat16 if case["out"] == "bf16" else torch.float32)
    state = {"kind": kind, "ctx": ctx, "x": x, "s": s, "bias": bias, "out": out, "epilogue": epilogue,
             "group": case.get("group", 0), "m": m, "k": k, "n": n}
    if kind == "in_place":
        state["w"] = q.t().contiguous()                      # the map's [K, N]
    elif kind == "q8":
        state["w"] = ctx.pack_blocks(q, s, 32, layout="nk", glu=glu)
    else:
        state["w"] = ctx.pack(q, layout="nk", glu=glu)
    return state


def run(state):
    kind = state["kind"]
    if kind == "block":
        return state["block"].forward(state["x"], state["temb"])
    ctx = state["ctx"]
    if kind == "linear":
        return ctx.product(state["x"], state["w"], state["s"], bias=state["bias"], epilogue=state["epilogue"],
                           out=state["out"])
    if kind == "q8":
        return ctx.product_blocks(state["x"], state["w"], bias=state["bias"], epilogue=state["epilogue"],
                                  out=state["out"])
    if kind == "w8a8":
        return ctx.product_quantized(state["x"], state["w"], state["s"], group=state["group"], bias=state["bias"],
                                     epilogue=state["epilogue"], out=state["out"])
    if kind == "fp32":
        return ctx.product(state["x"], state["w"], state["s"], bias=state["bias"], out=state["out"],
                           rotation=state["group"], rounding=False)
    ctx.linear(state["x"], int8=state["w"], scales=state["s"], per_column=True, c=state["out"], m=state["m"],
               k=state["k"], n=state["n"], settled=True)
    return state["out"]


# ---- what a pass cannot do without -----------------------------------------------------------------------------


def work(case):
    if case["kind"] == "block":
        s, d = case["tokens"], case["d"]
        weights = 18 * d * d                                  # modulation 6, QKV 3, out 1, up 4, down 4
        return {"bytes": weights + 8 * 18 * d + 8 * s * d,
                "flops": 2.0 * (6 * d * d + 12 * s * d * d) + 4.0 * s * s * d}
    m, k, n, kind = case["m"], case["k"], case["n"], case["kind"]
    n_out = n // 2 if case.get("epilogue") in GLU else n
    x = m * k * (4 if kind in ("w8a8", "fp32") else 2)
    scales = n * (k // 32) * 2 if kind == "q8" else 4 * n
    bias = 0 if kind == "in_place" else 4 * n
    return {"bytes": x + k * n + scales + bias + m * n_out * (2 if case["out"] == "bf16" else 4),
            "flops": 2.0 * m * k * n}


def tolerance(case):
    if case["kind"] == "block":
        # A rounding that falls the other way moves a bf16 operand or an int8 code, which travels on through the
        # block: its output is 1.4e-2 from the one in 64 bits.
        return {"rel": 3e-2, "max": 0.6}
    if case["out"] == "bf16":
        return {"rel": 7e-3, "max": 0.05}                     # the output's own rounding is 1.7e-3
    if case["kind"] == "w8a8":
        return {"rel": 2e-4, "max": 0.02}                     # a tie in the quantization that falls the other way
    return {"rel": 3e-6, "max": 5e-5}                         # fp32 sums of exact products: 1e-7 to 7e-7


# ---- the same in 64 bits, in plain torch -----------------------------------------------------------------------


def _rotate64(x, group):
    """x · R, R = H / sqrt(group) block-diagonal, H the Kronecker power of the regular 4 x 4 Hadamard matrix."""
    if not group:
        return x
    h4 = torch.tensor([[1, 1, 1, -1], [1, 1, -1, 1], [1, -1, 1, 1], [-1, 1, 1, 1]], dtype=torch.float64, device=x.device)
    h = torch.ones((1, 1), dtype=torch.float64, device=x.device)
    while h.shape[0] < group:
        h = torch.kron(h, h4)
    return (x.reshape(-1, group) @ (h / math.sqrt(group))).reshape(x.shape)


def _quantized64(x, group):
    y = _rotate64(x, group)
    s = (y.abs().amax(dim=1, keepdim=True) / 127.0).clamp_min(1e-30)
    return torch.round(y / s).clamp(-128, 127) * s


def _activated64(y, epilogue):
    half = y.shape[1] // 2
    if epilogue == "gelu_tanh":
        return torch.nn.functional.gelu(y, approximate="tanh")
    if epilogue == "silu_glu":
        return torch.nn.functional.silu(y[:, :half]) * y[:, half:]
    if epilogue == "situ_glu":
        v, g = y[:, :half], y[:, half:]
        return 4 * torch.tanh(g / 4) * torch.sigmoid(g) * 25 * torch.tanh(v / 25)
    return y


def exact(case, seed):
    if case["kind"] == "block":
        return _block64(case, seed)
    x, q, s, bias = _inputs(case, seed)
    kind, group = case["kind"], case.get("group", 0)
    x, w = x.double(), q.double()
    if kind == "q8":
        w = (w.view(w.shape[0], -1, 32) * s.double()[:, :, None]).view(w.shape)
    else:
        w = w * s.double()[:, None]
    x = _quantized64(x, group) if kind == "w8a8" else _rotate64(x, group)
    y = x @ w.t()
    if kind != "in_place":
        y = y + bias.double()
    return _activated64(y, case.get("epilogue", "none"))


def _block64(case, seed):
    """The block of siliconed_amd.dit_block in 64 bits, its weights drawn as its constructor draws them."""
    d, heads, group = case["d"], case["heads"], case["group"]
    hd, quantized = d // heads, case["route"] == "w8a8"
    g = _generator(seed)

    def linear(n, k):
        w = _normal(g, n, k) * 0.02
        s = (w.abs().amax(dim=1) / 127.0).clamp_min(1e-30)
        q = torch.round(w / s[:, None]).clamp(-127, 127)
        return q.double() * s.double()[:, None], (_normal(g, n) * 0.02).double()

    mod, qkv, out, up, down = linear(6 * d, d), linear(3 * d, d), linear(d, d), linear(4 * d, d), linear(d, 4 * d)
    norm_a, norm_f, norm_q, norm_k = ((1.0 + 0.02 * _normal(g, size)).double() for size in (d, d, hd, hd))
    x, temb = _block_inputs(case, seed)
    x = x.double()

    def rms(t, w):
        return t * torch.rsqrt((t * t).mean(dim=-1, keepdim=True) + 1e-6) * w

    def product(t, lin):
        return (_quantized64(t, group) if quantized else t) @ lin[0].t() + lin[1]

    six = temb.to(torch.bfloat16).double()[None] @ mod[0].t() + mod[1]
    shift_a, scale_a, gate_a, shift_f, scale_f, gate_f = six[0].chunk(6)
    q, k, v = product(rms(x, norm_a) * (1 + scale_a) + shift_a, qkv).view(-1, 3, heads, hd).unbind(1)
    q, k = rms(q, norm_q), rms(k, norm_k)
    o = torch.empty_like(x).view(-1, heads, hd)
    for i in range(heads):
        o[:, i] = torch.softmax(q[:, i] @ k[:, i].t() / math.sqrt(hd), dim=-1) @ v[:, i]
    x = x + gate_a * product(o.reshape(x.shape), out)
    h = torch.nn.functional.gelu(product(rms(x, norm_f) * (1 + scale_f) + shift_f, up), approximate="tanh")
    return x + gate_f * product(h, down)
