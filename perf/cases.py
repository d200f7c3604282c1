"""Performance cases of the BiGEMM framework: what a program that uses it has it do.

Four kinds of call, each through the package's public entry points:

* ``op``     ``bigemm(..., backend="hip")`` on pre-normalised activations, the operator alone;
* ``block``  one ``OmniWeaveBlock`` (RMSNorm, BiGEMM, residual) in inference, bf16 / fp16 / fp32,
             or with the fp8 channel side (``fp8``);
* ``train``  the same block forward and backward: output and every gradient, with or without
             the per-image drop-path (``drop``);
* ``model``  a whole OmniWeave-T forward: images to logits.

Shapes are the four stages of OmniWeave-T at 224 px (56x56x128, 28x28x256, 14x14x512, 7x7x1024),
the stages at other image sizes, and channel counts and sides that fill no tile.  Weights are
drawn at fan-in scale and LayerScale around one, as trained layers have them: at its initial 1e-5
the delta would vanish beside the residual.
"""

from __future__ import annotations

import math

import torch

import omniwave_amd
from omniwave_amd.block import OmniWeaveBlock, enable_fp8
from omniwave_amd.hip import bigemm_block_hip

G = 16  # tokens of a group
EPS = 1e-6
WIDTHS, DEPTHS, TILES, CLASSES = (128, 256, 512, 1024), (2, 3, 8, 2), (64, 64, 128, 128), 1000
ANCHORED = (2, 3)  # stages (from 0) that begin with a Linear
SCHEDULE = (("local", 0), ("shifted", 0), ("radix", 0), ("radix", 1), ("radix", 2))
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
DROP_RATE = 0.1
DEVICE = "cuda"

# Most values of x (or image pixels, for the model) of a drawn case.
MOST_16BIT, MOST_F32 = 128 * 56 * 56 * 128, 32 * 28 * 28 * 256
MOST_PIXELS_16BIT, MOST_PIXELS_F32 = 256 * 224 * 224, 8 * 224 * 224


def _layer(name, kind, b, h, w, c, d, route, level, dtype, **options):
    case = {"kind": kind, "b": b, "h": h, "w": w, "c": c, "d": d, "route": route, "level": level, "dtype": dtype,
            "fp8": False, "drop": False}
    case.update(options)
    return {"name": name, **case} if name else case


def _model(name, b, size, dtype):
    case = {"kind": "model", "b": b, "size": size, "dtype": dtype}
    return {"name": name, **case} if name else case


def listed():
    return [
        # One image through the operator in half precision: the latency point of the operator sweep.
        _layer("op_14x14x512_b1_f16", "op", 1, 14, 14, 512, 128, "local", 0, "f16"),
        # A few requests at once through a late layer: serving at low load, strided channel groups.
        _layer("block_7x7x1024_b8_bf16_radix1", "block", 8, 7, 7, 1024, 128, "radix", 1, "bf16"),
        # An early layer at full batch, the most activations of any layer: throughput inference.
        _layer("block_56x56x128_b128_bf16_shifted", "block", 128, 56, 56, 128, 64, "shifted", 0, "bf16"),
        # The stage that most layers belong to, at full batch.
        _layer("block_14x14x512_b128_bf16_local", "block", 128, 14, 14, 512, 128, "local", 0, "bf16"),
        # The same layer in the default dtype of a new model, at the operator sweep's largest batch.
        _layer("block_14x14x512_b32_f32_local", "block", 32, 14, 14, 512, 128, "local", 0, "f32"),
        # A narrower network at 160 px: a channel group that is only half there.
        _layer("block_40x40x96_b64_bf16_shifted", "block", 64, 40, 40, 96, 64, "shifted", 0, "bf16"),
        # Inference with the fp8 channel side, the middle of its batch sweep.
        _layer("fp8_14x14x512_b256_bf16_shifted", "block", 256, 14, 14, 512, 128, "shifted", 0, "bf16", fp8=True),
        # Training an early layer at full batch.
        _layer("train_56x56x128_b128_bf16_shifted", "train", 128, 56, 56, 128, 64, "shifted", 0, "bf16"),
        # Training a middle layer with strided channel groups and drop-path.
        _layer("train_14x14x512_b64_bf16_radix1_drop", "train", 64, 14, 14, 512, 128, "radix", 1, "bf16", drop=True),
        # Training in the default dtype of a new model.
        _layer("train_28x28x256_b32_f32_local", "train", 32, 28, 28, 256, 64, "local", 0, "f32"),
        # The whole network, throughput inference.
        _model("model_224_b256_bf16", 256, 224, "bf16"),
        # The whole network as created (fp32), a few images.
        _model("model_224_b8_f32", 8, 224, "f32"),
    ]


def _log_int(rng, low, high):
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def draw(rng):
    kind = rng.choices(["op", "block", "fp8", "train", "model"], [15, 30, 10, 30, 15])[0]
    dtype = rng.choices(["bf16", "f16", "f32"], [50, 25, 25])[0]
    if kind == "model":
        most = MOST_PIXELS_F32 if dtype == "f32" else MOST_PIXELS_16BIT
        size = 32 * rng.randint(2, 10)
        return _model(None, _log_int(rng, 1, max(1, min(256, most // (size * size)))), size, dtype)
    if kind == "fp8":
        dtype = rng.choice(["bf16", "f16"])
    if rng.random() < 0.8:  # a stage of the network at some image size
        stage = rng.randrange(2, 4) if kind == "fp8" else rng.randrange(4)
        c, d = WIDTHS[stage], TILES[stage]
        h = w = max(2, (8 * rng.randint(2, 12)) >> stage)
    else:  # other widths and sides
        d = 128 if kind == "fp8" else rng.choice([64, 128])
        c = _log_int(rng, d // 2 + 1, 8 * d)
        h, w = rng.randint(3, 40), rng.randint(3, 40)
    route, level = rng.choice(SCHEDULE)
    most = MOST_F32 if dtype == "f32" else MOST_16BIT
    b = _log_int(rng, 1, max(1, min(256, most // (h * w * c))))
    return _layer(None, "block" if kind == "fp8" else kind, b, h, w, c, d, route, level, dtype, fp8=kind == "fp8",
                  drop=kind == "train" and rng.random() < 0.25)


# ---------------------------------------------------------------------------------------
# Inputs


def _generator(seed):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    return gen


def _layer_weights(gen, c, d, dtype):
    """Parameters of one block in ``dtype``: token matrices and channel matrices at fan-in scale."""
    q_c, rd = -(-c // d), 2 * d

    def normal(*shape, fan):
        return (torch.randn(shape, generator=gen, device=DEVICE) / math.sqrt(fan)).to(dtype)

    def around_one(n):
        return (torch.rand(n, generator=gen, device=DEVICE) + 0.5).to(dtype)

    return {
        "norm_weight": around_one(c),
        "a_u": normal(G, G, fan=G), "a_v": normal(G, G, fan=G), "a_o": normal(G, G, fan=G),
        "b_u": normal(q_c, d, rd, fan=d), "b_v": normal(q_c, d, rd, fan=d), "b_o": normal(q_c, rd, d, fan=rd),
        "gamma": around_one(c),
    }


def _layer_inputs(case, seed):
    gen = _generator(seed)
    dtype = DTYPES[case["dtype"]]
    shape = (case["b"], case["h"], case["w"], case["c"])
    weights = _layer_weights(gen, case["c"], case["d"], dtype)
    data = {"x": torch.randn(shape, generator=gen, device=DEVICE).to(dtype), "dy": None, "keep": None}
    if case["kind"] == "train":
        data["dy"] = torch.randn(shape, generator=gen, device=DEVICE).to(dtype)
        if case["drop"]:
            data["keep"] = torch.rand(case["b"], generator=gen, device=DEVICE) >= DROP_RATE
    return weights, data


def _model_inputs(case, seed):
    """State dict and images; the residual branches are weighted 0.5 so that 15 of them keep scale."""
    gen = _generator(seed)
    dtype = DTYPES[case["dtype"]]

    def linear(n_out, n_in):
        return (torch.randn(n_out, n_in, generator=gen, device=DEVICE) / math.sqrt(n_in)).to(dtype)

    state = {"stem_proj.weight": linear(WIDTHS[0], 48)}
    for i in range(4):
        if i:
            state[f"downsamples.{i - 1}.weight"] = linear(WIDTHS[i], 4 * WIDTHS[i - 1])
        if i in ANCHORED:
            state[f"stages.{i}.anchor.weight"] = linear(WIDTHS[i], WIDTHS[i])
        for j in range(DEPTHS[i]):
            for name, t in _layer_weights(gen, WIDTHS[i], TILES[i], dtype).items():
                state[f"stages.{i}.blocks.{j}.{name}"] = t * 0.5 if name == "gamma" else t
    state["head.weight"] = linear(CLASSES, WIDTHS[3])
    state["head.bias"] = (0.1 * torch.randn(CLASSES, generator=gen, device=DEVICE)).to(dtype)
    images = torch.randn(case["b"], 3, case["size"], case["size"], generator=gen, device=DEVICE).to(dtype)
    return state, images


def prepare(case, seed):
    if case["kind"] == "model":
        weights, images = _model_inputs(case, seed)
        model = omniwave_amd.create_model("omniweave_t", input_size=case["size"], num_classes=CLASSES)
        model = model.to(device=DEVICE, dtype=DTYPES[case["dtype"]]).eval()
        model.load_state_dict(weights)
        return {"kind": "model", "model": model, "images": images}
    weights, data = _layer_inputs(case, seed)
    x = data["x"]
    if case["kind"] == "op":
        plan = omniwave_amd.build_route_plan(case["h"], case["w"], case["c"], G, case["d"], case["route"],
                                             case["level"])
        weights.pop("norm_weight")
        return {"kind": "op", "x": x, "plan": plan, "weights": weights}
    block = OmniWeaveBlock(case["h"], case["w"], case["c"], case["d"], case["route"], case["level"])
    block = block.to(device=DEVICE, dtype=x.dtype)
    block.load_state_dict(weights)
    if case["kind"] == "block":
        block.eval()
        if case["fp8"]:
            enable_fp8(block)
        return {"kind": "block", "x": x, "block": block}
    scale = None
    if case["drop"]:
        scale = data["keep"].float() / (1.0 - DROP_RATE)
    return {"kind": "train", "x": x.requires_grad_(True), "dy": data["dy"], "block": block, "scale": scale}


def run(state):
    kind = state["kind"]
    if kind == "op":
        with torch.inference_mode():
            return omniwave_amd.bigemm(x=state["x"], plan=state["plan"], backend="hip", **state["weights"])
    if kind == "block":
        with torch.inference_mode():
            return state["block"](state["x"])
    if kind == "model":
        with torch.inference_mode():
            return state["model"](state["images"])
    x, blk = state["x"], state["block"]
    if state["scale"] is None:
        out = blk(x)
    else:
        out = bigemm_block_hip(x, blk.norm_weight, blk.plan, blk.a_u, blk.a_v, blk.a_o, blk.b_u, blk.b_v, blk.b_o,
                               blk.gamma, eps=EPS, drop_scale=state["scale"])
    params = (blk.norm_weight, blk.a_u, blk.a_v, blk.a_o, blk.b_u, blk.b_v, blk.b_o, blk.gamma)
    return (out.detach(), *torch.autograd.grad(out, (x, *params), state["dy"]))


# ---------------------------------------------------------------------------------------
# Work and tolerance


def _layer_flops(tokens, c, rd):
    """Three token products (16 deep) and three channel products per token and channel."""
    return 6.0 * tokens * c * (G + rd)


def _layer_params(c, d):
    return 3 * G * G + 3 * (-(-c // d)) * d * 2 * d + 2 * c


def work(case):
    size = 4 if case["dtype"] == "f32" else 2
    if case["kind"] == "model":
        b, side = case["b"], case["size"] // 4
        flops = 2.0 * b * side * side * 48 * WIDTHS[0] + 2.0 * b * WIDTHS[3] * CLASSES
        params = 48 * WIDTHS[0] + WIDTHS[3] * CLASSES + CLASSES
        for i in range(4):
            tokens = b * (side >> i) ** 2
            if i:
                flops += 2.0 * tokens * 4 * WIDTHS[i - 1] * WIDTHS[i]
                params += 4 * WIDTHS[i - 1] * WIDTHS[i]
            if i in ANCHORED:
                flops += 2.0 * tokens * WIDTHS[i] * WIDTHS[i]
                params += WIDTHS[i] * WIDTHS[i]
            flops += DEPTHS[i] * _layer_flops(tokens, WIDTHS[i], 2 * TILES[i])
            params += DEPTHS[i] * _layer_params(WIDTHS[i], TILES[i])
        values = b * 3 * case["size"] ** 2 + params + b * CLASSES
        return {"bytes": float(values * size), "flops": flops}
    tokens = case["b"] * case["h"] * case["w"]
    flops = _layer_flops(tokens, case["c"], 2 * case["d"])
    values, params = tokens * case["c"], _layer_params(case["c"], case["d"])
    if case["kind"] == "train":  # x and dy in, out and dx out, the parameters in and their gradients out
        return {"bytes": float((4 * values + 2 * params) * size), "flops": 3 * flops}
    return {"bytes": float((2 * values + params) * size), "flops": flops}


def tolerance(case):
    """About four times the largest error against 64 bits seen over the declared ranges: bf16 layers
    4.8e-3 and gradients 7.0e-3, f16 5.9e-4 and 9.6e-4, f32 4.5e-7 and 7.7e-7, the fp8 channel side
    2.1e-2, logits 1.2e-2 (bf16), 1.5e-3 (f16) and 1.6e-6 (f32)."""
    if case["kind"] == "model":
        return {"rel": {"bf16": 5e-2, "f16": 6e-3, "f32": 7e-6}[case["dtype"]]}
    if case["fp8"]:
        return {"rel": 8e-2}
    if case["kind"] == "train":
        return {"rel": {"bf16": 2.8e-2, "f16": 4e-3, "f32": 4e-6}[case["dtype"]]}
    return {"rel": {"bf16": 2e-2, "f16": 2.5e-3, "f32": 2e-6}[case["dtype"]]}


# ---------------------------------------------------------------------------------------
# The same results in 64 bits


def _token_order(h, w, route, level):
    n = h * w
    if route == "radix":
        stride = G ** level
        return [i for base in range(0, n, stride * G) for off in range(stride)
                for i in range(base + off, base + off + stride * G, stride) if i < n]
    start = 0 if route == "local" else -2
    order = {}  # windows of 4x4, wrapped when shifted: the first window that holds a token takes it
    for r0 in range(start, h + start, 4):
        for c0 in range(start, w + start, 4):
            for r in range(r0, r0 + 4):
                for c in range(c0, c0 + 4):
                    if route == "local" and (r >= h or c >= w):
                        continue
                    order.setdefault((r % h) * w + c % w)
    return list(order)


def _channel_order(c, d, level):
    n = -(-c // d)
    if level == 0 or n == 1:
        return list(range(c))
    return [i for k in range(n) for i in range((k + level) % n, c, n)]


def _tables(h, w, c, d, route, level):
    """Positions of the tokens and channels in the padded tile order."""
    tok = torch.tensor(_token_order(h, w, route, level), device=DEVICE)
    chan = torch.tensor(_channel_order(c, d, level), device=DEVICE)
    return tok, chan


def _delta64(x, p, tables, d):
    """The BiGEMM delta of ``x`` [B, N, C], in the dtype of ``x``."""
    tok, chan = tables
    b, n, c = x.shape
    q_s, q_c = -(-n // G), -(-c // d)
    tiles = x[:, tok][:, :, chan]
    tiles = torch.nn.functional.pad(tiles, (0, q_c * d - c, 0, q_s * G - n))
    tiles = tiles.reshape(b, q_s, G, q_c, d).permute(0, 1, 3, 2, 4)
    u = p["a_u"] @ tiles @ p["b_u"]
    v = p["a_v"] @ tiles @ p["b_v"]
    delta = p["a_o"] @ (torch.nn.functional.silu(u) * v @ p["b_o"])
    delta = delta.permute(0, 1, 3, 2, 4).reshape(b, q_s * G, q_c * d)[:, :n, :c]
    # position i of the order holds token tok[i] / channel chan[i]
    delta = delta[:, torch.argsort(tok)][:, :, torch.argsort(chan)]
    return delta * p["gamma"]


def _block64(x, p, tables, d, keep=None):
    normed = x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + EPS) * p["norm_weight"]
    delta = _delta64(normed, p, tables, d)
    return x + (delta if keep is None else delta * keep)


def _images_at_once(n, c):
    return max(1, int(2.0e7 // (n * c)))


def _exact_model(case, seed):
    state, images = _model_inputs(case, seed)
    p = {k: v.double() for k, v in state.items()}

    def to_depth(x, f):
        b, h, w, c = x.shape
        x = x.reshape(b, h // f, f, w // f, f, c).permute(0, 1, 3, 2, 4, 5)
        return x.reshape(b, h // f, w // f, c * f * f)

    side = case["size"] // 4
    tables = [[_tables(side >> i, side >> i, WIDTHS[i], TILES[i], *SCHEDULE[j % 5]) for j in range(DEPTHS[i])]
              for i in range(4)]
    logits = []
    for part in images.split(_images_at_once(side * side, WIDTHS[0])):
        x = to_depth(part.double().permute(0, 2, 3, 1), 4) @ p["stem_proj.weight"].T
        for i in range(4):
            if i:
                x = to_depth(x, 2) @ p[f"downsamples.{i - 1}.weight"].T
            if i in ANCHORED:
                x = x @ p[f"stages.{i}.anchor.weight"].T
            b, h, w, c = x.shape
            x = x.reshape(b, h * w, c)
            for j in range(DEPTHS[i]):
                prefix = f"stages.{i}.blocks.{j}."
                block = {k[len(prefix):]: v for k, v in p.items() if k.startswith(prefix)}
                x = _block64(x, block, tables[i][j], TILES[i])
            x = x.reshape(b, h, w, c)
        logits.append(x.mean(dim=(1, 2)) @ p["head.weight"].T + p["head.bias"])
    return torch.cat(logits)


def exact(case, seed):
    if case["kind"] == "model":
        with torch.no_grad():
            return _exact_model(case, seed)
    weights, data = _layer_inputs(case, seed)
    b, h, w, c = data["x"].shape
    tables = _tables(h, w, c, case["d"], case["route"], case["level"])
    p = {k: v.double() for k, v in weights.items()}
    x = data["x"].reshape(b, h * w, c)
    step = _images_at_once(h * w, c)
    if case["kind"] != "train":
        fn = _delta64 if case["kind"] == "op" else _block64
        with torch.no_grad():
            out = torch.cat([fn(part.double(), p, tables, case["d"]) for part in x.split(step)])
        return out.reshape(b, h, w, c)
    dy = data["dy"].reshape(b, h * w, c)
    keep = None if data["keep"] is None else (data["keep"].double() / (1.0 - DROP_RATE)).reshape(b, 1, 1)
    names = ("norm_weight", "a_u", "a_v", "a_o", "b_u", "b_v", "b_o", "gamma")
    leaves = {k: p[k].requires_grad_(True) for k in names}
    outs, dxs, sums = [], [], None
    for i in range(0, b, step):
        xi = x[i:i + step].double().requires_grad_(True)
        out = _block64(xi, leaves, tables, case["d"], None if keep is None else keep[i:i + step])
        dx, *grads = torch.autograd.grad(out, (xi, *leaves.values()), dy[i:i + step].double())
        outs.append(out.detach())
        dxs.append(dx)
        sums = grads if sums is None else [s + g for s, g in zip(sums, grads)]
    return (torch.cat(outs).reshape(b, h, w, c), torch.cat(dxs).reshape(b, h, w, c), *sums)
