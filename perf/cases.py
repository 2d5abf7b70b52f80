"""The workloads this package is timed on: its public ops and refiner blocks at the sizes an image-matching program
calls them with, from one small convolution to a pass of the refiner stack.

A case names a ``kind`` (one public entry point or block) and its sizes. Activations and weights are drawn on the GPU
from the seed; the quantized operands are made here with plain torch, so the reference results of :func:`exact` need
nothing of this package. Activations carry per-channel outliers (log-uniform factors), as measured ones do.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from flashim_amd import blocks, ops

DEV = "cuda"
BF16 = torch.bfloat16
E4M3 = torch.float8_e4m3fn


def listed() -> list[dict]:
    return [
        # the smallest layer: a 64-channel INT8 conv of a backbone on a 128 x 128 image; launch latency counts
        dict(name="int8_conv3x3_64_128x128", kind="int8_conv", b=1, h=128, w=128, cin=64, cout=64, k=3, stride=1,
             relu=False, bias="fp32", out="bf16", residual=False),
        # a deep VGG layer whose output feeds the next INT8 layer: large K, ReLU, chained INT8 output
        dict(name="int8_conv3x3_512_112x150", kind="int8_conv", b=1, h=112, w=150, cin=512, cout=512, k=3, stride=1,
             relu=True, bias="bf16", out="int8", residual=False),
        # a ResNet-FPN layer with a channel count that is no multiple of 16 (196 -> 128 on half of an 896 x 1200 image)
        dict(name="int8_conv3x3_196_448x600", kind="int8_conv", b=1, h=448, w=600, cin=196, cout=128, k=3, stride=1,
             relu=True, bias="bf16", out="bf16", residual=False),
        # an MXFP8 3x3 layer with a folded BatchNorm on a batch of two 200 x 200 maps
        dict(name="mxfp8_conv3x3_128_200x200", kind="mxfp8_conv", b=2, h=200, w=200, cin=128, cout=128, k=3, stride=1,
             relu=True, gelu=False, bias="bf16", out="bf16", residual=False),
        # a wide MXFP8 3x3 layer in a chain of quantized layers: E4M3 output for the next one
        dict(name="mxfp8_conv3x3_256_224x300", kind="mxfp8_conv", b=1, h=224, w=300, cin=256, cout=256, k=3, stride=1,
             relu=True, gelu=False, bias="bf16", out="e4m3", residual=False),
        # a pointwise projection with GELU
        dict(name="mxfp8_conv1x1_512_gelu", kind="mxfp8_conv", b=2, h=100, w=100, cin=512, cout=512, k=1, stride=1,
             relu=False, gelu=True, bias="bf16", out="bf16", residual=False),
        # quantizing a BF16 activation for an MXFP8 layer: a memory stream
        dict(name="quantize_mxfp8_128_200x200", kind="quantize", format="mxfp8", layout="nhwc", b=2, h=200, w=200,
             c=128),
        # the first layer of VGG on a whole image: BF16 NCHW in, INT8 NHWC out
        dict(name="stem_896x1200", kind="stem", b=1, h=896, w=1200, cin=3, cout=64),
        # a depthwise-then-pointwise refiner block with dynamic MXFP8 between the two
        dict(name="dwpw_mxfp8_128_400x400", kind="dwpw", format="mxfp8", b=2, h=400, w=400, c=128),
        # one refiner block with its MLP at the finest scale (64 channels), MXFP8
        dict(name="block_mxfp8_64_400x400", kind="block", preset="mxfp8", b=2, h=400, w=400, c=64),
        # one refiner block at a coarser scale (256 channels), INT8
        dict(name="block_int8_256_200x200", kind="block", preset="int8", b=2, h=200, w=200, c=256),
        # a whole call: the refiner stack's four scales over both images (the two matching directions), two blocks a scale
        dict(name="stack_mxfp8_800_1024", kind="stack", preset="mxfp8", size_a=800, size_b=1024, blocks=2),
    ]


CHANNELS = (64, 96, 128, 160, 192, 224, 256, 320, 384, 512)
RAGGED = (36, 68, 100, 196)  # INT8 layers also come with channel counts that are no multiple of 16
MOST_FLOPS = 1.6e11  # of a drawn convolution


def _log_uniform(rng, lo: float, hi: float) -> float:
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _image(rng, lo: float, hi: float) -> tuple[int, int, int]:
    """A batch and an image size of ``lo`` to ``hi`` pixels in all, any aspect between 1:2 and 2:1, odd sizes too."""
    b = rng.choice((1, 1, 2, 2, 3))
    pixels = _log_uniform(rng, lo, hi) / b
    aspect = _log_uniform(rng, 0.5, 2.0)
    return b, max(3, round(math.sqrt(pixels * aspect))), max(3, round(math.sqrt(pixels / aspect)))


def draw(rng) -> dict:
    kind = rng.choice(("int8_conv", "int8_conv", "mxfp8_conv", "mxfp8_conv", "mxfp8_conv", "quantize", "stem", "dwpw",
                       "dwpw", "block", "block", "block", "stack"))
    if kind in ("int8_conv", "mxfp8_conv"):
        while True:
            b, h, w = _image(rng, 4096, 4e5)
            int8 = kind == "int8_conv"
            case = dict(kind=kind, b=b, h=h, w=w, cin=rng.choice(CHANNELS + (RAGGED if int8 else ())),
                        cout=rng.choice(CHANNELS + (RAGGED if int8 else ())), k=rng.choice((1, 3, 3, 3, 5)),
                        stride=rng.choice((1, 1, 1, 2)), relu=rng.random() < 0.6, bias=rng.choice(("bf16", "fp32")),
                        out=rng.choice(("bf16", "bf16", "int8" if int8 else "e4m3")), residual=rng.random() < 0.2)
            if not int8:
                case["gelu"] = case["k"] == 1 and not case["relu"]
            if work(case)["flops"] <= MOST_FLOPS:
                return case
    if kind == "quantize":
        b, h, w = _image(rng, 4096, 1e6)
        c = rng.choice((32, 64, 128, 192, 256))
        return dict(kind=kind, format=rng.choice(("mxfp8", "int8")), layout=rng.choice(("nhwc", "nhwc", "nchw")), b=b,
                    h=h, w=w, c=c)
    if kind == "stem":
        b, h, w = _image(rng, 6e4, 2e6)
        return dict(kind=kind, b=b, h=h, w=w, cin=rng.choice((1, 3, 3)), cout=rng.choice((32, 64, 64)))
    if kind == "dwpw":
        b, h, w = _image(rng, 8192, 4e5)
        return dict(kind=kind, format=rng.choice(("bf16", "mxfp8", "int8")), b=b, h=h, w=w,
                    c=rng.choice((32, 64, 96, 128, 128)))
    if kind == "block":
        c = rng.choice((64, 64, 128, 192, 256, 512))
        b, h, w = _image(rng, 4096, 4e5 * 64 / c)
        return dict(kind=kind, preset=rng.choice(("mxfp8", "int8")), b=b, h=h, w=w, c=c)
    size = round(_log_uniform(rng, 256, 900))
    return dict(kind=kind, preset=rng.choice(("mxfp8", "int8")), size_a=size, size_b=min(1000, round(size * 1.25)),
                blocks=rng.choice((1, 2)))


# -- inputs ------------------------------------------------------------------------------------------------------


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape) -> torch.Tensor:
    return torch.randn(*shape, generator=g, device=DEV)


def _activation(g, b: int, h: int, w: int, c: int, relu: bool) -> torch.Tensor:
    """FP32 NHWC, per-channel factors between 0.3 and 3, non-negative after a ReLU."""
    factor = torch.exp(torch.empty(c, device=DEV).uniform_(math.log(0.3), math.log(3.0), generator=g))
    x = _randn(g, b, h, w, c).mul_(factor)
    return x.relu_() if relu else x


def _exponent(amax: torch.Tensor) -> torch.Tensor:
    """The smallest power of two that brings ``amax`` into E4M3's range, as an int8 exponent (-127 for zero)."""
    e = torch.ceil(torch.log2(amax / 448.0))
    return torch.where(amax == 0, torch.full_like(e, -127.0), e).clamp(-127, 127).to(torch.int8)


def _e4m3(x: torch.Tensor, exponent: torch.Tensor) -> torch.Tensor:
    """``x`` ``[..., C]`` in blocks of 32 channels divided by ``2^exponent``, saturated, as E4M3."""
    blocks32 = x.reshape(*x.shape[:-1], -1, 32)
    scaled = blocks32 * torch.exp2(-exponent.to(blocks32.dtype))[..., None]
    return scaled.clamp(-448.0, 448.0).float().to(E4M3).reshape(x.shape)


def _mx_weight(w: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    e = _exponent(w.reshape(w.shape[0], -1, 32).abs().amax(dim=-1))
    return _e4m3(w, e), e


def _int8(x: torch.Tensor, scale: torch.Tensor) -> torch.Tensor:
    return (x / scale).round_().clamp_(-127, 127).to(torch.int8)


def _out_hw(c: dict) -> tuple[int, int]:
    pad = c["k"] // 2
    return (c["h"] + 2 * pad - c["k"]) // c["stride"] + 1, (c["w"] + 2 * pad - c["k"]) // c["stride"] + 1


def _prepare_conv(c: dict, g) -> dict:
    cin, cout, k, stride = c["cin"], c["cout"], c["k"], c["stride"]
    x = _activation(g, c["b"], c["h"], c["w"], cin, c["relu"])
    w = _randn(g, cout, k * k * cin) * (2.0 / (k * k * cin)) ** 0.5
    bias = (_randn(g, cout) * 0.1).to(BF16 if c["bias"] == "bf16" else torch.float32)
    kwargs = {"relu": c["relu"]}
    if c["residual"]:
        kwargs["residual"] = _randn(g, c["b"], *_out_hw(c), cout).to(BF16)
    geo = (k, k, stride, stride, k // 2, k // 2, 1, 1)
    if c["kind"] == "int8_conv":
        a_scale, w_scale = x.abs().amax() / 127, w.abs().amax(dim=1) / 127
        if c["out"] == "int8":
            kwargs["out_scale"] = torch.tensor(0.05, device=DEV)
        return dict(op="int8_conv2d", args=(_int8(x, a_scale), _int8(w, w_scale[:, None]), a_scale, w_scale, bias, *geo),
                    kwargs=kwargs)
    kwargs["gelu"] = c["gelu"]
    expo = _exponent(x.reshape(-1, cin // 32, 32).abs().amax(dim=(0, 2)))
    wq, w_expo = _mx_weight(w)
    if c["out"] == "e4m3":
        kwargs["out_exponent"] = torch.full((cout // 32,), -5, dtype=torch.int8, device=DEV)
    return dict(op="mxfp8_conv2d", args=(_e4m3(x, expo), expo, wq, w_expo, bias, *geo), kwargs=kwargs)


def _block(g, channels: int, preset: str) -> blocks.RefinerBlock:
    c, h = channels, 4 * channels
    u = lambda: torch.rand(c, generator=g, device=DEV) + 0.5  # noqa: E731
    return blocks.RefinerBlock(blocks.BlockWeights(
        dw_weight=_randn(g, c, 1, 5, 5) * 0.2, dw_bias=_randn(g, c) * 0.1, bn_gamma=u(), bn_beta=_randn(g, c) * 0.1,
        bn_mean=_randn(g, c) * 0.1, bn_var=u(), w1=_randn(g, h, c) * c ** -0.5, b1=_randn(g, h) * 0.1,
        w2=_randn(g, c, h) * h ** -0.5, b2=_randn(g, c) * 0.1), preset)


def prepare(case: dict, seed: int) -> dict:
    c, g, kind = case, _gen(seed), case["kind"]
    if kind in ("int8_conv", "mxfp8_conv"):
        return {"kind": "conv", **_prepare_conv(c, g)}
    if kind == "quantize":
        x = _activation(g, c["b"], c["h"], c["w"], c["c"], True).to(BF16)
        if c["layout"] == "nchw":  # the NHWC view of NCHW memory
            x = x.permute(0, 3, 1, 2).contiguous().permute(0, 2, 3, 1)
        amax = x.abs().amax(dim=(0, 1, 2)).float()
        scale = _exponent(amax.reshape(-1, 32).amax(dim=1)) if c["format"] == "mxfp8" else amax.amax() / 127
        return dict(kind=kind, op="quantize_" + c["format"], args=(x, scale))
    if kind == "stem":
        x = _randn(g, c["b"], c["cin"], c["h"], c["w"]).to(BF16)
        w = (_randn(g, c["cout"], c["cin"], 3, 3) * 0.3).to(BF16)
        bias = (_randn(g, c["cout"]) * 0.1).to(BF16)
        return dict(kind=kind, bound=ops.conv2d_small_cin_quantize_int8.bind(w, bias).warmup(),
                    args=(x, torch.tensor(0.04, device=DEV)))
    if kind == "dwpw":
        n = c["c"]
        x = (_randn(g, c["b"], c["h"], c["w"], n) * 2).to(BF16).permute(0, 3, 1, 2)
        dw_w, dw_b, pw_b = (_randn(g, 25, n) * 0.3).to(BF16), _randn(g, n), _randn(g, n)
        w = _randn(g, n, n) * n ** -0.5
        if c["format"] == "bf16":
            return dict(kind=kind, op="depthwise5x5_relu_pointwise",
                        args=(x, dw_w, dw_b.to(BF16), w.to(BF16), pw_b.to(BF16)))
        if c["format"] == "int8":
            w_scale = w.abs().amax(dim=1) / 127
            return dict(kind=kind, op="depthwise5x5_relu_pointwise_int8",
                        args=(x, dw_w, dw_b, _int8(w, w_scale[:, None]), w_scale, pw_b, torch.tensor(0.1, device=DEV)))
        wq, e = _mx_weight(w)
        e8m0 = (e.to(torch.int16) + 127).to(torch.uint8)
        rows, cols = -(-n // 128) * 128, -(-(n // 32) // 4) * 4
        swizzled = F.pad(e8m0, (0, cols - n // 32, 0, rows - n)).view(rows // 128, 4, 32, cols // 4, 4)
        swizzled = swizzled.permute(0, 3, 2, 1, 4).reshape(-1).contiguous()
        return dict(kind=kind, op="depthwise5x5_relu_pointwise_mxfp8",
                    args=(x, dw_w, dw_b, wq, swizzled.view(torch.float8_e8m0fnu), e8m0.view(torch.float8_e8m0fnu), pw_b))
    if kind == "block":
        x = _randn(g, c["b"], c["h"], c["w"], c["c"]).to(BF16)
        return dict(kind=kind, block=_block(g, c["c"], c["preset"]).calibrate(x), x=x)
    scales = []
    for stride, channels in blocks.STACK_SCALES:
        inputs = [_randn(g, 2, size // stride, size // stride, channels).to(BF16) for size in (c["size_a"], c["size_b"])]
        scales.append((inputs, [_block(g, channels, c["preset"]).calibrate(inputs[0]) for _ in range(c["blocks"])]))
    return dict(kind=kind, scales=scales, side=torch.cuda.Stream())


def run(state: dict):
    kind = state["kind"]
    if kind == "conv":
        return ops.OPS[state["op"]](*state["args"], **state["kwargs"])
    if kind == "quantize":
        return ops.OPS[state["op"]](*state["args"]).values
    if kind == "stem":
        return state["bound"](*state["args"]).values
    if kind == "dwpw":
        return ops.OPS[state["op"]](*state["args"])
    if kind == "block":
        return state["block"](state["x"])
    return blocks.run_stack(state["scales"], state["side"])


# -- what a pass cannot do without -----------------------------------------------------------------------------------


def _block_work(pixels: int, c: int) -> tuple[float, float]:
    """One block: its BF16 input (also the residual) and output once, its byte weights; two GEMMs and the depthwise."""
    return pixels * c * 4 + 8 * c * c, pixels * (2 * 25 * c + 2 * 2 * c * 4 * c)


def work(case: dict) -> dict:
    c, kind = case, case["kind"]
    if kind in ("int8_conv", "mxfp8_conv"):
        ho, wo = _out_hw(c)
        m, taps = c["b"] * ho * wo, c["k"] ** 2
        out = m * c["cout"] * (2 if c["out"] == "bf16" else 1) + (2 * m * c["cout"] if c["residual"] else 0)
        return {"bytes": c["b"] * c["h"] * c["w"] * c["cin"] + taps * c["cin"] * c["cout"] + out,
                "flops": 2 * m * taps * c["cin"] * c["cout"]}
    if kind == "quantize":
        n = c["b"] * c["h"] * c["w"] * c["c"]
        return {"bytes": 3 * n, "flops": 2 * n}
    pixels = c["b"] * c["h"] * c["w"] if kind != "stack" else 0
    if kind == "stem":
        return {"bytes": pixels * (2 * c["cin"] + c["cout"]), "flops": 2 * pixels * 9 * c["cin"] * c["cout"]}
    if kind == "dwpw":
        n = c["c"]
        return {"bytes": 4 * pixels * n + n * n, "flops": pixels * (2 * 25 * n + 2 * n * n)}
    if kind == "block":
        nbytes, flops = _block_work(pixels, c["c"])
        return {"bytes": nbytes, "flops": flops}
    parts = [_block_work(2 * (size // s) ** 2, ch) for s, ch in blocks.STACK_SCALES for size in (c["size_a"], c["size_b"])]
    return {"bytes": c["blocks"] * sum(p[0] for p in parts), "flops": c["blocks"] * sum(p[1] for p in parts)}


def tolerance(case: dict):
    """Whole numbers come from exact sums; BF16 results carry one rounding (2^-9); an FP32 sum in another order moves a
    BF16 rounding now and then, and with it an E4M3 or INT8 code of the layer behind it (one step of 2^-4 or 1/127)."""
    c, kind = case, case["kind"]
    if kind in ("quantize", "stem"):
        return "exact" if kind == "quantize" else {"differ": 1e-4}
    if kind == "int8_conv":
        return "exact" if c["out"] == "int8" else {"rel": 7e-3}
    return {"rel": 3e-2 if kind == "stack" else 8e-3 if kind == "block" else 7e-3}


# -- the same in 64 bits -----------------------------------------------------------------------------------------------


def _bf16(x: torch.Tensor) -> torch.Tensor:
    return x.to(BF16).double()


def _dequant(codes: torch.Tensor, exponent: torch.Tensor) -> torch.Tensor:
    x = codes.float().double()
    return (x.reshape(*x.shape[:-1], -1, 32) * torch.exp2(exponent.double())[..., None]).reshape(x.shape)


def _conv64(x: torch.Tensor, w: torch.Tensor, k: int, stride: int, ho: int, wo: int) -> torch.Tensor:
    """NHWC float64 convolution (pad k // 2), one product per tap."""
    cin, pad = x.shape[-1], k // 2
    x = F.pad(x, (0, 0, pad, pad, pad, pad))
    out = torch.zeros(x.shape[0] * ho * wo, w.shape[0], dtype=torch.float64, device=DEV)
    for t in range(k * k):
        ky, kx = divmod(t, k)
        rows = x[:, ky: ky + (ho - 1) * stride + 1: stride, kx: kx + (wo - 1) * stride + 1: stride].reshape(-1, cin)
        out += rows @ w[:, t * cin: (t + 1) * cin].t().contiguous()
    return out.reshape(x.shape[0], ho, wo, -1)


def _depthwise64(x: torch.Tensor, w: torch.Tensor, bias: torch.Tensor) -> torch.Tensor:
    """NHWC depthwise 5x5 (pad 2), ``w`` ``[25, C]``."""
    h, width = x.shape[1:3]
    x = F.pad(x.double(), (0, 0, 2, 2, 2, 2))
    out = bias.double().expand(x.shape[0], h, width, -1).clone()
    for t in range(25):
        out += x[:, t // 5: t // 5 + h, t % 5: t % 5 + width] * w[t].double()
    return out


def _exact_conv(c: dict, s: dict) -> torch.Tensor | None:
    args, kwargs = s["args"], s["kwargs"]
    if c["out"] == "int8":
        return None  # whole numbers: compared as they are
    if c["kind"] == "int8_conv":
        x, w, a_scale, w_scale, bias = args[:5]
        y = _conv64(x.double(), w.double(), c["k"], c["stride"], *_out_hw(c)) * (a_scale.double() * w_scale.double())
    else:
        x, expo, w, w_expo, bias = args[:5]
        y = _conv64(_dequant(x, expo), _dequant(w, w_expo), c["k"], c["stride"], *_out_hw(c))
    y = y + bias.double()
    if c.get("gelu"):
        y = F.gelu(_bf16(y))
    if c["residual"]:
        y = _bf16(y) + kwargs["residual"].double()
    if c["relu"]:
        y = y.relu()
    if c["out"] == "e4m3":
        y = _dequant(_e4m3(_bf16(y), kwargs["out_exponent"]), torch.zeros_like(kwargs["out_exponent"]))
    return y


def _exact_block(c: dict, s: dict) -> torch.Tensor:
    block, x = s["block"], s["x"]
    y = F.gelu(_bf16(_depthwise64(x, block.dw_weight, block.dw_bias)))

    def requantize(v, scale):
        if c["preset"] == "mxfp8":
            return _dequant(_e4m3(_bf16(v), scale), scale)
        return (_bf16(v) / scale.double()).round().clamp(-127, 127) * scale.double()

    if c["preset"] == "mxfp8":
        w1, w2 = (_dequant(w.values, w.scale_exponent) for w in (block.w1, block.w2))
    else:
        w1, w2 = block.w1_q.double() * block.w1_s.double()[:, None], block.w2_q.double() * block.w2_s.double()[:, None]
    rows = requantize(y, block.in_scale).reshape(-1, c["c"])
    hidden = F.gelu(_bf16(rows @ w1.t().contiguous() + block.b1.double()))
    y = requantize(hidden, block.hidden_scale) @ w2.t().contiguous() + block.b2.double()
    return _bf16(y).reshape(x.shape) + x.double()


def _exact_dwpw(c: dict, s: dict) -> torch.Tensor:
    x, dw_w, dw_b, w, *rest = s["args"]
    y = _depthwise64(x.permute(0, 2, 3, 1), dw_w, dw_b).relu().reshape(-1, c["c"])
    if c["format"] == "bf16":
        y, w = _bf16(y), w.double()
    elif c["format"] == "int8":
        w_scale, scale = rest[0].double(), rest[2].double()
        y, w = (_bf16(y) / scale).round().clamp(-127, 127) * scale, w.double() * w_scale[:, None]
    else:
        e = _exponent(y.reshape(-1, c["c"] // 32, 32).amax(dim=-1))
        y, w = _dequant(_e4m3(y, e), e), _dequant(w, (rest[1].view(torch.uint8).to(torch.int16) - 127).to(torch.int8))
    bias = rest[0] if c["format"] == "bf16" else rest[1] if c["format"] == "int8" else rest[2]
    out = y @ w.t().contiguous() + bias.double()
    return out.reshape(c["b"], c["h"], c["w"], -1).permute(0, 3, 1, 2)


def exact(case: dict, seed: int):
    c, kind = case, case["kind"]
    if kind == "stack" or kind == "stem":
        return None  # the stack: eight layers of codes behind each other; the stem: whole numbers
    s = prepare(case, seed)
    if kind in ("int8_conv", "mxfp8_conv"):
        return _exact_conv(c, s)
    if kind == "quantize":
        x, scale = s["args"]
        return _dequant(_e4m3(x.double(), scale), torch.zeros_like(scale)) if c["format"] == "mxfp8" else None
    return _exact_block(c, s) if kind == "block" else _exact_dwpw(c, s)
