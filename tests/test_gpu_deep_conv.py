"""The deep convolution kernel (csrc/deep.h) at the edges of its tiles, K walk and channel counts, against the general
path: a zero FP32 residual sends the same call to the 128-row kernels (the residual of the deep kernel is BF16), which
the oracle tests cover. INT8 sums are exact, so the results are equal; MXFP8 sums in another order move a BF16 rounding
now and then (relative L2 1e-3, the MXFP8 convs' bar against the oracle). Every launch's plan is read back, so a row that
the deep kernel does not take fails."""

import ctypes

import pytest
import torch

from flashim_amd import _lib, ops, quant

pytestmark = pytest.mark.gpu

# b, h, w, cin, cout, k, stride, pad, dilation: tile remainders in rows and channels, K tails, several taps per step
# (Cin 36, 64, 96), no padding, stride and dilation 2, a filter of 25 taps, one row of pixels
INT8_SHAPES = [
    (1, 64, 67, 196, 128, 3, 1, 1, 1), (1, 33, 41, 36, 68, 3, 1, 1, 1), (2, 37, 45, 100, 196, 3, 2, 1, 1),
    (1, 61, 59, 68, 100, 5, 1, 2, 1), (1, 50, 52, 196, 512, 1, 1, 0, 1), (1, 1, 700, 132, 132, 3, 1, 1, 1),
    (1, 112, 150, 512, 512, 3, 1, 1, 1), (2, 90, 101, 160, 272, 3, 1, 1, 1), (1, 131, 127, 256, 144, 3, 1, 0, 1),
    (1, 130, 140, 192, 192, 3, 1, 2, 2), (2, 257, 255, 96, 128, 5, 2, 2, 1), (1, 165, 198, 64, 68, 3, 1, 1, 1),
]
MX_SHAPES = [
    (1, 224, 300, 256, 256, 3, 1, 1, 1), (3, 97, 57, 160, 128, 3, 1, 1, 1), (1, 108, 157, 512, 160, 3, 1, 1, 1),
    (1, 148, 290, 96, 256, 5, 1, 2, 1), (1, 85, 144, 192, 384, 5, 1, 2, 1), (2, 131, 140, 224, 112, 3, 1, 0, 1),
    (1, 130, 140, 192, 192, 3, 1, 2, 2), (2, 64, 67, 320, 160, 5, 1, 2, 1), (2, 249, 251, 160, 96, 3, 2, 1, 1),
]
# Every tile that is compiled, as (wavefronts across the columns, 32-row blocks per wavefront, ragged channels, two
# workgroups per CU), and the smallest launch found that the planner gives it on 256 CUs, whatever the output format; rows
# and channels end inside a tile
INT8_TILES = {
    (2, 2, 0, 0): (1, 11, 9, 48, 224, 5, 1, 0, 2), (2, 2, 0, 1): (3, 73, 80, 48, 144, 3, 1, 0, 1),
    (2, 3, 0, 0): (1, 143, 119, 144, 144, 3, 1, 0, 1), (2, 4, 0, 0): (2, 376, 33, 288, 144, 3, 1, 1, 1),
    (2, 5, 0, 0): (1, 76, 449, 48, 144, 3, 1, 0, 1), (4, 4, 0, 0): (1, 69, 93, 288, 1216, 3, 1, 2, 2),
    (4, 5, 0, 0): (1, 324, 104, 64, 144, 3, 1, 0, 1), (4, 6, 0, 0): (3, 48, 285, 48, 144, 3, 1, 1, 1),
    (4, 7, 0, 0): (2, 67, 369, 48, 144, 3, 1, 1, 1), (4, 8, 0, 0): (3, 38, 254, 48, 272, 5, 1, 2, 1),
    (2, 2, 1, 0): (1, 10, 9, 36, 312, 5, 2, 0, 2), (2, 2, 1, 1): (1, 8, 10, 44, 88, 3, 2, 0, 1),
    (2, 3, 1, 0): (1, 323, 204, 196, 136, 3, 2, 2, 2), (2, 4, 1, 0): (3, 314, 53, 284, 68, 5, 1, 4, 2),
    (2, 5, 1, 0): (2, 375, 47, 36, 132, 3, 1, 0, 1), (4, 4, 1, 0): (2, 310, 41, 164, 132, 5, 1, 2, 1),
    (4, 5, 1, 0): (3, 24, 499, 52, 132, 3, 1, 0, 1), (4, 6, 1, 0): (3, 118, 124, 52, 132, 3, 1, 0, 2),
    (4, 7, 1, 0): (1, 111, 492, 36, 140, 5, 1, 2, 1), (4, 8, 1, 0): (3, 234, 84, 84, 132, 5, 1, 2, 1),
}
MX_TILES = {
    (2, 2, 0, 0): (3, 9, 9, 64, 96, 5, 1, 0, 2), (2, 2, 0, 1): (1, 482, 51, 64, 160, 3, 1, 1, 1),
    (2, 3, 0, 0): (1, 482, 34, 64, 160, 3, 1, 1, 1), (2, 4, 0, 0): (3, 152, 234, 128, 160, 3, 2, 1, 1),
    (2, 5, 0, 0): (1, 404, 215, 64, 288, 3, 2, 2, 2), (4, 4, 0, 0): (3, 107, 39, 128, 672, 3, 1, 0, 2),
    (4, 5, 0, 0): (1, 241, 136, 64, 160, 3, 1, 1, 1), (4, 6, 0, 0): (2, 52, 394, 64, 160, 3, 1, 1, 1),
    (4, 7, 0, 0): (1, 243, 112, 64, 288, 3, 1, 1, 1), (4, 8, 0, 0): (2, 424, 36, 64, 288, 3, 1, 0, 1),
}
DEV = "cuda"


def deep_plan(kind, shape, quantized, residual):
    """The tile the deep kernel takes this launch on (all zeros: not taken); none of the shapes here is one that the
    kernels asked before it take (3x3 at Cin = 128 and stride 1, and 1x1 at Cin % 128 == 0)."""
    b, h, w, cin, cout, k, stride, pad, dilation = shape
    assert not (k == 3 and cin == 128 and stride == dilation == 1) and not (k == 1 and cin % 128 == 0)
    plan = (ctypes.c_int * 4)()
    _lib.probe_call("fim_test_deep_plan", 0 if kind == "int8" else 1, b, h, w, cin, cout,
                    *_geometry(k, stride, pad, dilation), 0 if not quantized else 1 if kind == "int8" else 2, int(residual),
                    ctypes.addressof(plan))
    return tuple(plan)


def _geometry(k, stride, pad, dilation):
    return (k, k, stride, stride, pad, pad, dilation, dilation)


def _out_hw(h, w, k, stride, pad, dilation):
    return tuple((n + 2 * pad - dilation * (k - 1) - 1) // stride + 1 for n in (h, w))


def _check_int8(shape, out_int8, residual, relu=True, with_bias=True):
    assert deep_plan("int8", shape, out_int8, residual)[0] != 0
    b, h, w, cin, cout, k, stride, pad, dilation = shape
    g = torch.Generator(device=DEV).manual_seed(sum(shape))
    x = torch.randint(-127, 128, (b, h, w, cin), dtype=torch.int8, generator=g, device=DEV)
    weight = torch.randint(-127, 128, (cout, k * k * cin), dtype=torch.int8, generator=g, device=DEV)
    w_scale = torch.rand(cout, generator=g, device=DEV) * 0.01 + 0.001
    a_scale = torch.tensor(0.017, device=DEV)
    bias = torch.randn(cout, generator=g, device=DEV).to(torch.bfloat16)
    res = torch.randn(b, *_out_hw(h, w, k, stride, pad, dilation), cout, generator=g, device=DEV).to(torch.bfloat16)
    kwargs = {"relu": relu, "out_scale": torch.tensor(0.8, device=DEV) if out_int8 else None}
    args = (x, weight, a_scale, w_scale, bias if with_bias else None, *_geometry(k, stride, pad, dilation))
    got = ops.int8_conv2d(*args, residual=res if residual else None, **kwargs)
    want = ops.int8_conv2d(*args, residual=res.float() if residual else torch.zeros_like(res, dtype=torch.float32),
                           **kwargs)
    assert torch.equal(got, want)


def _check_mxfp8(shape, out_e4m3, residual, relu=True, with_bias=True):
    assert deep_plan("mxfp8", shape, out_e4m3, residual)[0] != 0
    b, h, w, cin, cout, k, stride, pad, dilation = shape
    g = torch.Generator(device=DEV).manual_seed(sum(shape))
    act = torch.randn(b, h, w, cin, generator=g, device=DEV)
    act *= torch.exp(torch.randn(cin, generator=g, device=DEV))  # the blocks' exponents differ
    exponent = quant.calibrate_block32_exponent(act)
    x = ops.quantize_mxfp8(act, exponent).values
    scale = torch.exp(torch.randn(cout, k * k * cin // 32, 1, generator=g, device=DEV))
    weight = (torch.randn(cout, k * k * cin // 32, 32, generator=g, device=DEV) * 0.03 * scale).reshape(cout, -1)
    values, w_exponent = quant.quantize_dynamic_2d(weight)
    bias = torch.randn(cout, generator=g, device=DEV)
    res = torch.randn(b, *_out_hw(h, w, k, stride, pad, dilation), cout, generator=g, device=DEV).to(torch.bfloat16)
    out_exponent = torch.arange(cout // 32, device=DEV).to(torch.int8) % 3 - 4 if out_e4m3 else None
    args = (x, exponent, values, w_exponent, bias if with_bias else None, *_geometry(k, stride, pad, dilation))
    kwargs = {"relu": relu, "out_exponent": out_exponent}
    got = ops.mxfp8_conv2d(*args, residual=res if residual else None, **kwargs).float()
    want = ops.mxfp8_conv2d(*args, residual=res.float() if residual else torch.zeros_like(res, dtype=torch.float32),
                            **kwargs).float()
    # E4M3: a code moves by one step (2^-3 of its value) where its BF16 value moved across a rounding boundary: about one
    # in 2^5 of the moved BF16 values, themselves rarer than one in 10^3, so the same bar holds
    assert ((got - want).norm() / want.norm()).item() <= 1e-3


@pytest.mark.parametrize("residual", [False, True])
@pytest.mark.parametrize("out_int8", [False, True])
@pytest.mark.parametrize("shape", INT8_SHAPES)
def test_int8_deep_conv_matches_general_path(shape, out_int8, residual):
    _check_int8(shape, out_int8, residual)


@pytest.mark.parametrize("residual", [False, True])
@pytest.mark.parametrize("out_e4m3", [False, True])
@pytest.mark.parametrize("shape", MX_SHAPES)
def test_mxfp8_deep_conv_matches_general_path(shape, out_e4m3, residual):
    if out_e4m3 and shape[4] % 32:
        pytest.skip("E4M3 output needs whole 32-channel blocks")
    _check_mxfp8(shape, out_e4m3, residual)


@pytest.mark.parametrize("shape", [(2, 111, 177, 196, 320, 1, 1, 0, 1), (2, 208, 326, 68, 160, 3, 1, 1, 1),
                                   (2, 392, 214, 68, 224, 1, 1, 0, 1)])
@pytest.mark.parametrize("out_int8", [False, True])
def test_int8_deep_conv_two_workgroups_per_cu(shape, out_int8):
    """Several rounds of few K steps: 128 x 128 tiles, two workgroups per CU."""
    _check_int8(shape, out_int8, False)


# quantized output, residual, ReLU, bias
FORMS = [(False, False, True, True), (False, True, False, False), (True, False, False, True), (True, True, True, False)]


@pytest.mark.parametrize("quantized, residual, relu, bias", FORMS)
@pytest.mark.parametrize("tile", INT8_TILES)
def test_int8_deep_conv_tiles(tile, quantized, residual, relu, bias):
    assert deep_plan("int8", INT8_TILES[tile], quantized, residual) == tile
    _check_int8(INT8_TILES[tile], quantized, residual, relu, bias)


@pytest.mark.parametrize("quantized, residual, relu, bias", FORMS)
@pytest.mark.parametrize("tile", MX_TILES)
def test_mxfp8_deep_conv_tiles(tile, quantized, residual, relu, bias):
    assert deep_plan("mxfp8", MX_TILES[tile], quantized, residual) == tile
    _check_mxfp8(MX_TILES[tile], quantized, residual, relu, bias)
