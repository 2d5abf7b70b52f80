"""The deep convolution kernel (csrc/deep.h) at the edges of its tiles, K walk and channel counts, against the general
path: a zero FP32 residual sends the same call to the 128-row kernels (the residual of the deep kernel is BF16), which
the oracle tests cover. INT8 sums are exact, so the results are equal; MXFP8 sums in another order move a BF16 rounding
now and then (relative L2 1e-3, the MXFP8 convs' bar against the oracle)."""

import pytest
import torch

from flashim_amd import ops, quant

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
    (1, 130, 140, 192, 192, 3, 1, 2, 2), (1, 64, 67, 320, 128, 5, 1, 2, 1), (2, 249, 251, 160, 96, 3, 2, 1, 1),
]
DEV = "cuda"


def _geometry(k, stride, pad, dilation):
    return (k, k, stride, stride, pad, pad, dilation, dilation)


def _out_hw(h, w, k, stride, pad, dilation):
    return tuple((n + 2 * pad - dilation * (k - 1) - 1) // stride + 1 for n in (h, w))


@pytest.mark.parametrize("residual", [False, True])
@pytest.mark.parametrize("out_int8", [False, True])
@pytest.mark.parametrize("shape", INT8_SHAPES)
def test_int8_deep_conv_matches_general_path(shape, out_int8, residual):
    b, h, w, cin, cout, k, stride, pad, dilation = shape
    g = torch.Generator(device=DEV).manual_seed(sum(shape))
    x = torch.randint(-127, 128, (b, h, w, cin), dtype=torch.int8, generator=g, device=DEV)
    weight = torch.randint(-127, 128, (cout, k * k * cin), dtype=torch.int8, generator=g, device=DEV)
    w_scale = torch.rand(cout, generator=g, device=DEV) * 0.01 + 0.001
    a_scale = torch.tensor(0.017, device=DEV)
    bias = torch.randn(cout, generator=g, device=DEV).to(torch.bfloat16)
    res = torch.randn(b, *_out_hw(h, w, k, stride, pad, dilation), cout, generator=g, device=DEV).to(torch.bfloat16)
    kwargs = {"relu": True, "out_scale": torch.tensor(0.8, device=DEV) if out_int8 else None}
    args = (x, weight, a_scale, w_scale, bias, *_geometry(k, stride, pad, dilation))
    got = ops.int8_conv2d(*args, residual=res if residual else None, **kwargs)
    want = ops.int8_conv2d(*args, residual=res.float() if residual else torch.zeros_like(res, dtype=torch.float32),
                           **kwargs)
    assert torch.equal(got, want)


@pytest.mark.parametrize("residual", [False, True])
@pytest.mark.parametrize("out_e4m3", [False, True])
@pytest.mark.parametrize("shape", MX_SHAPES)
def test_mxfp8_deep_conv_matches_general_path(shape, out_e4m3, residual):
    b, h, w, cin, cout, k, stride, pad, dilation = shape
    if out_e4m3 and cout % 32:
        pytest.skip("E4M3 output needs whole 32-channel blocks")
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
    args = (x, exponent, values, w_exponent, bias, *_geometry(k, stride, pad, dilation))
    kwargs = {"relu": True, "out_exponent": out_exponent}
    got = ops.mxfp8_conv2d(*args, residual=res if residual else None, **kwargs).float()
    want = ops.mxfp8_conv2d(*args, residual=res.float() if residual else torch.zeros_like(res, dtype=torch.float32),
                            **kwargs).float()
    # E4M3: a code moves by one step (2^-3 of its value) where its BF16 value moved across a rounding boundary: about one
    # in 2^5 of the moved BF16 values, themselves rarer than one in 10^3, so the same bar holds
    assert ((got - want).norm() / want.norm()).item() <= 1e-3


@pytest.mark.parametrize("shape", [(2, 111, 177, 196, 320, 1, 1, 0, 1), (2, 208, 326, 68, 160, 3, 1, 1, 1),
                                   (2, 392, 214, 68, 224, 1, 1, 0, 1)])
@pytest.mark.parametrize("out_int8", [False, True])
def test_int8_deep_conv_two_workgroups_per_cu(shape, out_int8):
    """Several rounds of few K steps: 128 x 128 tiles, two workgroups per CU."""
    test_int8_deep_conv_matches_general_path(shape, out_int8, False)
