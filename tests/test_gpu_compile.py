"""``torch.compile(fullgraph=True)`` traces the HIP impls (custom ops with fakes, flashim_amd.library) and gives the
eager result, the contract of FlashIM's tests/ops/test_depthwise_cuda.py:115-119. Each compiled function runs the op
through this package's dispatcher, as FlashIM's region compile would through its own."""

import pytest
import torch

from flashim_amd import _lib, ops, quant
from oracle import reference as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _same(a, b):
    if isinstance(a, (tuple, list)):
        return all(_same(x, y) for x, y in zip(a, b))
    if isinstance(a, quant.QuantizedTensor):
        return _same(a.values, b.values) and _same(a.scale_exponent, b.scale_exponent)
    if isinstance(a, quant.Int8Tensor):
        return _same(a.values, b.values)
    if a.dtype in (torch.float8_e4m3fn, torch.float8_e8m0fnu):
        a, b = a.view(torch.uint8), b.view(torch.uint8)
    return torch.equal(a, b)


def _check(fn, *args):
    torch._dynamo.reset()
    eager = fn(*args)
    compiled = torch.compile(fn, fullgraph=True)(*args)
    assert _same(compiled, eager)


def test_compile_convs():
    g = torch.Generator().manual_seed(0)
    x = torch.randint(-127, 127, (2, 20, 21, 64), dtype=torch.int8, generator=g).to(DEV)
    w = torch.randint(-127, 127, (96, 9 * 64), dtype=torch.int8, generator=g).to(DEV)
    a_s, w_s, b = torch.tensor(0.02, device=DEV), (torch.rand(96, generator=g) * 0.01).to(DEV), torch.randn(96).to(DEV)
    _check(lambda x: ops.int8_conv2d(x, w, a_s, w_s, b, 3, 3, 1, 1, 1, 1, 1, 1, relu=True), x)
    xb = torch.randn(2, 20, 21, 64, generator=g).to(torch.bfloat16).to(DEV)
    e = ref.calibrate_block32_exponent(xb.float().cpu()).to(DEV)
    wq = quant.QuantizedWeight.from_float((torch.randn(96, 9 * 64, generator=g) * 0.05).to(DEV))

    def mx_block(xb):
        q = ops.quantize_mxfp8(xb, e)
        return ops.mxfp8_conv2d(q.values, e, wq.values, wq.scale_exponent, b, 3, 3, 1, 1, 1, 1, 1, 1, gelu=True)

    _check(mx_block, xb)


def test_compile_quantizers():
    g = torch.Generator().manual_seed(1)
    xb = (torch.randn(2, 13, 17, 96, generator=g) * 3).to(torch.bfloat16).to(DEV)
    e = ref.calibrate_block32_exponent(xb.float().cpu()).to(DEV)
    s = torch.tensor(0.03, device=DEV)
    _check(lambda v: ops.quantize_mxfp8(v, e), xb)
    _check(lambda v: ops.quantize_int8(v, s), xb)
    _check(lambda v: ops.gelu_quantize(v, e), xb)
    _check(lambda v: ops.quantize_mxfp8(v.permute(0, 2, 3, 1), e), xb.permute(0, 3, 1, 2).contiguous())


def test_compile_depthwise_and_blocks():
    g = torch.Generator().manual_seed(2)
    c = 128
    x = (torch.randn(2, c, 24, 40, generator=g) * 2).to(torch.bfloat16).contiguous(
        memory_format=torch.channels_last).to(DEV)
    dw_w = (torch.randn(25, c, generator=g) * 0.3).to(torch.bfloat16).to(DEV)
    dw_b, pw_b = torch.randn(c, generator=g).to(DEV), torch.randn(c, generator=g).to(DEV)
    s = torch.tensor(0.03, device=DEV)
    _check(lambda v: ops.depthwise5x5_relu_mxfp8(v, dw_w, dw_b), x)
    _check(lambda v: ops.depthwise5x5_relu_int8(v, dw_w, dw_b, s), x)
    pw = quant.QuantizedWeight.from_float((torch.randn(c, c, generator=g) * 0.1).to(DEV))
    swz, e8 = quant.swizzle_scales(pw.scale_exponent), quant.exponent_to_e8m0(pw.scale_exponent)
    _check(lambda v: ops.depthwise5x5_relu_pointwise_mxfp8(v, dw_w, dw_b, pw.values, swz, e8, pw_b), x)
    w8 = torch.randint(-127, 128, (c, c), dtype=torch.int8, generator=g).to(DEV)
    ws = (torch.rand(c, generator=g) * 0.01 + 0.001).to(DEV)
    _check(lambda v: ops.depthwise5x5_relu_pointwise_int8(v, dw_w, dw_b, w8, ws, pw_b, s), x)
    pw16 = (torch.randn(c, c, generator=g) * 0.1).to(torch.bfloat16).to(DEV)
    _check(lambda v: ops.depthwise5x5_relu_pointwise(v, dw_w, dw_b, pw16, pw_b), x)


def test_backward_through_an_op_raises():
    x = torch.randn(1, 8, 8, 32, device=DEV).to(torch.bfloat16).requires_grad_()
    w, b = torch.randn(25, 32, device=DEV).to(torch.bfloat16), torch.randn(32, device=DEV)
    y = torch.ops.flashim_amd.depthwise5x5(x, w, b, 1, 2, None, None)
    with pytest.raises(RuntimeError, match="not implemented"):
        y.float().sum().backward()


def _zeros(*shape, dtype=torch.int8):
    return torch.zeros(shape, device=DEV, dtype=dtype)


GEO3 = (3, 3, 1, 1, 1, 1, 1, 1)
_F32, _BF16, _U8 = torch.float32, torch.bfloat16, torch.uint8
# op, its arguments with an input of the shape the op takes, the index of that input
RANKS = {
    "quantize_mxfp8_dynamic": lambda: [_zeros(32, 32, dtype=_F32), True],
    "quantize_int8_rows": lambda: [_zeros(32, 32, dtype=_F32), True],
    "calibrate_block32": lambda: [_zeros(32, 32, dtype=_F32)],
    "int8_conv2d": lambda: [_zeros(2, 8, 8, 32), _zeros(32, 288), _zeros(1, dtype=_F32), _zeros(32, dtype=_F32), None,
                            *GEO3, False, False, None, None],
    "int8_conv2d_maxpool": lambda: [_zeros(2, 8, 8, 32), _zeros(32, 288), _zeros(1, dtype=_F32),
                                    _zeros(32, dtype=_F32), None, *GEO3, False, torch.ones(1, device=DEV)],
    "mxfp8_conv2d": lambda: [_zeros(2, 8, 8, 32, dtype=_U8), _zeros(1), _zeros(32, 288, dtype=_U8), _zeros(32, 9), None,
                             *GEO3, False, False, None, None],
    "int8_linear": lambda: [_zeros(32, 32), _zeros(32, 32), _zeros(1, dtype=_F32), _zeros(32, dtype=_F32), None, False,
                            False, None],
    "int8_linear_quantize_": lambda: [_zeros(32, 32), _zeros(32, 32), _zeros(1, dtype=_F32), _zeros(32, dtype=_F32),
                                      None, torch.ones(1, device=DEV), _zeros(32, 32)],
    "mxfp8_scaled_mm": lambda: [_zeros(32, 32, dtype=_U8), _zeros(512, dtype=_U8), _zeros(32, 32, dtype=_U8),
                                _zeros(32, 1), None],
    "im2col_gather": lambda: [_zeros(2, 8, 8, 32, dtype=_U8), *GEO3],
    "refiner_mlp": lambda: [0, 0, _zeros(32, 64), _zeros(1, dtype=_F32), _zeros(256, 64), _zeros(256, dtype=_F32), None,
                            torch.ones(1, device=DEV), _zeros(64, 256), _zeros(64, dtype=_F32), None, None],
    "depthwise5x5": lambda: [_zeros(2, 8, 8, 32, dtype=_BF16), _zeros(25, 32, dtype=_BF16), _zeros(32, dtype=_F32), 0, 2,
                             None, None],
    "depthwise5x5_mx_dynamic": lambda: [_zeros(2, 8, 8, 32, dtype=_BF16), _zeros(25, 32, dtype=_BF16),
                                        _zeros(32, dtype=_F32)],
    "conv3x3_small_cin_quantize_int8": lambda: [_zeros(2, 3, 8, 8, dtype=_BF16), _zeros(16, 32, dtype=_BF16),
                                                _zeros(16, dtype=_F32), torch.ones(1, device=DEV)],
    "bias_relu_quantize_int8": lambda: [_zeros(2, 16, 8, 8, dtype=_BF16), _zeros(16, dtype=_F32),
                                        torch.ones(1, device=DEV)],
    "pointwise_bf16": lambda: [_zeros(32, 32, dtype=_BF16), _zeros(32, 32, dtype=_BF16), None],
}


@pytest.mark.parametrize("name", RANKS)
def test_ops_refuse_inputs_of_another_rank(name):
    """The ops read leading sizes only, so an input of one dimension more would be taken for its first dimensions (a
    [2, 32, 32] as [2, 32]): they raise ValueError before anything is allocated or launched."""
    op = getattr(torch.ops.flashim_amd, name)
    args = RANKS[name]()
    op(*args)
    at = 2 if name == "refiner_mlp" else 0
    for wrong in (args[at].unsqueeze(0), args[at][0]):
        with pytest.raises(ValueError, match="dimensions"):
            op(*args[:at], wrong, *args[at + 1:])


def test_int8_rows_of_a_3d_tensor_are_refused():
    for fn in (quant.quantize_int8_rows, quant.weight_scales_and_values, quant.quantize_dynamic_2d):
        with pytest.raises(ValueError):
            fn(torch.randn(2, 32, 32, device=DEV))


def test_conv_residual_of_five_dimensions_is_refused():
    args = RANKS["int8_conv2d"]()
    with pytest.raises(IndexError):
        torch.ops.flashim_amd.int8_conv2d(*args[:-2], _zeros(1, 2, 8, 8, 32, dtype=_BF16), None)


def test_unsupported_shapes_raise_their_own_type_compiled_too():
    """The BF16 pointwise kernel takes up to 128 output channels: status 99 from the library."""
    x, weight = _zeros(32, 32, dtype=_BF16), _zeros(144, 32, dtype=_BF16)
    op = torch.ops.flashim_amd.pointwise_bf16
    torch._dynamo.reset()
    for fn in (op, torch.compile(lambda x: op(x, weight, None), fullgraph=True)):
        with pytest.raises(_lib.UnsupportedShape, match="no HIP kernel"):
            fn(x, weight, None) if fn is op else fn(x)
