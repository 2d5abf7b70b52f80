"""The C entry points as ``torch.library`` ops (namespace ``flashim_amd``), so ``torch.compile`` traces the HIP impls
instead of breaking its graph at every call into the library (the pattern of FlashIM's CUDA backend,
``flashim/backends/cuda/conv.py:55-76, 148-161``).

The ops are defined and implemented in C++ (``csrc/torch_ops.cpp``: outputs from torch's caching allocator, one C call on
the current stream, an exception on a nonzero status, :class:`flashim_amd._lib.UnsupportedShape` for 99), registered when
``libflashim_amd_torch.so`` is loaded; their fakes, which return empty outputs of the same shape, dtype and device, are here. Arguments arrive normalized by the impls in
:mod:`flashim_amd.backends.hip` (dtypes, contiguity, devices): the bodies only read pointers, sizes and strides.
"""

from __future__ import annotations

import logging
import threading
from collections.abc import Callable

import torch

from flashim_amd._build import TORCH_LIBRARY

logger = logging.getLogger(__name__)

NS = "flashim_amd"
BLOCK = 32
DW_MX_DYNAMIC, DW_INT8, DW_BF16, DW_MX_STATIC = 0, 1, 2, 3
_DW_OUT_DTYPE = {DW_INT8: torch.int8, DW_BF16: torch.bfloat16, DW_MX_STATIC: torch.uint8}

_FAKES: dict[str, Callable] = {}
_OVERLOADS: dict[str, Callable] = {}
_lock = threading.Lock()


def load() -> None:
    """Load the op library and register the fakes, once. Raises if it has not been built."""
    with _lock:
        if _OVERLOADS:
            return
        if not TORCH_LIBRARY.is_file():
            raise RuntimeError(f"flashim_amd op library missing at {TORCH_LIBRARY}: build it with "
                               "`python -m flashim_amd._build`")
        torch.ops.load_library(str(TORCH_LIBRARY))
        loaded = {}
        for name, fake in _FAKES.items():
            torch.library.register_fake(f"{NS}::{name}", fake)
            loaded[name] = getattr(getattr(torch.ops, NS), name).default
        _OVERLOADS.update(loaded)


def _op(name: str) -> Callable:
    """The op as a function that loads the library on first use."""

    def call(*args, **kwargs):
        if name not in _OVERLOADS:
            load()
        return _OVERLOADS[name](*args, **kwargs)

    call.__name__ = name
    return call


def _fake(fn: Callable) -> Callable:
    """Register ``fn`` as the fake of the op of its name and return the op."""
    _FAKES[fn.__name__] = fn
    op = _op(fn.__name__)
    op.__doc__ = fn.__doc__
    return op


def conv_out_hw(h: int, w: int, kh: int, kw: int, sh: int, sw: int, ph: int, pw: int, dh: int, dw: int):
    return (h + 2 * ph - dh * (kh - 1) - 1) // sh + 1, (w + 2 * pw - dw * (kw - 1) - 1) // sw + 1


# -- quantizers ------------------------------------------------------------------------------------------------------


@_fake
def quantize_mxfp8(value, exponent, padded):
    return value.new_empty((*value.shape[:-1], padded), dtype=torch.uint8)


@_fake
def gelu_quantize_mxfp8(value, exponent, padded, input_bias, tanh=False):
    return value.new_empty((*value.shape[:-1], padded), dtype=torch.uint8)


@_fake
def quantize_int8(value, scale, channel_scale):
    return value.new_empty(value.shape, dtype=torch.int8)


@_fake
def gelu_quantize_int8(value, scale, tanh=False):
    return value.new_empty(value.shape, dtype=torch.int8)


@_fake
def quantize_mxfp8_dynamic(value, swizzled):
    """``[rows, K]`` -> E4M3 codes (``uint8``) and either int8 exponents ``[rows, K/32]`` or the swizzled E8M0 bytes."""
    rows, cols = value.shape
    groups = cols // BLOCK
    if swizzled:
        return (value.new_empty((rows, cols), dtype=torch.uint8),
                value.new_empty((-(-rows // 128) * 128 * -(-groups // 4) * 4,), dtype=torch.uint8))
    return value.new_empty((rows, cols), dtype=torch.uint8), value.new_empty((rows, groups), dtype=torch.int8)


@_fake
def quantize_int8_rows(value, reciprocal):
    rows, k = value.shape
    return value.new_empty((rows, k), dtype=torch.int8), value.new_empty((rows,), dtype=torch.float32)


@_fake
def calibrate_block32(matrix):
    return matrix.new_empty((-(-matrix.shape[1] // BLOCK),), dtype=torch.int8)


# -- implicit-GEMM convolutions and GEMMs ----------------------------------------------------------------------------


@_fake
def int8_conv2d(x, weight, a_scale, w_scale, bias, kh, kw, sh, sw, ph, pw, dh, dw, relu, gelu, residual, out_scale):
    b, h, w, _ = x.shape
    ho, wo = conv_out_hw(h, w, kh, kw, sh, sw, ph, pw, dh, dw)
    return x.new_empty((b, ho, wo, weight.shape[0]), dtype=torch.int8 if out_scale is not None else torch.bfloat16)


@_fake
def int8_conv2d_maxpool(x, weight, a_scale, w_scale, bias, kh, kw, sh, sw, ph, pw, dh, dw, relu, out_scale):
    b, h, w, _ = x.shape
    ho, wo = conv_out_hw(h, w, kh, kw, sh, sw, ph, pw, dh, dw)
    cout = weight.shape[0]
    return (x.new_empty((b, ho, wo, cout), dtype=torch.bfloat16),
            x.new_empty((b, ho // 2, wo // 2, cout), dtype=torch.int8))


@_fake
def mxfp8_conv2d(x, channel_exponent, weight, weight_exponent, bias, kh, kw, sh, sw, ph, pw, dh, dw, relu, gelu,
                 residual, out_exponent):
    """``x`` / ``weight``: E4M3 tensors or their ``uint8`` views; E4M3 output (``uint8``) with ``out_exponent``."""
    b, h, w, _ = x.shape
    ho, wo = conv_out_hw(h, w, kh, kw, sh, sw, ph, pw, dh, dw)
    return x.new_empty((b, ho, wo, weight.shape[0]),
                       dtype=torch.uint8 if out_exponent is not None else torch.bfloat16)


@_fake
def int8_linear(a, weight, a_scale, w_scale, bias, relu, gelu, residual):
    """``a_scale``: one value, or ``[M]`` per-row scales."""
    return a.new_empty((a.shape[0], weight.shape[0]), dtype=torch.bfloat16)


@_fake
def int8_linear_quantize_(a, weight, a_scale, w_scale, bias, out_scale, out):
    """Writes the INT8 result into ``out`` (``[M, N]``, unit column stride, any row stride)."""
    return None


@_fake
def mxfp8_scaled_mm(a, a_scale_swizzled, weight, weight_exponent, bias, weight_scale_e8m0=False):
    """``a [M, K]`` / ``weight [N, K]``: ``uint8`` views of E4M3; ``a_scale_swizzled`` ``uint8`` E8M0 bytes;
    ``weight_exponent`` ``[N, K/32]`` int8 exponents, or (``weight_scale_e8m0``) their E8M0 bytes."""
    return a.new_empty((a.shape[0], weight.shape[0]), dtype=torch.bfloat16)


@_fake
def im2col_gather(x, kh, kw, sh, sw, ph, pw, dh, dw):
    """``x``: ``uint8`` ``[B, H, W, C]`` -> ``uint8`` ``[B*Ho*Wo, kh*kw*C]``."""
    b, h, w, c = x.shape
    ho, wo = conv_out_hw(h, w, kh, kw, sh, sw, ph, pw, dh, dw)
    return x.new_empty((b * ho * wo, kh * kw * c), dtype=torch.uint8)


@_fake
def refiner_mlp(kind, semantics, x, x_scale, w1, w1_scale, b1, h_scale, w2, w2_scale, b2, residual):
    """The fused 64 -> 256 -> 64 MLP over ``x`` (INT8 or E4M3) ``[rows, 64]`` -> BF16 ``[rows, 64]``."""
    return x.new_empty((x.shape[0], w2.shape[0]), dtype=torch.bfloat16)


# -- depthwise producers and the one-kernel refiner block ------------------------------------------------------------


@_fake
def depthwise5x5(x, weight, bias, act, mode, scale, exponent):
    """``x`` BF16 NHWC ``[B, H, W, C]`` -> ``[B*H*W, C]``: INT8 (mode 1), BF16 (2) or E4M3 codes (3, ``uint8``)."""
    b, h, w, c = x.shape
    return x.new_empty((b * h * w, c), dtype=_DW_OUT_DTYPE[mode])


@_fake
def depthwise5x5_mx_dynamic(x, weight, bias):
    """``relu(dwconv5x5(x) + bias)`` -> dynamic MXFP8: E4M3 codes ``[B*H*W, C]`` and swizzled E8M0 bytes."""
    b, h, w, c = x.shape
    rows, groups = b * h * w, c // BLOCK
    return (x.new_empty((rows, c), dtype=torch.uint8),
            x.new_empty((-(-rows // 128) * 128 * -(-groups // 4) * 4,), dtype=torch.uint8))


@_fake
def depthwise5x5_relu_pointwise_mxfp8(x, dw_weight, dw_bias, pw_weight, pw_e8m0, pw_bias):
    """The one-kernel MXFP8 block at C = N = 128: ``x`` BF16 NHWC -> BF16 NHWC ``[B, H, W, N]``."""
    b, h, w, _ = x.shape
    return x.new_empty((b, h, w, pw_weight.shape[0]), dtype=torch.bfloat16)


@_fake
def depthwise5x5_relu_pointwise_int8(x, dw_weight, dw_bias, scale, pw_weight, pw_wscale, pw_bias):
    """The one-kernel INT8 block at C = N = 128: ``x`` BF16 NHWC -> BF16 NHWC ``[B, H, W, N]``; ``scale`` the static
    activation scale (FP32, one value), ``pw_wscale`` FP32 ``[N]``."""
    b, h, w, _ = x.shape
    return x.new_empty((b, h, w, pw_weight.shape[0]), dtype=torch.bfloat16)


# -- the VGG stem and the BF16 pointwise GEMM ------------------------------------------------------------------------


@_fake
def conv3x3_small_cin_quantize_int8(x, packed, bias, scale):
    b, _, h, w = x.shape
    return x.new_empty((b, h, w, packed.shape[0]), dtype=torch.int8)


@_fake
def bias_relu_quantize_int8(raw, bias, scale):
    b, c, h, w = raw.shape
    return raw.new_empty((b, h, w, c), dtype=torch.int8)


@_fake
def pointwise_bf16(x, weight, bias):
    """``x`` BF16 ``[M, K]`` times ``weight`` BF16 ``[N, K]`` transposed, plus FP32 or BF16 ``bias`` -> BF16 ``[M, N]``."""
    return x.new_empty((x.shape[0], weight.shape[0]), dtype=torch.bfloat16)


# ``torch.ops.flashim_amd`` is there on import. A library that is built later is loaded on first use, and so is one that
# does not load now (built against another torch, a missing HIP runtime): the first op raises the loader's error.
if TORCH_LIBRARY.is_file():
    try:
        load()
    except OSError as error:
        logger.warning("%s does not load: %s", TORCH_LIBRARY, error)
