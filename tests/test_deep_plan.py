"""The deep convolution kernel's planner (csrc/deep_plan.hip) on the CPU, for 256 CUs: the shapes of the GPU tests reach
every tile that is compiled, so a changed constant that moves one to another tile shows here."""

import re
from pathlib import Path

import pytest

from tests.test_gpu_deep_conv import INT8_SHAPES, INT8_TILES, MX_SHAPES, MX_TILES, deep_plan

CSRC = Path(__file__).resolve().parents[1] / "flashim_amd" / "csrc"
TILES = {"int8": INT8_TILES, "mxfp8": MX_TILES}


@pytest.mark.parametrize("quantized", [False, True])
@pytest.mark.parametrize("kind", TILES)
def test_planner_reaches_every_tile(kind, quantized):
    for tile, shape in TILES[kind].items():
        for residual in (False, True):
            assert deep_plan(kind, shape, quantized, residual) == tile, (shape, residual)
        b, h, w, _, cout, k, stride, pad, dilation = shape
        rows = b * ((h + 2 * pad - dilation * (k - 1) - 1) // stride + 1) * (
            (w + 2 * pad - dilation * (k - 1) - 1) // stride + 1)
        assert rows % (4 // tile[0] * tile[1] * 32) and cout % (64 * tile[0]), "rows and channels end inside a tile"


@pytest.mark.parametrize("kind, source", [("int8", "deep_int8.hip"), ("mxfp8", "deep_mx.hip")])
def test_every_compiled_tile_has_a_shape(kind, source):
    text = (CSRC / source).read_text()
    tiles = set()
    for wn, mbw, rag, two in re.findall(r"launch_deep_tile<\w+, OUT, (\d), (\d), (\w+)(, true)?>", text):
        for r in (0, 1) if rag == "RAG" else (0,):
            tiles.add((int(wn), int(mbw), r, int(bool(two))))
    assert tiles == set(TILES[kind])


def test_the_other_shapes_are_taken():
    for kind, shapes in (("int8", INT8_SHAPES), ("mxfp8", MX_SHAPES)):
        for shape in shapes:
            assert deep_plan(kind, shape, False, False)[0] != 0, shape


def test_planner_refuses_what_the_kernel_does_not_take():
    refused = [
        ("int8", (1, 64, 67, 196, 64, 3, 1, 1, 1), "64 channels out"),
        ("int8", (1, 64, 67, 32, 128, 3, 1, 1, 1), "fewer than 36 channels in"),
        ("int8", (1, 64, 67, 198, 128, 3, 1, 1, 1), "Cin % 4"),
        ("int8", (1, 64, 67, 196, 130, 3, 1, 1, 1), "Cout % 4"),
        ("int8", (1, 64, 67, 64, 128, 6, 1, 0, 1), "36 taps"),
        ("mxfp8", (1, 64, 67, 64, 100, 3, 1, 1, 1), "Cout % 16"),
        ("mxfp8", (1, 512, 512, 96, 256, 1, 1, 0, 1), "under 128 bytes of K"),
    ]
    for kind, shape, why in refused:
        assert deep_plan(kind, shape, False, False)[0] == 0, why
