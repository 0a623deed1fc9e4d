"""Plans as the host builds them (no GPU): what the arena gives the input and
which kernels the layers get, read through the test-only probe library."""

import ctypes

import pytest

from helpers import model_path
from test_conv_kernels_gpu import PROBE

SIZE_CODE = {"medium": 0, "small": 1, "tiny": 2}


def plan(kind, size, shape, bf16=False, greedy=False):
    """Ops of a plan as (name, kernel), whether its input is kept, and the
    bytes of its weight blob."""
    fn = ctypes.CDLL(str(PROBE)).ppocr_probe_plan
    fn.restype = ctypes.c_long
    fn.argtypes = [ctypes.c_char_p] + [ctypes.c_int] * 7 + [ctypes.c_char_p, ctypes.c_size_t]
    args = (str(model_path(kind, size)).encode(), 0 if kind == "det" else 1, SIZE_CODE[size], *shape, int(bf16),
            int(greedy))
    n = fn(*args, None, 0)
    assert n > 0, "plan could not be built"
    buf = ctypes.create_string_buffer(n)
    assert fn(*args, buf, n) == n
    lines = buf.value.decode().splitlines()
    ops = [tuple(line.split("\t")) for line in lines if "\t" in line]
    return ops, "input kept" in lines, int(lines[-1].split()[1])


@pytest.mark.parametrize("kind,size,shape,bf16", [
    ("det", "tiny", (1, 96, 160), False), ("det", "small", (2, 416, 736), False), ("det", "medium", (8, 416, 736), True),
    ("rec", "tiny", (64, 48, 320), False), ("rec", "medium", (16, 48, 320), True)])
def test_the_input_outlives_the_pass(kind, size, shape, bf16):
    """benchmark and profile replay a plan on an input that is uploaded once;
    an activation in its place would have the next replay run on that."""
    assert plan(kind, size, shape, bf16)[1]


# Layers that the split kernel measured slower on than the fp32 kernels, and
# neighbours of each in size, K or gate that it measured faster on.
@pytest.mark.parametrize("kind,size,shape,layer,split", [
    ("rec", "small", (6, 48, 500), "blocks.3.blocks.1.channel_conv1", False),  # gated K = 384, 864 64x32 tiles
    ("det", "small", (8, 416, 736), "blocks.3.blocks.1.channel_conv1", False),  # gated K = 384, 912
    ("det", "medium", (1, 416, 736), "blocks.2.blocks.1.channel_conv1", True),  # gated K = 512, 608
    ("rec", "medium", (1, 48, 1200), "blocks.2.blocks.1.channel_conv1", False),  # gated K = 512, 928
    ("rec", "medium", (1, 48, 320), "blocks.2.blocks.1.channel_conv1", True),  # gated K = 512, fewer
    ("rec", "medium", (16, 48, 320), "blocks.0.blocks.0.channel_conv2", False),  # K = 256, 960
    ("det", "small", (1, 160, 320), "blocks.1.blocks.1.channel_conv1", True),  # gated K = 96, 78
    ("rec", "small", (64, 48, 320), "blocks.0.blocks.0.channel_conv1", True),  # gated K = 96, 64x64
    ("det", "small", (8, 416, 736), "convolution.stem2b", False),  # K = 48, 24 columns
    ("det", "small", (8, 416, 736), "input_conv.0.pointwise_convolution", False),  # K = 96, 24 columns
    ("rec", "small", (64, 48, 320), "convolution.stem2a", True),  # K = 192, 24 columns
    ("det", "medium", (4, 416, 736), "path_aggregation_lateral_convolution.0.pointwise", False),  # K = 64, 64 columns
    ("det", "medium", (2, 416, 736), "convolution.stem4", True),  # K = 64, 128 columns
    ("det", "medium", (8, 416, 736), "conv_up+conv_final", True),  # K = 64, 256 columns
])
def test_layers_run_on_the_faster_kernel(kind, size, shape, layer, split):
    ops, _, _ = plan(kind, size, shape, greedy=kind == "rec")
    kernels = [k for n, k in ops if n.endswith(layer)]
    assert len(kernels) == 1
    assert kernels[0].startswith("conv_split" if split else "conv_gemm"), kernels


def test_a_level_with_its_own_launch_splits_k():
    """The largest level of the medium neck's long step runs on wider tiles
    than the others there: 299 of them, which K splits spread over the GPU."""
    ops = dict(plan("det", "medium", (2, 416, 736))[0])
    assert ops["model.neck.intraclass_blocks.0.long"] == "conv_split<128x32>+split_k3"
    assert ops["model.neck.intraclass_blocks.long.1"] == "conv_split<64x32>x3"


@pytest.mark.parametrize("kind,size,limit", [("det", "tiny", 3.1e6), ("rec", "medium", 183.5e6)])
def test_fused_layers_hold_no_split_weights(kind, size, limit):
    """The pairs of the tiny detector and the layer-norm linear layers of the
    medium recognizer read fp32 weights only (3.8 and 186.1 MB with both)."""
    assert plan(kind, size, (1, 416, 736) if kind == "det" else (1, 48, 320))[2] < limit
