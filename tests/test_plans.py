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
