"""The host path of the synchronous calls: uploads and downloads through the
context's pinned area, and the kept postprocess buffer.

Outputs of one piece, of a partial last piece and of more pieces than the area
has slots come back as the device holds them (the same model through the image
path, and twice in a row); a bad input is refused after its transfer was
queued and leaves the next call right; and calls of db_postprocess of growing
and shrinking sizes, which share one buffer, agree with a fresh context.
"""

import ctypes

import numpy as np
import pytest

import ppocr_hip
import seeded
from helpers import model_path, quad_corners

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    g = ppocr_hip.Gpu(0)
    yield g
    g.close()


# Map values: 2048 (below one piece), 73 728 (a piece and a tail), 1 105 920
# (five slots of 262 144 and less: the area wraps).
@pytest.mark.parametrize("shape", [(1, 3, 32, 64), (2, 3, 128, 288), (5, 3, 288, 768)])
def test_host_and_image_calls_agree(gpu, shape):
    n, _, h, w = shape
    rgb = seeded.seeded_rgb(h * n, w, 5, "blocks")
    x = np.stack([seeded.normalize_identity(rgb[i * h:(i + 1) * h], True) for i in range(n)])
    det = ppocr_hip.Detector.load(gpu, model_path("det", "tiny"), "tiny", shape)
    image = gpu.upload_rgb(rgb)
    quads = np.stack([quad_corners(0, i * h, w, (i + 1) * h) for i in range(n)])
    first = det.forward(x).array()
    assert first.shape == (n, 1, h, w) and np.isfinite(first).all() and first.std() > 0
    assert np.array_equal(first, det.forward(x).array())
    assert np.array_equal(first, det.forward_image(image, quads).array())
    det.close()


@pytest.mark.parametrize("at", [0, 12345, -1])
def test_non_finite_input_is_refused(gpu, at):
    shape = (1, 3, 160, 320)
    x = seeded.seeded_batch(1, 160, 320, 4)
    det = ppocr_hip.Detector.load(gpu, model_path("det", "tiny"), "tiny", shape)
    want = det.forward(x).array()
    for bad_value in (np.nan, np.inf, -np.inf):
        bad = x.copy()
        bad.reshape(-1)[at] = bad_value
        with pytest.raises(ppocr_hip.GpuError) as e:
            det.forward(bad)
        assert e.value.kind == "InvalidInput"
        with pytest.raises(ppocr_hip.GpuError) as e:
            det.detect(bad, [(320, 160, 320, 160)])
        assert e.value.kind == "InvalidInput"
        assert np.array_equal(det.forward(x).array(), want)
    det.close()


def test_postprocess_buffer_is_shared_by_sizes(gpu):
    rng = np.random.default_rng(8)

    def maps(n, h, w):
        m = rng.uniform(0.0, 0.1, (n, h, w)).astype(np.float32)
        for i in range(n):
            for y in range(3, h - 8, 12):
                m[i, y:y + 4, 5:5 + 9 + 3 * i] = 0.9
        return m

    for n, h, w in [(1, 64, 96), (4, 320, 320), (1, 32, 32), (2, 64, 96)]:
        m = maps(n, h, w)
        t = [(w, h, w, h)] * n
        other = ppocr_hip.Gpu(0)
        want = other.db_postprocess(m, t)
        got = gpu.db_postprocess(m, t)
        other.close()
        assert [len(g) for g in got] == [len(v) for v in want]
        for g, v in zip(got, want):
            for a, b in zip(g, v):
                assert a.score == b.score and np.array_equal(a.polygon, b.polygon)
        with pytest.raises(ppocr_hip.GpuError):
            gpu.db_postprocess(m, [(0, h, w, h)] * n)


# Maps go up by copy kernels: 16-byte lanes where the size allows, else 4-byte
# ones; whole and partial pieces of 2^17 values; 2^20 - 1 values, the most
# below the pinned slots' 4 MiB that has a remainder, and more (no pinned
# area).  A block of its own value at both ends of every map and of every
# piece (scores are means of equal values: exact up to one rounding).
@pytest.mark.parametrize("n,h,w", [(1, 33, 35), (3, 35, 61), (1, 256, 512), (1, 257, 511), (2, 701, 703),
                                   (1, 1023, 1025), (1, 1024, 1024), (1, 1027, 1029)])
def test_maps_arrive_whole(gpu, n, h, w):
    m = np.zeros((n, h, w), np.float32)
    rows = {0, h - 4} | {p // w for p in range(0, h * w, 1 << 17) if p // w < h - 12}  # blocks apart
    want = [[] for _ in range(n)]
    for i in range(n):
        for k, r in enumerate(sorted(rows)):
            for j, x in enumerate((0, w - 12)):
                v = np.float32(0.6 + 0.005 * (2 * k + j) + 0.1 * i)
                m[i, r:r + 4, x:x + 12] = v
                want[i].append(float(v))
    got = gpu.db_postprocess(m, [(w, h, w, h)] * n)
    for g, v in zip(got, want):
        assert np.allclose(sorted(d.score for d in g), sorted(v), atol=1e-6)


def test_a_bad_input_is_refused_first(gpu):
    """A non-finite input is what is reported also where the output buffer is
    too small or the transforms are missing."""
    shape = (1, 3, 64, 96)
    x = seeded.seeded_batch(1, 64, 96, 4)
    det = ppocr_hip.Detector.load(gpu, model_path("det", "tiny"), "tiny", shape)
    lib = ppocr_hip.lib()
    out = np.empty(det.output_len, np.float32)
    F = ctypes.POINTER(ctypes.c_float)

    def forward(values, cap):
        code = lib.ppocr_hip_forward(det.handle, values.ctypes.data_as(F), values.size, out.ctypes.data_as(F), cap)
        return code, lib.ppocr_hip_last_error().decode() if code else ""

    def detect(values):
        counts, total = (ctypes.c_size_t * 1)(), ctypes.c_size_t()
        code = lib.ppocr_hip_detect(det.handle, values.ctypes.data_as(F), values.size, None, None, None, 0, counts,
                                    ctypes.byref(total))
        return code, lib.ppocr_hip_last_error().decode() if code else ""

    bad = x.copy()
    bad.reshape(-1)[77] = np.nan
    assert "capacity" in forward(x, out.size - 1)[1]
    assert "non-finite" in forward(bad, out.size - 1)[1]
    assert "transforms" in detect(x)[1]
    assert "non-finite" in detect(bad)[1]
    assert forward(x, out.size)[0] == 0
    det.close()
