"""fp32 convolutions on the bf16 matrix cores (conv_split_kernel).

Every fp32 operand is split into three bf16 parts and a product takes six of
the nine partial products.  Each case asserts the kernel instance it runs and
compares with a float64 convolution.  The bound per output is
(K / 16 + 8) 2^-24 sum |a w| (the running fp32 sum is rounded once per 16
products; the split itself and the terms left out are below 2^-24 of a
product, and a gate product is rounded once), plus a few ulp of the output for
the bias and the activation.  That bound grows with K, where a partial product
gone missing grows with its root only; the 2-norm of each case is held to
(sqrt(K / 16) + 4) 2^-24 of the products' sum as well (independent roundings of
a sum growing like a random walk, with the gate's and the store's), which a sum
without any one of the six partial products exceeds.
"""
import ctypes
import zlib

import numpy as np
import pytest

from test_conv_kernels_gpu import ACT_HSWISH, ACT_NONE, ACT_RELU, PROBE, _lib, _ptr, act, bf16_round, conv_ref

# name, n, h, w, c, co, k, stride, pads (top, left, bottom, right), gated, splits, act, kernel
CASES = [
    ("1x1 whole tiles", 2, 64, 64, 64, 256, (1, 1), 1, (0, 0, 0, 0), False, 1, ACT_RELU, "conv_split<64x64,1x1>"),
    ("1x1 M, N and K tails", 3, 61, 67, 100, 180, (1, 1), 1, (0, 0, 0, 0), False, 1, ACT_HSWISH,
     "conv_split<64x64,1x1>"),
    ("1x1 columns past a block", 1, 130, 131, 64, 132, (1, 1), 1, (0, 0, 0, 0), False, 1, ACT_NONE,
     "conv_split<64x64,1x1>"),
    ("1x1 even columns", 1, 130, 131, 72, 134, (1, 1), 1, (0, 0, 0, 0), False, 1, ACT_NONE, "conv_split<64x64,1x1>"),
    ("gated, tiles straddling images", 9, 59, 41, 84, 132, (1, 1), 1, (0, 0, 0, 0), True, 1, ACT_RELU,
     "conv_split<64x64,1x1,gate>"),
    ("1x1 odd columns", 1, 130, 131, 72, 133, (1, 1), 1, (0, 0, 0, 0), False, 1, ACT_NONE, "conv_split<64x64,1x1>"),
    ("gated, odd columns", 9, 59, 41, 84, 131, (1, 1), 1, (0, 0, 0, 0), True, 1, ACT_RELU,
     "conv_split<64x64,1x1,gate>"),
    ("3x3 odd columns", 1, 131, 127, 12, 131, (3, 3), 1, (1, 1, 1, 1), False, 1, ACT_RELU, "conv_split<64x64>"),
    ("3x3 stride 1, channels not in 32", 1, 131, 127, 12, 128, (3, 3), 1, (1, 1, 1, 1), False, 1, ACT_RELU,
     "conv_split<64x64>"),
    ("3x3 stride 2", 2, 190, 200, 36, 160, (3, 3), 2, (1, 1, 1, 1), False, 1, ACT_HSWISH, "conv_split<64x64>"),
    ("2x2 padded below", 1, 180, 190, 32, 64, (2, 2), 1, (0, 0, 1, 1), False, 1, ACT_RELU, "conv_split<64x64>"),
    ("3x3 split K", 1, 127, 131, 128, 64, (3, 3), 1, (1, 1, 1, 1), False, 3, ACT_RELU, "conv_split<64x64>"),
    ("1x1 split K, uneven", 1, 127, 131, 1060, 64, (1, 1), 1, (0, 0, 0, 0), False, 5, ACT_NONE,
     "conv_split<64x64,1x1>"),
    ("7x7 narrow", 2, 181, 190, 32, 32, (7, 7), 1, (3, 3, 3, 3), False, 1, ACT_NONE, "conv_split<128x32>"),
    ("1x1 narrow, N tail", 1, 270, 256, 68, 28, (1, 1), 1, (0, 0, 0, 0), False, 1, ACT_RELU, "conv_split<128x32,1x1>"),
    ("1x1 gated narrow", 3, 170, 140, 64, 24, (1, 1), 1, (0, 0, 0, 0), True, 1, ACT_RELU,
     "conv_split<128x32,1x1,gate>"),
    ("1x1 narrow, odd columns", 1, 270, 256, 68, 27, (1, 1), 1, (0, 0, 0, 0), False, 1, ACT_RELU,
     "conv_split<128x32,1x1>"),
    ("1x1 gated narrow, odd columns", 3, 170, 140, 64, 27, (1, 1), 1, (0, 0, 0, 0), True, 1, ACT_NONE,
     "conv_split<128x32,1x1,gate>"),
    ("3x3 narrow, odd columns", 1, 270, 256, 16, 31, (3, 3), 1, (1, 1, 1, 1), False, 1, ACT_NONE, "conv_split<128x32>"),
    ("1x1 deep, wide tiles with tails", 2, 140, 141, 776, 772, (1, 1), 1, (0, 0, 0, 0), False, 1, ACT_RELU,
     "conv_split<128x128,1x1>"),
    ("3x3 deep, wide tiles", 2, 120, 129, 88, 516, (3, 3), 1, (1, 1, 1, 1), False, 1, ACT_NONE,
     "conv_split<128x128>"),
    ("small 1x1 whole tiles", 1, 16, 24, 256, 64, (1, 1), 1, (0, 0, 0, 0), False, 1, ACT_RELU, "conv_split<64x32,1x1>"),
    ("small 1x1 M, N and K tails", 2, 9, 13, 84, 46, (1, 1), 1, (0, 0, 0, 0), False, 1, ACT_HSWISH,
     "conv_split<64x32,1x1>"),
    ("small 1x1 one slice", 1, 5, 7, 48, 24, (1, 1), 1, (0, 0, 0, 0), False, 1, ACT_NONE, "conv_split<64x32,1x1>"),
    ("small 1x1 two slices", 1, 5, 7, 64, 33, (1, 1), 1, (0, 0, 0, 0), False, 1, ACT_NONE, "conv_split<64x32,1x1>"),
    ("small gated, many slices", 3, 9, 11, 420, 60, (1, 1), 1, (0, 0, 0, 0), True, 1, ACT_RELU,
     "conv_split<64x32,1x1,gate>"),
    ("small gated, one slice", 2, 8, 9, 52, 32, (1, 1), 1, (0, 0, 0, 0), True, 1, ACT_NONE,
     "conv_split<64x32,1x1,gate>"),
    ("small 3x3", 2, 13, 23, 20, 40, (3, 3), 1, (1, 1, 1, 1), False, 1, ACT_RELU, "conv_split<64x32>"),
    ("small 3x3 stride 2, split K", 1, 26, 46, 64, 64, (3, 3), 2, (1, 1, 1, 1), False, 4, ACT_NONE,
     "conv_split<64x32>"),
    ("small 1x1 split K, uneven", 1, 13, 23, 900, 96, (1, 1), 1, (0, 0, 0, 0), False, 3, ACT_RELU,
     "conv_split<64x32,1x1>"),
    ("small gated, split K uneven", 3, 9, 11, 900, 60, (1, 1), 1, (0, 0, 0, 0), True, 3, ACT_RELU,
     "conv_split<64x32,1x1,gate>"),
    ("small gated, odd columns", 3, 9, 11, 420, 61, (1, 1), 1, (0, 0, 0, 0), True, 1, ACT_NONE,
     "conv_split<64x32,1x1,gate>"),
    ("small 3x3, odd columns", 2, 13, 23, 20, 41, (3, 3), 1, (1, 1, 1, 1), False, 1, ACT_RELU, "conv_split<64x32>"),
]


def _split_lib():
    lib = _lib()
    f, i = ctypes.POINTER(ctypes.c_float), ctypes.c_int
    lib.ppocr_probe_conv_split3.argtypes = [f, i, i, i, i, f, f] + [i] * 10 + [f, i, f, ctypes.POINTER(i), f,
                                                                               ctypes.POINTER(ctypes.c_char_p)]
    lib.ppocr_probe_conv_split3.restype = i
    name = ctypes.POINTER(ctypes.c_char_p)
    lib.ppocr_probe_split_terms.argtypes = [f, i, i, i, i, f, f, i, i, f, f, f, i, i, i, f, ctypes.c_float, i, f, name]
    lib.ppocr_probe_split_multi.argtypes = [i, ctypes.POINTER(i), f, f, f, i, f, f, f, f, name]
    return lib


def norm_bound(k):
    """Largest 2-norm of the error over that of the exact sums."""
    return (np.sqrt(k / 16) + 4) * 2.0 ** -24


def _run(case, se=False):
    name, n, h, w, c, co, (kh, kw), stride, pads, gated, splits, kind, want = case
    rng = np.random.default_rng(zlib.crc32(name.encode()))
    x = (rng.standard_normal((n, h, w, c)) * np.exp2(rng.integers(-6, 7, (n, h, w, c)))).astype(np.float32)
    wt = (rng.standard_normal((co, c, kh, kw)) / np.sqrt(c * kh * kw)).astype(np.float32)
    b = rng.standard_normal(co).astype(np.float32)
    g = rng.uniform(0.0, 1.0, (n, c)).astype(np.float32) if gated else None
    ho = (h + pads[0] + pads[2] - kh) // stride + 1
    wo = (w + pads[1] + pads[3] - kw) // stride + 1
    out = np.empty((n, ho, wo, co), dtype=np.float32)
    kernel = ctypes.c_char_p()
    rows = ctypes.c_int()
    part = np.zeros((-(-ho * wo // 16) + 4, co), np.float32) if se else None
    rc = _split_lib().ppocr_probe_conv_split3(_ptr(x), n, h, w, c, _ptr(wt), _ptr(b), co, kh, kw, stride, stride, *pads,
                                              kind, _ptr(g), splits, _ptr(out), ctypes.byref(rows) if se else None,
                                              _ptr(part), ctypes.byref(kernel))
    assert rc == 0
    assert kernel.value.decode() == want
    xs = x.astype(np.float64) * (g[:, None, None, :] if gated else 1.0)
    ref = conv_ref(xs, wt, b, (stride, stride), pads, ACT_NONE)
    size = conv_ref(np.abs(xs), np.abs(wt), None, (stride, stride), pads, ACT_NONE)
    tol = (c * kh * kw / 16 + 8) * 2.0 ** -24 * size + 2.0 ** -21 * np.abs(ref)
    err = np.abs(out - act(ref, kind))
    assert np.all(err <= tol), (name, float((err / tol).max()))
    lipschitz = 1.5 if kind == ACT_HSWISH else 1.0
    off = np.linalg.norm(err) / lipschitz - 2.0 ** -23 * np.linalg.norm(ref)
    assert off <= norm_bound(c * kh * kw) * np.linalg.norm(ref - b), (name, off / np.linalg.norm(ref - b))
    return out, part[:rows.value] if se else None


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_split_conv_matches_float64(case):
    _run(case)


@pytest.mark.parametrize("k", sorted({c[4] * c[6][0] * c[6][1] for c in CASES}))
def test_norm_bound_sees_a_lost_product(k):
    """In float64 (no GPU): the six partial products are within the bound the
    kernel's cases are held to, any five of them are not."""
    rng = np.random.default_rng(k)
    x = (rng.standard_normal((64, k)) * np.exp2(rng.integers(-6, 7, (64, k)))).astype(np.float32)
    w = (rng.standard_normal((32, k)) / np.sqrt(k)).astype(np.float32)

    def parts(v):
        h = bf16_round(v)
        m = bf16_round(v - h)
        return [p.astype(np.float64) for p in (h, m, bf16_round(v - h - m))]

    a, b = parts(x), parts(w)
    terms = [a[i] @ b[j].T for i, j in ((0, 0), (0, 1), (1, 0), (0, 2), (1, 1), (2, 0))]
    ref = x.astype(np.float64) @ w.T.astype(np.float64)
    off = [np.linalg.norm(sum(terms) - lost - ref) / np.linalg.norm(ref) for lost in [0.0, *terms]]
    assert off[0] < 0.1 * norm_bound(k)
    assert min(off[1:]) > 1.5 * norm_bound(k), min(off[1:]) / norm_bound(k)


@pytest.mark.gpu
@pytest.mark.parametrize("h,w,co,waves,kernel", [(131, 129, 132, 2, "conv_split<64x64,1x1>"),
                                                 (270, 256, 28, 4, "conv_split<128x32,1x1>"),
                                                 (19, 23, 44, 4, "conv_split<64x32,1x1>")])
def test_split_conv_leaves_se_sums(h, w, co, waves, kernel):
    """A single image's 1x1 layer also leaves its channel sums (one row per
    wave's rows of a tile), within fp32 summation order of the stored output."""
    case = ("se sums", 1, h, w, 64, co, (1, 1), 1, (0, 0, 0, 0), False, 1, ACT_RELU, kernel)
    out, part = _run(case, se=True)
    assert part.shape[0] == -(-h * w // (128 if "128x32" in kernel else 64)) * waves
    want = out.reshape(-1, out.shape[-1]).astype(np.float64)
    assert np.all(np.abs(part.astype(np.float64).sum(0) - want.sum(0)) <= 1e-5 * np.abs(want).sum(0) + 1e-5)


# Inputs of one sign (as after a ReLU) let the running sum grow with every
# product, where each of its roundings counts most.
@pytest.mark.gpu
@pytest.mark.parametrize("positive", [True, False])
@pytest.mark.parametrize("h,w,k,co,kernel", [(64, 128, 96, 256, "conv_split<64x64,1x1>"),
                                             (64, 128, 512, 256, "conv_split<64x64,1x1>"),
                                             (256, 260, 192, 32, "conv_split<128x32,1x1>"),
                                             (8, 16, 96, 256, "conv_split<64x32,1x1>"),
                                             (8, 16, 1024, 256, "conv_split<64x32,1x1>"),
                                             (128, 130, 800, 512, "conv_split<128x128,1x1>")])
def test_split_conv_is_as_accurate_as_fp32(h, w, k, co, kernel, positive):
    """The 2-norm error against float64 is not above the fp32 matrix
    instructions' on the same layer, for inputs of both signs and of one."""
    lib = _split_lib()
    n = 2 if "128x128" in kernel else 1
    rng = np.random.default_rng(k + co)
    x = rng.standard_normal((n, h, w, k)).astype(np.float32)
    if positive:
        x = np.maximum(x, 0)
    wt = (rng.standard_normal((co, k, 1, 1)) / np.sqrt(k)).astype(np.float32)
    one = [co, 1, 1, 1, 1, 0, 0, 0, 0, ACT_NONE, None, 1]
    plain, split = (np.empty((n, h, w, co), np.float32) for _ in range(2))
    assert lib.ppocr_probe_conv(_ptr(x), n, h, w, k, _ptr(wt), None, *one, 0, _ptr(plain)) == 0
    name = ctypes.c_char_p()
    assert lib.ppocr_probe_conv_split3(_ptr(x), n, h, w, k, _ptr(wt), None, *one, _ptr(split), None, None,
                                       ctypes.byref(name)) == 0
    assert name.value.decode() == kernel
    ref = (x.reshape(-1, k).astype(np.float64) @ wt[:, :, 0, 0].T.astype(np.float64)).reshape(plain.shape)
    err = [np.linalg.norm(o - ref) / np.linalg.norm(ref) for o in (split, plain)]
    assert err[0] <= err[1], err


# name, n, h, w, c, co, act, terms, kernel: the epilogues a 1x1 layer's plan
# can ask for, on every tile (registers and LDS).
TERMS_CASES = [
    ("64x64 residual", 1, 130, 131, 72, 132, ACT_NONE, {"res"}, "conv_split<64x64,1x1>"),
    ("64x64 gated residual", 3, 73, 75, 72, 132, ACT_RELU, {"res", "res_gate"}, "conv_split<64x64,1x1>"),
    ("64x64 upsample-add", 2, 96, 92, 72, 132, ACT_NONE, {"up"}, "conv_split<64x64,1x1>"),
    ("64x64 residual, blocks of 2", 2, 91, 93, 96, 132, ACT_RELU, {"res", "rep2"}, "conv_split<64x64,1x1>"),
    ("64x64 residual, blocks of 4, short K", 2, 91, 93, 48, 132, ACT_RELU, {"res", "rep4"}, "conv_split<64x64,1x1>"),
    ("64x64 greedy", 1, 1, 2100, 120, 1003, ACT_NONE, {"ctc"}, "conv_split<64x64,1x1>"),
    ("64x64 head, 64 channels", 2, 67, 71, 64, 256, ACT_RELU, {"db64"}, "conv_split<64x64,1x1>"),
    ("64x64 head, 32 channels", 1, 130, 131, 48, 128, ACT_RELU, {"db32"}, "conv_split<64x64,1x1>"),
    ("64x64 head, 16 channels", 3, 108, 110, 48, 64, ACT_RELU, {"db16"}, "conv_split<64x64,1x1>"),
    ("128x32 gated residual", 2, 190, 180, 68, 28, ACT_NONE, {"res", "res_gate"}, "conv_split<128x32,1x1>"),
    ("128x32 upsample-add", 2, 190, 180, 68, 28, ACT_NONE, {"up"}, "conv_split<128x32,1x1>"),
    ("128x32 residual, blocks of 8", 1, 258, 256, 68, 32, ACT_RELU, {"res", "rep8"}, "conv_split<128x32,1x1>"),
    ("128x128 gated residual", 2, 140, 141, 776, 516, ACT_NONE, {"res", "res_gate"}, "conv_split<128x128,1x1>"),
    ("128x128 greedy", 3, 1, 9000, 768, 515, ACT_NONE, {"ctc"}, "conv_split<128x128,1x1>"),
    ("64x32 gated residual", 3, 9, 11, 420, 60, ACT_RELU, {"res", "res_gate"}, "conv_split<64x32,1x1>"),
    ("64x32 upsample-add", 2, 10, 12, 84, 60, ACT_NONE, {"up"}, "conv_split<64x32,1x1>"),
    ("64x32 residual, blocks of 2", 2, 9, 13, 84, 60, ACT_NONE, {"res", "rep2"}, "conv_split<64x32,1x1>"),
    ("64x32 greedy", 2, 1, 41, 120, 690, ACT_NONE, {"ctc"}, "conv_split<64x32,1x1>"),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", TERMS_CASES, ids=[c[0] for c in TERMS_CASES])
def test_split_epilogues(case):
    name, n, h, w, c, co, kind, terms, want = case
    rng = np.random.default_rng(zlib.crc32(name.encode()))
    x = rng.standard_normal((n, h, w, c)).astype(np.float32)
    wt = (rng.standard_normal((co, c)) / np.sqrt(c)).astype(np.float32)
    b = rng.standard_normal(co).astype(np.float32)
    res = rng.standard_normal((n, h, w, co)).astype(np.float32) if "res" in terms else None
    res_gate = rng.uniform(0.0, 1.0, (n, co)).astype(np.float32) if "res_gate" in terms else None
    up = rng.standard_normal((n, h // 2, w // 2, co)).astype(np.float32) if "up" in terms else None
    rep = next((int(t[3:]) for t in terms if t.startswith("rep")), 1)
    db = next((int(t[2:]) for t in terms if t.startswith("db")), 0)
    ctc = "ctc" in terms
    wf = (rng.standard_normal((db, 4)) / np.sqrt(db)).astype(np.float32) if db else None
    shape = (n * h * w, 2) if ctc else (n, 4 * h, 4 * w) if db else (n, h * rep, w * rep, co)
    out = np.empty(shape, np.float32)
    kernel = ctypes.c_char_p()
    assert _split_lib().ppocr_probe_split_terms(_ptr(x), n, h, w, c, _ptr(wt), _ptr(b), co, kind, _ptr(res),
                                                _ptr(res_gate), _ptr(up), 2, rep, db, _ptr(wf), 0.25, int(ctc),
                                                _ptr(out), ctypes.byref(kernel)) == 0
    assert kernel.value.decode() == want
    y = x.reshape(-1, c).astype(np.float64) @ wt.T.astype(np.float64) + b
    size = np.abs(x).reshape(-1, c).astype(np.float64) @ np.abs(wt).T.astype(np.float64)
    tol = (c / 16 + 8) * 2.0 ** -24 * size + 2.0 ** -21 * np.abs(y)
    if ctc:
        # The class's logit is within both errors of the largest; the
        # probability's relative error is that of a logit difference, and of the
        # device's exp2 and reciprocal (a few ulp of exponents up to 2^4).
        at = out[:, 0].astype(int)
        rows = np.arange(len(y))
        assert np.all(y[rows, at] >= y.max(1) - 2 * tol.max(1))
        p = 1.0 / np.exp(y - y[rows, at][:, None]).sum(1)
        assert np.all(np.abs(out[:, 1] - p) <= p * (2 * tol.max(1) + 2.0 ** -19))
        return
    y, tol = act(y, kind).reshape(n, h, w, co), tol.reshape(n, h, w, co)
    if db:
        # conv_up's taps [2][2] of db channels each, then conv_final's 2x2 per
        # hidden pixel: sums of db products and a sigmoid (slope up to 1/4).
        taps = y.reshape(n, h, w, 2, 2, db).transpose(0, 1, 3, 2, 4, 5).reshape(n, 2 * h, 2 * w, db)
        slack = tol.reshape(n, h, w, 2, 2, db).transpose(0, 1, 3, 2, 4, 5).reshape(n, 2 * h, 2 * w, db)

        def final(v, weights):
            return (v @ weights).reshape(n, 2 * h, 2 * w, 2, 2).transpose(0, 1, 3, 2, 4).reshape(n, 4 * h, 4 * w)

        z = final(taps, wf.astype(np.float64)) + 0.25
        off = final(slack, np.abs(wf).astype(np.float64)) + db * 2.0 ** -24 * final(taps, np.abs(wf).astype(np.float64))
        assert np.all(np.abs(out - 1.0 / (1.0 + np.exp(-z))) <= off / 4 + 2.0 ** -21)
        return
    if res is not None:
        r = res.astype(np.float64) * (res_gate[:, None, None, :] if res_gate is not None else 1.0)
        y, tol = y + r, tol + 2.0 ** -23 * (np.abs(r) + np.abs(y))
    if up is not None:
        u = up.repeat(2, 1).repeat(2, 2)
        y, tol = y + u, tol + 2.0 ** -23 * (np.abs(u) + np.abs(y))
    y, tol = (v.repeat(rep, 1).repeat(rep, 2) for v in (y, tol))
    assert np.all(np.abs(out - y) <= tol)


# Layers [n, h, w, c, co, k] that share a launch, per instance.
MULTI_CASES = [
    ("64x64 1x1", [(1, 130, 131, 64, 132, 1), (1, 129, 140, 96, 192, 1)], False, "conv_split<64x64,1x1>"),
    ("64x64 1x1 odd columns", [(1, 130, 131, 64, 131, 1), (2, 91, 93, 100, 129, 1)], False, "conv_split<64x64,1x1>"),
    ("64x64 3x3", [(1, 130, 131, 12, 132, 3), (2, 95, 97, 20, 128, 3)], False, "conv_split<64x64>"),
    ("64x64 3x3 odd columns", [(1, 130, 131, 12, 131, 3), (1, 131, 130, 8, 129, 3)], False, "conv_split<64x64>"),
    ("64x64 sums", [(1, 130, 131, 64, 132, 1), (1, 129, 140, 96, 192, 1)], True, "conv_split<64x64,1x1>"),
    ("128x32 1x1", [(1, 270, 256, 68, 28, 1), (1, 258, 256, 160, 32, 1)], False, "conv_split<128x32,1x1>"),
    ("128x32 1x1 odd columns", [(1, 270, 256, 68, 27, 1), (1, 258, 256, 96, 31, 1)], False, "conv_split<128x32,1x1>"),
    ("128x32 3x3", [(1, 270, 256, 32, 32, 3), (1, 258, 256, 20, 28, 3)], False, "conv_split<128x32>"),
    ("128x32 3x3 odd columns", [(1, 270, 256, 12, 25, 3), (1, 258, 256, 20, 27, 3)], False, "conv_split<128x32>"),
    ("128x32 sums", [(1, 270, 256, 68, 28, 1), (1, 258, 256, 160, 32, 1)], True, "conv_split<128x32,1x1>"),
    ("64x32 1x1", [(1, 52, 92, 64, 64, 1), (1, 26, 46, 128, 64, 1), (1, 13, 23, 256, 64, 1), (1, 7, 12, 512, 64, 1)],
     False, "conv_split<64x32,1x1>"),
    ("64x32 1x1 odd columns", [(1, 52, 92, 64, 61, 1), (1, 26, 46, 128, 63, 1)], False, "conv_split<64x32,1x1>"),
    ("64x32 3x3", [(1, 52, 92, 32, 32, 3), (1, 26, 46, 32, 32, 3), (1, 13, 23, 32, 32, 3)], False,
     "conv_split<64x32>"),
    ("64x32 3x3 odd columns", [(2, 13, 23, 32, 41, 3), (1, 7, 5, 20, 43, 3)], False, "conv_split<64x32>"),
    ("64x32 sums", [(1, 52, 92, 64, 64, 1), (1, 13, 23, 100, 48, 1)], True, "conv_split<64x32,1x1>"),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", MULTI_CASES, ids=[c[0] for c in MULTI_CASES])
def test_layers_of_one_launch_equal_their_own(case):
    """A shared launch runs every layer as a launch of its own does, bit for
    bit (whose values the cases above pin), the channel sums included."""
    name, layers, sums, want = case
    rng = np.random.default_rng(zlib.crc32(name.encode()))
    dims = (ctypes.c_int * (6 * len(layers)))(*[v for layer in layers for v in layer])

    def flat(sizes, scale):
        return np.concatenate([rng.standard_normal(k).astype(np.float32) * np.float32(s) for k, s in zip(sizes, scale)])

    x = flat([n * h * w * c for n, h, w, c, co, k in layers], [1.0] * len(layers))
    wt = flat([co * c * k * k for n, h, w, c, co, k in layers], [(c * k * k) ** -0.5 for n, h, w, c, co, k in layers])
    b = flat([co for n, h, w, c, co, k in layers], [1.0] * len(layers))
    multi, single = (np.zeros(sum(n * h * w * co for n, h, w, c, co, k in layers), np.float32) for _ in range(2))
    room = sum((-(-h * w // 16) + 8) * co for n, h, w, c, co, k in layers)
    se = [np.zeros(room, np.float32) if sums else None for _ in range(2)]
    kernel = ctypes.c_char_p()
    assert _split_lib().ppocr_probe_split_multi(len(layers), dims, _ptr(x), _ptr(wt), _ptr(b), ACT_RELU, _ptr(multi),
                                                _ptr(single), _ptr(se[0]), _ptr(se[1]), ctypes.byref(kernel)) == 0
    assert kernel.value.decode() == want
    assert np.isfinite(multi).all() and multi.std() > 0
    assert np.array_equal(multi, single)
    if sums:
        assert se[0].any() and np.array_equal(se[0], se[1])


def _probe(x, wt, stride, pads, gate, splits, kind):
    """Output and kernel name of one layer on the split path, without bias."""
    n, h, w, c = x.shape
    co, _, kh, kw = wt.shape
    ho, wo = (h + pads[0] + pads[2] - kh) // stride + 1, (w + pads[1] + pads[3] - kw) // stride + 1
    out = np.empty((n, ho, wo, co), np.float32)
    name = ctypes.c_char_p()
    assert _split_lib().ppocr_probe_conv_split3(_ptr(x), n, h, w, c, _ptr(wt), None, co, kh, kw, stride, stride, *pads,
                                                kind, _ptr(gate), splits, _ptr(out), None, None,
                                                ctypes.byref(name)) == 0
    return out, name.value.decode()


# name, n, h, w, c, co, k, pads, gated, splits, kernel
RANGE_CASES = [
    ("64x64", 1, 128, 130, 64, 132, (1, 1), (0, 0, 0, 0), False, 1, "conv_split<64x64,1x1>"),
    ("64x64 gated", 2, 96, 90, 68, 128, (1, 1), (0, 0, 0, 0), True, 1, "conv_split<64x64,1x1,gate>"),
    ("64x64 3x3 split K", 1, 127, 131, 128, 64, (3, 3), (1, 1, 1, 1), False, 3, "conv_split<64x64>"),
    ("128x32 odd columns", 1, 270, 256, 68, 27, (1, 1), (0, 0, 0, 0), False, 1, "conv_split<128x32,1x1>"),
    ("128x128", 2, 120, 129, 88, 516, (3, 3), (1, 1, 1, 1), False, 1, "conv_split<128x128>"),
    ("64x32", 1, 20, 30, 84, 46, (1, 1), (0, 0, 0, 0), False, 1, "conv_split<64x32,1x1>"),
    ("64x32 gated split K", 3, 9, 11, 900, 60, (1, 1), (0, 0, 0, 0), True, 3, "conv_split<64x32,1x1,gate>"),
]


# A bf16 part of an infinite value, or of one above 3.38e38, is infinite.
@pytest.mark.gpu
@pytest.mark.parametrize("case", RANGE_CASES, ids=[c[0] for c in RANGE_CASES])
def test_infinities_and_the_top_of_the_range(case):
    """Infinite inputs and weights give infinities and NaN as the products of
    real numbers do, finite values of any size finite results, and other
    outputs are untouched."""
    name, n, h, w, c, co, (kh, kw), pads, gated, splits, want = case
    rng = np.random.default_rng(zlib.crc32(name.encode()))
    x = rng.standard_normal((n, h, w, c)).astype(np.float32)
    wt = (rng.standard_normal((co, c, kh, kw)) / np.sqrt(c * kh * kw)).astype(np.float32)
    wt[np.abs(wt) < 1e-6] = 1e-3
    gate = rng.uniform(0.1, 1.0, (n, c)).astype(np.float32) if gated else None
    x[..., c // 2] *= 0.01  # meets a weight of 3.395e38 below
    top = np.finfo(np.float32).max
    for at, v in [((0, 0, 0, 0), np.inf), ((0, 3, 5, 7), -np.inf), ((n - 1, h - 1, w - 1, c - 1), top),
                  ((n - 1, h // 2, 2, c // 2), -top), ((0, h // 2, w // 2, 1), np.float32(3.39e38)),
                  ((0, h - 2, 1, 33), np.nan)]:
        x[at] = v
    wt[3, c // 2, 0, 0] = np.float32(3.395e38)
    wt[co - 1, 0, 0, 0] = np.inf
    out, kernel = _probe(x, wt, 1, pads, gate, splits, ACT_NONE)
    assert kernel == want
    with np.errstate(invalid="ignore", over="ignore"):
        xs = x.astype(np.float64) * (gate[:, None, None, :] if gated else 1.0)
        ref = conv_ref(xs, wt, None, (1, 1), pads, ACT_NONE)
        size = conv_ref(np.abs(xs), np.abs(wt), None, (1, 1), pads, ACT_NONE)
        near = size > 2.0 ** 127  # may overflow on the way
        wide = ref.astype(np.float32)
        assert np.isinf(wide[~near]).sum() == 0
        special = ~np.isfinite(ref)
        assert np.array_equal(out[special], ref[special].astype(np.float32), equal_nan=True)
        assert np.isinf(out[special]).any() and np.isnan(out[special]).any()
        plain = ~near & ~special
        k = c * kh * kw
        assert np.all(np.abs(out - ref)[plain] <= ((k + 8) * 2.0 ** -24 * size)[plain])
        assert np.abs(ref[plain]).max() > 1e36
        relu, _ = _probe(x, wt, 1, pads, gate, splits, ACT_RELU)
        assert np.array_equal(relu[~near], np.fmax(out, 0.0)[~near])
        assert np.array_equal(relu[np.isposinf(ref)], np.full(np.isposinf(ref).sum(), np.inf, np.float32))


# The low parts of a value below 2^-110 reach bf16's smallest, 2^-133.
@pytest.mark.gpu
@pytest.mark.parametrize("scale", [2.0 ** -100, 2.0 ** -112, 2.0 ** -120, 2.0 ** -126])
@pytest.mark.parametrize("small_weights", [False, True])
def test_the_bottom_of_the_range(scale, small_weights):
    """Denormal parts count: a value is off by at most half of 2^-133, and an
    fp32 sum of 96 products by half of 2^-149 each."""
    rng = np.random.default_rng(5)
    x = (rng.standard_normal((1, 20, 30, 96)) * (1.0 if small_weights else scale)).astype(np.float32)
    wt = (rng.standard_normal((48, 96, 1, 1)) / 10 * (scale if small_weights else 1.0)).astype(np.float32)
    out, kernel = _probe(x, wt, 1, (0, 0, 0, 0), None, 1, ACT_NONE)
    assert kernel == "conv_split<64x32,1x1>"
    ref = conv_ref(x.astype(np.float64), wt, None, (1, 1), (0, 0, 0, 0), ACT_NONE)
    size = conv_ref(np.abs(x).astype(np.float64), np.abs(wt), None, (1, 1), (0, 0, 0, 0), ACT_NONE)
    off = 2.0 ** -134 * (np.abs(x).sum(3)[..., None] if small_weights else np.abs(wt).sum((1, 2, 3)))
    assert np.all(np.abs(out - ref) <= (96 / 16 + 8) * 2.0 ** -24 * size + off + 96 * 2.0 ** -149)


@pytest.mark.parametrize("co,k", [(32, 32), (33, 20), (70, 100)])
def test_packed_parts_are_the_weights(co, k):
    """The three parts of each weight add up to it within 2^-25, in the order
    the 32x32x16 product reads: lane l of step s holds column l % 32 and
    k = 16 s + 4 (l // 32) + i (i < 4) and 8 more from i = 4 on; zero past
    the matrix (no GPU needed)."""
    lib = ctypes.CDLL(str(PROBE))
    lib.ppocr_probe_split3_size.restype = ctypes.c_size_t
    rng = np.random.default_rng(co)
    w = (rng.standard_normal((co, k)) * np.exp2(rng.integers(-20, 21, (co, k)))).astype(np.float32)
    blocks, steps = -(-co // 32), 2 * -(-k // 32)
    packed = np.empty((blocks, steps, 3, 64, 8), np.uint16)
    assert lib.ppocr_probe_split3_size(co, k) == packed.size
    lib.ppocr_probe_split3_weights(_ptr(w), co, k, packed.ctypes.data_as(ctypes.POINTER(ctypes.c_uint16)))
    parts = (packed.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    back = np.zeros((blocks * 32, steps * 16))
    for lane in range(64):
        for i in range(8):
            at = 4 * (lane // 32) + i % 4 + 8 * (i // 4)
            back[lane % 32::32, at::16] = parts[:, :, :, lane, i].sum(2)
    assert np.all(np.abs(back[:co, :k] - w) <= 2.0 ** -25 * np.abs(w))
    assert not back[co:].any() and not back[:, k:].any()
    assert np.all(np.abs(parts[:, :, 1]) <= 2.0 ** -8 * np.abs(parts[:, :, 0]))
