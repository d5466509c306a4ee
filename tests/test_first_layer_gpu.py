"""First-layer kernels on pixels that are not finite: such a pixel belongs to the outputs whose filter covers it and to no other -- neither to
those that only meet it at a padding tap of the kernel's own (an MFMA multiplies those by zero, and zero times infinity is NaN) nor as NaN
where a single infinity gives an infinity."""
import numpy as np
import pytest

from msnhnet_amd import hipabi as abi

pytestmark = pytest.mark.gpu


def _spots(h, w):
    return [(0, 0), (0, w - 1), (h - 1, 0), (h - 1, w - 1), (h // 2, w // 2), (h // 2 + 1, 3)]


def _check(dtype, c, h, w, oc, k, stride, pad, algo="stem"):
    """one image per position and value; weights without zeros, so that the one non-finite pixel decides what each output has to be"""
    import gpuutil as gu
    rng = np.random.default_rng(c * 100 + k * 10 + oc)
    wt = rng.uniform(0.25, 1.0, (oc, c, k, k)).astype(np.float32) * rng.choice((-1.0, 1.0), (oc, c, k, k)).astype(np.float32) / (c * k * k)
    base = rng.uniform(0.0, 1.0, (c, h, w)).astype(np.float32)
    if dtype == abi.F16:
        wt, base = gu.round_f16(wt), gu.round_f16(base)
    cases = [(ci, y, x, v) for ci in range(c) for (y, x) in _spots(h, w) for v in ((np.inf, -np.inf, np.nan, 1e5) if ci == c - 1 and (y, x) == (h // 2, w // 2) else (np.inf,))]
    imgs = np.stack([base] * len(cases))
    for i, (ci, y, x, v) in enumerate(cases):
        imgs[i, ci, y, x] = v
    print("first layer", dtype, c, h, w, oc, k, stride, pad, algo, flush=True)
    y, used = gu.conv2d(imgs, wt, dtype=dtype, stride=stride, pad=pad, algo=algo, out_ld=(oc + 7) // 8 * 8)
    assert used == algo
    clean, _ = gu.conv2d(np.stack([base] * 2), wt, dtype=dtype, stride=stride, pad=pad, algo=algo, out_ld=(oc + 7) // 8 * 8)
    oh, ow = y.shape[2:]
    for i, (ci, py, px, v) in enumerate(cases):
        want = clean[0].astype(np.float64)
        for oy in range(oh):
            ky = py - (oy * stride - pad)
            for ox in range(ow):
                kx = px - (ox * stride - pad)
                if 0 <= ky < k and 0 <= kx < k:
                    big = v if dtype == abi.F16 or not np.isfinite(v) else np.nan             # (1e5: infinite as float16, an ordinary number as float32)
                    want[:, oy, ox] = np.nan if np.isnan(big) else np.inf * np.sign(big) * np.sign(wt[:, ci, ky, kx])
        got = y[i].astype(np.float64)
        if v == 1e5 and dtype == abi.F32:
            assert np.isfinite(got).all()
            continue
        assert np.array_equal(np.isnan(got), np.isnan(want)), (ci, py, px, v, "NaN in other places")
        inf = np.isinf(want)
        assert np.array_equal(got[inf], want[inf]) and np.array_equal(np.isinf(got), inf), (ci, py, px, v)
        fin = np.isfinite(want)
        assert np.array_equal(got[fin], want[fin]), (ci, py, px, v, "a pixel that this output does not cover changed it")


@pytest.mark.parametrize("dtype", [abi.F16, abi.F32])
@pytest.mark.parametrize("c,h,w,oc,k,stride,pad", [(3, 24, 70, 32, 3, 1, 1), (3, 24, 70, 16, 3, 2, 1), (1, 24, 70, 32, 3, 1, 1), (4, 20, 66, 16, 3, 1, 0), (3, 20, 72, 64, 5, 2, 2),
                                                   (2, 20, 72, 16, 5, 1, 2), (3, 30, 150, 64, 7, 2, 3), (3, 30, 150, 16, 7, 2, 3), (3, 22, 70, 128, 7, 1, 3), (1, 22, 70, 16, 7, 2, 3)])
def test_pixels_that_are_not_finite(dtype, c, h, w, oc, k, stride, pad):
    _check(dtype, c, h, w, oc, k, stride, pad)


@pytest.mark.parametrize("dtype", [abi.F16, abi.F32])
@pytest.mark.parametrize("c,h,w,oc", [(3, 32, 32, 32), (3, 30, 146, 32), (3, 26, 72, 16), (3, 64, 128, 64), (3, 12, 66, 128), (2, 20, 70, 32), (1, 22, 68, 16), (3, 2, 2, 32)])
def test_focus_opening(dtype, c, h, w, oc):
    """the 6x6 stride-2 filter: against slices, concatenation and a 3x3 convolution in float64, and the pixels that are not finite"""
    import gpuutil as gu
    rng = np.random.default_rng(oc + c + h)
    w3 = (rng.standard_normal((oc, 4 * c, 3, 3)) / np.sqrt(36 * c)).astype(np.float32)
    x = rng.uniform(-1.0, 1.0, (2, c, h, w)).astype(np.float32)
    if dtype == abi.F16:
        x, w3 = gu.round_f16(x), gu.round_f16(w3)
    at = {(0, 0): 0, (1, 0): c, (0, 1): 2 * c, (1, 1): 3 * c}                     # row and column parity -> channel of the concatenation (YOLOv5's order)
    joined = np.zeros((2, 4 * c, h // 2 + 2, w // 2 + 2))
    w6 = np.zeros((oc, c, 6, 6), np.float32)
    for (dy, dx), ch in at.items():
        joined[:, ch:ch + c, 1:-1, 1:-1] = x[:, :, dy::2, dx::2]
        w6[:, :, dy::2, dx::2] = w3[:, ch:ch + c]
    ref = np.zeros((2, oc, h // 2, w // 2))
    for ky in range(3):
        for kx in range(3):
            ref += np.einsum("oc,bchw->bohw", w3[:, :, ky, kx].astype(np.float64), joined[:, :, ky:ky + h // 2, kx:kx + w // 2])
    print("focus", dtype, c, h, w, oc, flush=True)
    got, used = gu.conv2d(x, w6, dtype=dtype, stride=2, pad=2, algo="stem_focus", out_ld=oc + 8)
    assert used == "stem_focus" and got.shape == ref.shape
    # float32: 36 c products summed in another order; float16: the result rounded to 11 bits
    assert gu.rel_err(got, ref) <= (2e-6 if dtype == abi.F32 else 1e-3)
    if h > 8:
        _check(dtype, c, h, w, oc, 6, 2, 2, "stem_focus")
