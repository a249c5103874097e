"""The two firefly filters (GPU) against a numpy restatement that sorts: images of 3 x 3 up,
where most windows are cut by the border, dense fireflies (every candidate count from none to
24 occurs) and tied luminances (grey levels from a short list, so that tied neighbours are the
same colour). The display filter only picks pixels, so it is exact; the denoiser's is followed
by the regression, whose bound is derived with its own tests."""

import numpy as np
import pytest

from test_gpu_nfor_tiles import _denoise

pytestmark = pytest.mark.gpu

LUM = np.array([0.2722287168, 0.6740817658, 0.0536895174])


def _window(img, y, x, reach):
    h, w = img.shape[:2]
    return [img[sy, sx] for sy in range(y - reach, y + reach + 1) for sx in range(x - reach, x + reach + 1)
            if (sy, sx) != (y, x) and 0 <= sy < h and 0 <= sx < w]


def _lum(c):
    return c[0] * LUM[0] + c[1] * LUM[1] + c[2] * LUM[2]


def _median(colors):
    return sorted(colors, key=_lum)[len(colors) // 2]


def _display(img):
    firefly = lambda c: max(c) >= 0.99 and min(c) >= 0.85 and _lum(c) >= 0.95
    saturated = lambda c: max(c) >= 0.995 and min(c) >= 0.96 and _lum(c) >= 0.98
    out = img.copy()
    for y in range(img.shape[0]):
        for x in range(img.shape[1]):
            p = img[y, x]
            bright = max(p) >= 0.50 and _lum(p) >= 0.35
            if not firefly(p) and not bright:
                continue
            around = _window(img, y, x, 2)
            candidates = [c for c in around if not firefly(c)]
            if not candidates:
                continue
            replace = False
            if not firefly(p):
                near = sorted(_lum(c) for c in _window(img, y, x, 1))
                median = near[len(near) // 2]
                if _lum(p) < median * 1.65 or _lum(p) < median + 0.08:
                    continue
                replace = True
            replace = replace or (saturated(p) and sum(map(saturated, around)) < 3)
            replace = replace or (sum(_lum(c) >= _lum(p) * 0.65 for c in around) < 4 and sum(_lum(c) >= 0.80 for c in around) < 6)
            if replace:
                out[y, x] = _median(candidates)
    return out


@pytest.mark.parametrize("w,h", [(3, 3), (4, 3), (3, 9), (5, 5), (33, 17), (64, 40)])
@pytest.mark.parametrize("share", [0.02, 0.3, 0.9])
@pytest.mark.parametrize("ties", [False, True])
def test_display_fireflies_match_numpy(ctx, w, h, share, ties):
    from luz_amd import Renderer
    rng = np.random.default_rng(w * 100 + h + int(share * 1000))
    if ties:
        img = rng.choice([0.0, 0.05, 0.1, 0.4], size=(h, w, 1)) * np.ones(3)
    else:
        img = 0.3 * rng.random((h, w, 3))
    hot = rng.random((h, w)) < share
    img[hot] = rng.choice([1.0, 4.0, 60.0], size=(hot.sum(), 1)) * (np.ones(3) if ties else 0.8 + 0.2 * rng.random((hot.sum(), 3)))
    post = {"exposure": 0.0, "contrast": 1.0, "bloom": False, "view_transform": "standard"}
    out = Renderer.postprocess(ctx, img, post)
    # one row high, an image has no windows: the same pixels, encoded but not filtered
    encoded = Renderer.postprocess(ctx, img.reshape(1, h * w, 3), post).reshape(h, w, 3)
    expect = _display(encoded)
    print(f"{w}x{h} share {share}: {(expect != encoded).any(-1).sum()} replaced")
    assert np.array_equal(out, expect)


def _suppress(img):
    out = img.copy()
    for y in range(img.shape[0]):
        for x in range(img.shape[1]):
            p = img[y, x]
            around = _window(img, y, x, 2)
            darker = [c for c in around if not _lum(c) >= _lum(p) * 0.65]
            if not darker or _lum(p) < 0.30 or len(around) - len(darker) >= 2:
                continue
            median = sorted(map(_lum, around))[len(around) // 2]
            if _lum(p) >= median * 2.5 and _lum(p) >= median + 0.18:
                out[y, x] = _median(darker)
    return out


@pytest.mark.parametrize("w,h,share", [(3, 3, 0.1), (4, 7, 0.1), (33, 18, 0.03), (29, 16, 0.03)])
def test_denoise_fireflies_match_numpy(ctx, w, h, share):
    from luz_amd import Renderer
    rng = np.random.default_rng(w + h)
    base = 0.3 + 0.1 * rng.random((h, w, 3))
    hot = rng.random((h, w)) < share
    hot[0, 0] = True
    a, c = (base + 0.01 * rng.random((h, w, 3)) + np.where(hot, 5.0, 0.0)[..., None] for _ in range(2))
    b = {"color_a": a, "color_b": c, "color_variance": 1e-4 * (0.5 + rng.random((h, w, 1))), "features_a": rng.random((h, w, 11)),
         "features_b": rng.random((h, w, 11)), "feature_variance": 0.01 * rng.random((h, w, 11))}
    clean = dict(b, color_a=_suppress(a), color_b=_suppress(c))
    mean = 0.5 * (clean["color_a"] + clean["color_b"])
    # the second filter, over the mean, finds nothing left (no close groups of them)
    assert np.array_equal(_suppress(mean), mean) and not np.array_equal(clean["color_a"], a)
    out, _ = Renderer.nfor(ctx, b, {"regression_radius": 2, "patch_radius": 1, "min_variance": 1e-5})
    ref = _denoise(clean, 2, 1, 1e-5)
    assert np.linalg.norm(out - ref) / np.linalg.norm(ref) <= 1e-11
