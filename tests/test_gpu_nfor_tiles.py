"""The matrix-unit regression of the device NFOR at the edges of its tiles and windows (GPU),
against the same denoiser restated in numpy FP64: images smaller than, equal to and just over
a 16 x 8 tile, windows wider than the image, the widest staged window (regression radius 9,
patch radius 1) and unstaged ones, patches up to 7 x 7, and a variance floor above 1/4, where
the two bandwidths take a pass each.

The two differ by the order of FP64 sums of at most 625 terms and by the solver. With features
in [0, 1] and a ridge of 1e-4 the systems' condition is below 1e6 or so: 1e-16 x 1e6 bounds the
relative difference, and 1e-11 leaves the constants room."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LUM = np.array([0.2722287168, 0.6740817658, 0.0536895174])


def _shift(a, oy, ox):
    h, w = a.shape[:2]
    return a[np.clip(np.arange(h) + oy, 0, h - 1)][:, np.clip(np.arange(w) + ox, 0, w - 1)]


def _patch_distance(g, v, oy, ox, patch, floor):
    h, w = v.shape
    ys, xs = np.arange(h), np.arange(w)
    ty, tx = np.clip(ys + oy, 0, h - 1), np.clip(xs + ox, 0, w - 1)
    out = np.zeros_like(v)
    for py in range(-patch, patch + 1):
        for px in range(-patch, patch + 1):
            a = np.ix_(np.clip(ys + py, 0, h - 1), np.clip(xs + px, 0, w - 1))
            b = np.ix_(np.clip(ty + py, 0, h - 1), np.clip(tx + px, 0, w - 1))
            out += ((g[a] - g[b]) ** 2).sum(-1) / 3.0 / (v[a] + v[b] + floor)
    return np.where((ty == ys)[:, None] & (tx == xs)[None, :], 0.0, out / (2 * patch + 1) ** 2)


def _regress(img, feat, v, radius, patch, k, floor):
    h, w = v.shape
    system = np.zeros((h, w, 12, 15))
    for oy in range(-radius, radius + 1):
        for ox in range(-radius, radius + 1):
            weight = np.exp(-_patch_distance(img, v, oy, ox, patch, floor) / max(floor, k * k))
            basis = np.concatenate([np.ones((h, w, 1)), _shift(feat, oy, ox) - feat], -1)
            columns = np.concatenate([basis, _shift(img, oy, ox)], -1)
            system += (basis * weight[..., None])[..., :, None] * columns[..., None, :]
    return np.linalg.solve(system[..., :12] + 1e-4 * np.eye(12), system[..., 12:])[..., 0, :]


def _denoise(b, radius, patch, floor):
    # colours without fireflies: the suppression leaves them alone
    a, c = b["color_a"], b["color_b"]
    mean, var = 0.5 * (a + c), b["color_variance"][..., 0]
    dist2 = lambda x, y: ((x - y) ** 2).sum(-1) / 3.0
    spread = b["feature_variance"].mean(-1)

    def prefilter(image, guide):
        total, acc = np.zeros_like(var), np.zeros_like(image)
        for oy in (-1, 0, 1):
            for ox in (-1, 0, 1):
                d = ((guide - _shift(guide, oy, ox)) ** 2).mean(-1) / (spread + _shift(spread, oy, ox) + floor)
                wt = np.exp(-d / 0.25) * np.exp(-(oy * oy + ox * ox) / 2.0)
                acc, total = acc + _shift(image, oy, ox) * wt[..., None], total + wt
        return acc / total[..., None]

    fa, fb = prefilter(b["features_a"], b["features_b"]), prefilter(b["features_b"], b["features_a"])
    a0, a1 = (_regress(a, fb, 2 * var, radius, patch, k, floor) for k in (0.5, 1.0))
    c0, c1 = (_regress(c, fa, 2 * var, radius, patch, k, floor) for k in (0.5, 1.0))
    error = lambda x, y: np.maximum(0.0, 0.5 * (dist2(c, x) + dist2(a, y) - 8.0 * var) - 0.25 * dist2(x, y))

    def smooth(x, y):
        sx = sy = total = 0.0
        for oy in range(-3, 4):
            for ox in range(-3, 4):
                wt = np.exp(-_patch_distance(mean, var, oy, ox, 1, floor) / max(floor, 1.0))
                sx, sy, total = sx + _shift(x, oy, ox) * wt, sy + _shift(y, oy, ox) * wt, total + wt
        return sx / total, sy / total

    m0, m1 = smooth(error(a0, c0), error(a1, c1))
    s0, s1 = smooth((m0 <= m1).astype(float), (m1 <= m0).astype(float))
    w0 = np.where(s0 + s1 > floor, s0 / (s0 + s1), (m0 <= m1).astype(float))[..., None]
    blend = 0.5 * ((a0 + c0) * w0 + (a1 + c1) * (1.0 - w0))
    return _regress(blend, 0.5 * (fa + fb), 0.25 * dist2(a1, c1), radius, patch, 1.0, floor)


@pytest.mark.parametrize("w,h,radius,patch,floor", [
    (1, 1, 1, 1, 1e-5), (2, 5, 2, 1, 1e-5), (16, 8, 2, 1, 1e-5), (17, 9, 2, 1, 1e-5), (15, 7, 9, 1, 1e-5), (33, 25, 9, 1, 1e-5),
    (33, 18, 10, 1, 1e-5), (20, 30, 9, 2, 1e-5), (35, 17, 3, 3, 1e-5), (48, 16, 1, 2, 1e-5), (19, 21, 12, 2, 1e-5),
    (31, 20, 4, 1, 0.4), (24, 9, 2, 1, 2.0)])
def test_regression_tiles_match_numpy(ctx, w, h, radius, patch, floor):
    from luz_amd import Renderer
    rng = np.random.default_rng(w * 1000 + h)
    base = 0.3 + 0.1 * rng.random((h, w, 3))
    b = {"color_a": base + 0.01 * rng.random((h, w, 3)), "color_b": base + 0.01 * rng.random((h, w, 3)),
         "color_variance": 1e-4 * (0.5 + rng.random((h, w, 1))), "features_a": rng.random((h, w, 11)),
         "features_b": rng.random((h, w, 11)), "feature_variance": 0.01 * rng.random((h, w, 11))}
    out, _ = Renderer.nfor(ctx, b, {"regression_radius": radius, "patch_radius": patch, "min_variance": floor})
    ref = _denoise(b, radius, patch, floor)
    e = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    print(f"{w}x{h} radius {radius} patch {patch} floor {floor}: relative difference {e:.2e}")
    assert e <= 1e-11
