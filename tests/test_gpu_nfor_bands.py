"""The NFOR regression's bands of image rows (GPU): an image whose per-pixel systems take more
than the 4 GiB of one band, so that its last rows are a short second band, against the same
rows denoised as an image of their own, which is one band. Every pixel's sums are formed in
the same order wherever its tile lies, so the rows are equal bit for bit from as far below the
crop's upper edge as that edge reaches. Both forms: two bandwidths in a pass, and one."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WIDTH = 512
SYSTEM_BYTES = 114 * 8 * 2		# a pixel's systems at both bandwidths
BAND = (1 << 32) // (SYSTEM_BYTES * WIDTH * 8) * 8	# rows of a band: whole tiles of 8


@pytest.mark.parametrize("floor", [1e-5, 0.4])
def test_rows_of_a_second_band(ctx, floor):
    from luz_amd import Renderer
    height, top = BAND + 29, BAND - 96
    rng = np.random.default_rng(11)
    shapes = {"color_a": 3, "color_b": 3, "color_variance": 1, "features_a": 11, "features_b": 11, "feature_variance": 11}
    # a strip of random rows, repeated (an odd number of rows, so that no two bands start alike)
    tile = {k: rng.random((331, WIDTH, n)) * (0.01 if "variance" in k else 1.0) for k, n in shapes.items()}
    whole = {k: np.resize(v, (height, WIDTH, v.shape[2])) for k, v in tile.items()}
    crop = {k: np.ascontiguousarray(v[top:]) for k, v in whole.items()}
    settings = {"regression_radius": 1, "patch_radius": 1, "min_variance": floor}
    got = Renderer.nfor(ctx, whole, settings)[0]
    want = Renderer.nfor(ctx, crop, settings)[0]
    assert np.isfinite(got).all()
    # fireflies 2 rows, features 1, the regressions 2 each, the two filters 4 each
    assert np.array_equal(got[top + 48:], want[48:])
    assert not np.array_equal(got[BAND:BAND + 20], got[:20])
