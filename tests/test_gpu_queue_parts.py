"""The wavefront's queue parts at their edges (GPU): passes of one path, one short of, exactly
and one more than a tile (512 paths) or a row of eight tiles, with grids of fewer blocks than
parts and grids that are no multiple of them. The parts only decide which block works on a
path, so every grid gives the same bits, and the megakernel, which has no queues, the same
image to FP32 rounding (the bound of the parity tests)."""

import numpy as np
import pytest

from conftest import rel_mse

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height,samples", [
    (1, 1, 1), (7, 73, 1), (512, 1, 1), (27, 19, 1), (13, 5, 63), (64, 64, 1), (17, 241, 1), (40, 30, 11)])
def test_parts_hold_every_path(ctx, cornell, width, height, samples):
    from luz_amd import Renderer, SceneFile
    scene = SceneFile.read(ctx, cornell.scene_path)
    args = dict(seed=5, samples=samples, resolution=(width, height))
    ref, _ = Renderer.render(scene, integrator="megakernel", **args)
    img, st = Renderer.render(scene, integrator="wavefront", **args)
    assert rel_mse(img, ref) < 1e-6
    assert st.closest_hit_rays >= width * height * samples
    for grid in (1, 3, 8, 9, 1283):
        other, st2 = Renderer.render(scene, integrator="wavefront", tuning={"grid": grid}, **args)
        assert np.array_equal(other, img), grid
        assert (st2.closest_hit_rays, st2.shadow_rays) == (st.closest_hit_rays, st.shadow_rays), grid
