"""Coincident primitives (GPU), against the FP64 oracle's hits of each alone: of primitives hit at the same distance
the last in the scene's list is the hit.

Four mesh quads that overlap on the camera's axis lie on one of three planes each, in every
combination (81): the children of one node, in the list's order (from left to right, the
first quad the largest), whose entry distances tie as the planes do. The quads' sizes are
powers of two, so hits on one plane have the same FP32 distance and every pixel that sees a
tie shows the order in which equally near children are visited."""

import itertools
import os

import numpy as np
import pytest

import oracle_lib

pytestmark = pytest.mark.gpu

SETTINGS = """[settings]
resolution=48,36
samples=1
maxlightbounces=2
adaptive=0
denoise=0
view_transform=raw
bloom=0
outputfilename=render.tiff
sky=none
background=(0.4,0.5,0.6)

[materials]
material a {
type=lambertian
color=(0.6,0.5,0.4)
}

[scene]
camera main {
position=(0.1,0.2,-8)
direction=(0,0,1)
up=(0,1,0)
focal_length_mm=24
sensor_width_mm=36
sensor_height_mm=27
pinhole=1
focus_distance=10
}
objects{
"""


def _write(directory, name, objects):
    os.makedirs(directory, exist_ok=True)
    with open(os.path.join(directory, "quad.obj"), "w") as fh:
        fh.write("v -1 -1 0\nv 1 -1 0\nv 1 1 0\nv -1 1 0\nf 1 3 2\nf 1 4 3\n")
    path = os.path.join(directory, name + ".luz")
    with open(path, "w") as fh:
        fh.write(SETTINGS + objects + "}\n")
    return path


def _quad(i, z):
    size = 2 if i else 4
    return f"object o{i} {{\nfile=quad.obj\nposition=({i - 1.5},0,{z})\nscale=({size},{size},1)\nmaterial=a\n}}\n"


def _oracle(path):
    return np.asarray(oracle_lib.primary(path, 3, 48, 36)[0]).reshape(36, 48, 2)[..., 0]


@pytest.mark.parametrize("last", [0, 1, 2])
def test_equally_near_children_keep_their_order(ctx, workload_dir, last):
    from luz_amd import Renderer, SceneFile
    directory = os.path.join(workload_dir, "ties")
    covers = {(i, z): _oracle(_write(directory, "alone", _quad(i, z))) >= 0 for i in range(4) for z in range(3)}
    for planes in itertools.product((0, 1, 2), repeat=3):
        planes += (last,)
        want = np.full((36, 48), -1)
        for z in (2, 1, 0):	# the nearest plane, and on it the last quad
            for i in range(4):
                if planes[i] == z:
                    want[covers[i, z]] = i
        path = _write(directory, f"quads{last}", "".join(_quad(i, z) for i, z in enumerate(planes)))
        ids, _ = Renderer.primary_hits(SceneFile.read(ctx, path), seed=3)
        # a pixel on a quad's edge may see past it in FP32
        assert (ids[..., 0] != want).sum() <= 2, planes


@pytest.mark.parametrize("kinds", ["RT", "TR", "RTR", "TRT", "RRT", "TTR", "RTRT", "TRRT"])
def test_the_last_of_a_leaf_of_triangles_and_rectangles_is_hit(ctx, workload_dir, kinds):
    """T a triangle over half of the rectangle R, one on another in one leaf of the top level."""
    from luz_amd import Renderer, SceneFile
    directory = os.path.join(workload_dir, "ties")
    text = {"T": "triangle=(-2,-2,0),(-2,2,0),(2,-2,0),material=a\n", "R": "rectangle=(0,0,0),(0,0,-1),4,4,material=a\n"}
    shared = _oracle(_write(directory, "triangle", text["T"])) == 0
    assert shared.sum() > 80
    path = _write(directory, kinds, "".join(text[k] for k in kinds))
    want = _oracle(path)
    assert (want[shared] == len(kinds) - 1).all()
    scene = SceneFile.read(ctx, path)
    got = Renderer.primary_hits(scene, seed=3)[0][..., 0]
    assert (got[~shared] == want[~shared]).all()
    assert np.isin(got[shared], [kinds.rindex("T"), kinds.rindex("R")]).all()
    # The FP32 distances of a triangle and a rectangle differ by an ulp in some pixels, either way,
    # and only there may the earlier one be nearer: were ties given to it, it had most of them
    assert (got[shared] == len(kinds) - 1).mean() > 0.5
    one, _ = Renderer.render(scene, seed=3, samples=2, integrator="wavefront")
    for image in Renderer.render_batch([scene, scene], [3, 3], samples=[2, 2])[0]:
        assert np.array_equal(image, one)
