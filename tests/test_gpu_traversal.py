"""The device node and leaf layout at its edges (GPU), against the FP64 oracle: top levels of
1 to 40 primitives (leaves hold at most 4 of one kind: triangle runs, single instances, lists
of the rest), kinds mixed in one leaf, meshes whose root is a leaf or one node, rays parallel
to axes (a sun straight overhead: every shadow ray has two zero direction components), and
deep stacks that leave the LDS part (lds_stack 8)."""

import os
import random

import numpy as np
import pytest

import oracle_lib
from conftest import rel_mse

pytestmark = pytest.mark.gpu


def _obj(rng, quads):
    """A bumpy quads x quads sheet of 2 quads^2 triangles."""
    n = quads + 1
    out = [f"v {i / quads - 0.5:.6f} {0.2 * rng.random():.6f} {j / quads - 0.5:.6f}" for j in range(n) for i in range(n)]
    for j in range(quads):
        for i in range(quads):
            a = j * n + i + 1
            out += [f"f {a} {a + n} {a + 1}", f"f {a + 1} {a + n} {a + n + 1}"]
    return "\n".join(out) + "\n"


def _scene(directory, count, analytic, seed):
    rng = random.Random(seed)
    os.makedirs(directory, exist_ok=True)
    lines = ["[settings]", "resolution=48,36", "samples=4", "maxlightbounces=5", "adaptive=0", "denoise=0", "view_transform=raw",
             "bloom=0", "outputfilename=render.tiff", "sky=none", "background=(0.4,0.5,0.6)", "", "[materials]",
             "material a {", "type=lambertian", "color=(0.6,0.5,0.4)", "}", "material m {", "type=metal", "color=(0.8,0.8,0.7)",
             "roughness=0.4", "}", "", "[scene]", "camera main {", "position=(0,2,-9)", "direction=(0,-0.15,1)", "up=(0,1,0)",
             "focal_length_mm=24", "sensor_width_mm=36", "sensor_height_mm=27", "pinhole=1", "focus_distance=10", "}", "objects{"]
    kinds = ["triangle", "triangle", "rectangle", "mesh"] + (["sphere", "cube"] if analytic else [])
    for i in range(count):
        x, y, z = (rng.uniform(-4, 4), rng.uniform(-1, 3), rng.uniform(-4, 4))
        mat = rng.choice(["a", "m"])
        kind = kinds[i % len(kinds)]
        if kind == "triangle":
            p = [(x + rng.uniform(-2, 2), y + rng.uniform(-1, 1), z + rng.uniform(-2, 2)) for _ in range(3)]
            lines.append("triangle=" + ",".join("(%.6f,%.6f,%.6f)" % v for v in p) + f",material={mat}")
        elif kind == "rectangle":
            lines.append(f"rectangle=({x:.6f},{y:.6f},{z:.6f}),(0.2,1,-0.3),1.5,1.1,material={mat}")
        elif kind == "sphere":
            lines.append(f"sphere=({x:.6f},{y:.6f},{z:.6f}),{rng.uniform(0.2, 0.8):.6f},material={mat}")
        elif kind == "cube":
            lines.append(f"cube=({x:.6f},{y:.6f},{z:.6f}),(0,0,-1),0.9,0.7,1.1,material={mat}")
        else:
            quads = (1, 2, 5, 24)[(i // len(kinds)) % 4]
            name = f"sheet{quads}.obj"
            with open(os.path.join(directory, name), "w") as fh:
                fh.write(_obj(random.Random(quads), quads))
            lines += [f"object o{i} {{", f"file={name}", f"position=({x:.6f},{y:.6f},{z:.6f})", "scale=(2.5,2,2.5)",
                      f"material={mat}", "}"]
    if analytic:
        lines += ["directional_light sun {", "direction=(0,-1,0)", "color=(1,0.95,0.9)", "irradiance=3", "}"]
    path = os.path.join(directory, f"t{count}_{int(analytic)}.luz")
    with open(path, "w") as fh:
        fh.write("\n".join(lines + ["}"]) + "\n")
    return path


@pytest.mark.parametrize("analytic", [False, True])
@pytest.mark.parametrize("count", [1, 2, 3, 4, 5, 8, 9, 16, 17, 40])
def test_layout_edges_match_oracle(ctx, workload_dir, count, analytic):
    from luz_amd import Renderer, SceneFile
    path = _scene(os.path.join(workload_dir, "traversal"), count, analytic, 100 + count)
    scene = SceneFile.read(ctx, path)
    ids, t = Renderer.primary_hits(scene, seed=3)
    rids, rt = oracle_lib.primary(path, 3, 48, 36)
    assert (ids != np.asarray(rids).reshape(ids.shape)).any(axis=-1).sum() <= 1	# an fp32 edge at most
    same = (ids == np.asarray(rids).reshape(ids.shape)).all(axis=-1)
    assert np.allclose(t[same], np.asarray(rt).reshape(t.shape)[same], rtol=2e-5, atol=2e-5)
    ref, _ = oracle_lib.render(path, 3, 4, 48, 36)
    base = None
    for integrator, tuning in (("megakernel", None), ("wavefront", None), ("wavefront", {"lds_stack": 8, "extend_refill": 1})):
        img, _ = Renderer.render(scene, seed=3, integrator=integrator, tuning=tuning)
        assert np.isfinite(img).all()
        # the bar of every image against the FP64 paths: a few samples may flip
        assert rel_mse(img, ref) <= 1e-4, (integrator, tuning)
        if integrator == "wavefront":
            assert base is None or np.array_equal(img, base)
            base = img
    merged, _ = Renderer.render_batch([scene, scene], seeds=[3, 3], samples=[4, 4])
    assert np.array_equal(merged[0], base) and np.array_equal(merged[1], base)
