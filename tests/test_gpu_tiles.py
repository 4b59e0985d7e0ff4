"""The tile kernel (a wave classifies an 8x8 tile's rays together) against the
per-lane state machine on the same frame, which `coop=-1` selects: both give
every ray the same crossing, so all outputs are equal bit for bit."""
import numpy as np
import pytest
import torch
import csgray as C
from csgray import scenes as S
import deep_trees as deep

pytestmark = pytest.mark.gpu


def _mixed(n, seed):
    rng = np.random.default_rng(seed)
    leaves = []
    for i in range(n):
        c, k = rng.uniform(-1, 1, 3), i % 3
        if k == 0:
            leaves.append(S.sphere(c, "C8503C", float(rng.uniform(0.2, 0.6))))
        elif k == 1:
            leaves.append(S.cube(c, "3CC850", float(rng.uniform(0.3, 0.9))))
        else:
            leaves.append(S.cylinder(c, "3C50C8", float(rng.uniform(0.1, 0.4)), float(rng.uniform(0.5, 1.6)),
                                     tuple(rng.uniform(0, 180, 3))))
    return "\n".join(S.random_ops_balanced(rng, leaves)) + "\n"


SCENES = {
    # a Union group is walked by its boxes from 24 members on
    "sphere": lambda: S.sphere((0, 0, 0), "C8503C", 0.9) + "\n",
    # trees of 448 operators or more have longer lists in exact mode and go by
    # tiles from 2000 tiles on in fast mode, 5 an operator in exact mode
    **{f"cheese{n}": lambda n=n: S.cheese(n, seed=n) for n in (1, 22, 23, 24, 25, 64, 65, 447, 448, 512)},
    **{f"mixed{n}": lambda n=n: _mixed(n, n) for n in (2, 8, 9, 39, 40, 41, 128)},
    "difference64": lambda: deep.left_deep_difference(64, seed=3),
    "union64": lambda: deep.right_deep_union(64, seed=3),
    "unbalanced48": lambda: deep.mixed_unbalanced(48, seed=3),
    # equal times at an operator: shared faces, and a solid cut by itself
    "shared": lambda: "\n".join(["Union", "Difference", S.cube((0, 0, 0), "5A5AC8", 1.0),
                                 S.cube((0.5, 0, 0), "5AC85A", 1.0), "Intersection",
                                 S.cube((0, 0, 0), "C85A5A", 1.0), S.cube((0, 0, 0), "C85A5A", 1.0)]) + "\n",
}


@pytest.mark.parametrize("mode", [C.MODE_FAST, C.MODE_EXACT], ids=["fast", "exact"])
@pytest.mark.parametrize("name", list(SCENES))
def test_tiles_equal_the_state_machine(gpu, name, mode):
    scene = C.Scene(SCENES[name]())
    light, phong = C.light((0.4, 0.7, 0.6)), C.phong(0.2, 0.7, 0.3, 16.0)
    eyes = [(2.2, 1.3, 2.9), (0.05, 0.02, 0.04), (0.0, 0.0, 4.0)]  # outside, inside the solid, along an axis
    for (w, h, samples), eye in zip([(2, 2, 1), (8, 8, 1), (65, 33, 1), (130, 71, 3), (320, 200, 1),
                                   (397, 319, 1), (400, 320, 1), (400, 360, 1)], eyes + eyes + eyes[:2]):
        cam = C.camera_look_at(eye, (0.0, 0.01, 0.0), 55)
        print(f"[case] {name} {w}x{h} samples {samples}", flush=True)
        got = scene.render(cam, light, phong, w, h, samples=samples, seed=5, mode=mode)
        ref = scene.render(cam, light, phong, w, h, samples=samples, seed=5, mode=mode, coop=-1)
        torch.cuda.synchronize()
        for key in ("rgba", "depth", "prim_id", "flags"):
            a, b = got[key].cpu().numpy(), ref[key].cpu().numpy()
            assert a.tobytes() == b.tobytes(), (key, int((a != b).sum()))
    scene.close()
