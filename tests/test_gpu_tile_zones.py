"""Primitives that leave their boxes in the tile kernel: re-entered beyond a
box's exit the state machine takes the primitive for missed, also where the
operator's own list is empty.  Default launches against the per-lane state
machine (`coop=-1`), bit for bit, and exact mode against the FP32 oracle."""
import numpy as np
import pytest
import torch
import csgray as C
import oracle as O
from csgray import scenes as S

pytestmark = pytest.mark.gpu

# A Difference whose right cylinder covers its left one at first, but not once
# a crossing of the Union beyond its box has been returned.
COVERED = """Difference
Cylinder -0.117325613 0.18570037 -0.489595215 5A5AC8 0.566062539 1.34301435 141.975537 129.780645 40.6430064
Union
Difference
Cylinder -0.297049015 0.418227952 0.504441603 5A5AC8 0.48135446 1.11875635 144.580262 70.1748793 48.9932158
Cylinder 0.104677926 0.53860785 -0.043005307 5A5AC8 0.537101549 1.14923033 103.04601 95.8871428 147.939817
Cylinder -0.402513119 0.0262948883 0.462163949 5A5AC8 0.572131429 1.30865856 22.6424859 43.8798792 140.797453
"""
COVERED_CAM = ((2.3377389907836914, 1.511763095855713, 1.1178319454193115), -0.5281323790550232, 1.1247663497924805,
               0.7853975296020508)
# Two cubes whose far faces tie, beside a Difference whose spheres' rounding
# moves their crossings past their boxes (seen from 2e4 units away).
TIED = """Union
Sphere 0 0 0.25 5AC85A 0.25
Union
Union
Cube -0.25 -0.5 -0.75 C85A5A 0.75
Cube 0 -0.4999999 -0.5 C85A5A 0.75
Difference
Sphere -0.5 0 -0.5 5AC85A 0.375
Sphere -0.5 0.1875 -0.5 5AC85A 0.375
"""
# The same by a cylinder and a cube, and a Difference of two far cylinders cut
# off by a cube.
TIED_CYLINDER = """Union
Union
Union
Cube 0.25 1 0.25 C85A5A 0.25
Cylinder 0.5 1 0.5 5A5AC8 0.125 0.75 90 90 0
Union
Difference
Sphere -0.5 0 -1 5AC85A 0.125
Sphere -0.375 0 -1 5AC85A 0.125
Sphere 0.75 0.5 0.75 5AC85A 0.375
Sphere 0.5 0.25 0.75 5AC85A 0.375
"""
CYLINDERS = """Union
Cube 0.5 -0.75 0 C85A5A 0.75
Union
Difference
Cylinder 0.25 -0.75 0 5A5AC8 0.25 1 0 0 0
Cylinder 0.25 -0.75 -0.25 5A5AC8 0.25 1 0 0 0
Sphere 0 -0.5 0.25 5AC85A 0.375
"""


# Cameras 2e4 units away (position, pitch, yaw; vertical fov 0.02 degrees).
FAR = {
    "cubes": (TIED, ((7608.66064453125, -8857.33984375, -16237.4814453125), 0.45879384875297546, 2.70339035987854), 72, 48),
    "cylinder and cube": (TIED_CYLINDER, ((9081.9072265625, 13158.810546875, 12015.1845703125), -0.7180806994438171,
                                          0.647246778011322), 72, 48),
    "cylinders": (CYLINDERS, ((4549.111328125, 15977.7548828125, -11136.2900390625), -0.925443708896637,
                              2.7537851333618164), 256, 256),
}


def _compare(text, cam, w, h):
    scene, oracle = C.Scene(text), O.OracleScene(text)
    light, phong = (0.4, 0.7, 0.6), (0.2, 0.7, 0.3, 16.0)
    for mode in (C.MODE_FAST, C.MODE_EXACT):
        got = scene.render(cam, C.light(light), C.phong(*phong), w, h, mode=mode)
        ref = scene.render(cam, C.light(light), C.phong(*phong), w, h, mode=mode, coop=-1)
        torch.cuda.synchronize()
        for key in ("rgba", "depth", "prim_id", "flags"):
            a, b = got[key].cpu().numpy(), ref[key].cpu().numpy()
            assert a.tobytes() == b.tobytes(), (mode, key, int((a != b).sum()))
    ref = oracle.render(C.cam_tuple(cam), light, O.phong8(*phong), w, h, bits=32)
    for key in ("depth", "prim_id", "flags"):
        assert got[key].cpu().numpy().tobytes() == ref[key].tobytes(), ("oracle", key)
    scene.close()


def test_a_covered_operand_reappears_beyond_the_box(gpu):
    pos, pitch, yaw, vfov = COVERED_CAM
    _compare(COVERED, C.camera(pos, pitch, yaw, vfov), 160, 120)


@pytest.mark.parametrize("name", list(FAR))
def test_views_whose_rounding_leaves_the_boxes(gpu, name):
    text, cam, w, h = FAR[name]
    _compare(text, C.camera(*cam, 0.0003490655799396336), w, h)


def _inside_out(seed, group):
    """A tree of 16 parts, or a Union of 30 small Differences, every fourth part of a negative size."""
    rng = np.random.default_rng(seed)

    def part(i):
        c, sign, kind = rng.uniform(-0.8, 0.8, 3), (-1.0 if i % 4 == 0 else 1.0), int(rng.integers(0, 3))
        if kind == 0:
            return S.sphere(c, "5AC85A", sign * rng.uniform(0.2, 0.6))
        if kind == 1:
            return S.cube(c, "C85A5A", sign * rng.uniform(0.3, 0.9))
        r, h = rng.uniform(0.15, 0.4), rng.uniform(0.4, 1.2)
        if i % 8 == 4:
            r, h = r, sign * h
        else:
            r = sign * r
        return S.cylinder(c, "5A5AC8", r, h, rng.uniform(0, 180, 3))

    if group:
        lines = S.balanced("Union", ["\n".join(["Difference", part(2 * i), part(2 * i + 1)]) for i in range(30)])
    else:
        lines = S.random_ops_balanced(rng, [part(i) for i in range(16)])
    return "\n".join(lines) + "\n"


@pytest.mark.parametrize("group", [False, True], ids=["tree", "group"])
def test_negative_sizes_turn_boxes_inside_out(gpu, group):
    for seed in range(6):
        text = _inside_out(seed, group)
        print(f"[case] seed {seed}", flush=True)
        for eye in [(2.2, 1.3, 2.9), (0.1, 0.2, 4.0)]:
            _compare(text, C.camera_look_at(eye, (0, 0.01, 0), 50), 120, 90)


def test_negative_sizes_in_a_batch(gpu):
    light, phong = C.light((0.4, 0.7, 0.6)), C.phong(0.2, 0.7, 0.3, 16.0)
    cam = C.camera_look_at((2.2, 1.3, 2.9), (0, 0.01, 0), 50)
    texts = [_inside_out(1, True), S.WIKIPEDIA, _inside_out(2, False), S.cheese(40, seed=40)]
    specs = [(C.Scene(t), cam, light, phong, 120, 90, C.alloc_outputs(120, 90)) for t in texts]
    for mode in (C.MODE_FAST, C.MODE_EXACT):
        refs = [sp[0].render(cam, light, phong, 120, 90, mode=mode, coop=-1) for sp in specs]
        C.render_batch(C.make_jobs(specs), mode=mode)
        torch.cuda.synchronize()
        for spec, ref in zip(specs, refs):
            for key in ("rgba", "depth", "prim_id", "flags"):
                assert torch.equal(spec[6][key].view(torch.uint8), ref[key].view(torch.uint8)), key
