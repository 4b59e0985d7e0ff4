"""Union groups of 24 members and more in the tile kernel, with operators,
flush faces and tilted cylinders among the members, against the per-lane state
machine on the same frame (`coop=-1`): all outputs are equal bit for bit."""
import numpy as np
import pytest
import torch
import csgray as C
from csgray import scenes as S

pytestmark = pytest.mark.gpu

KEYS = ("rgba", "depth", "prim_id", "flags")
LIGHT, PHONG = (0.4, 0.7, 0.6), (0.2, 0.7, 0.3, 16.0)


def _grid(rng, step):
    return tuple(float(v) * step for v in rng.integers(-4, 5, 3) * (0.25 / step))


def _part(rng, kind):
    c = _grid(rng, 0.25)
    if kind == "sphere":
        return S.sphere(c, "C8503C", float(rng.integers(1, 5)) * 0.125)
    if kind == "cube":
        return S.cube(c, "3CC850", float(rng.integers(1, 5)) * 0.25)
    rot = tuple(rng.uniform(0, 180, 3)) if kind == "tilted" else tuple(float(a) for a in rng.choice([0, 90], 3))
    return S.cylinder(c, "3C50C8", float(rng.integers(1, 4)) * 0.125, float(rng.integers(2, 7)) * 0.25, rot)


def _group(n, seed, kinds, ops=("Difference", "Intersection", "Union"), wrap=None):
    """A Union of n members on a grid of 1/4 (many flush faces): operators over two or three
    parts, one in four a part alone; `wrap` puts it on the right of an operator over a cube."""
    rng = np.random.default_rng(seed)
    leaves = []
    for i in range(n):
        part = lambda: _part(rng, str(rng.choice(kinds)))
        if i % 4 == 3:
            leaves.append(part())
        elif i % 4 == 2:
            leaves.append("\n".join([str(rng.choice(ops)), str(rng.choice(ops)), part(), part(), part()]))
        else:
            leaves.append("\n".join([str(rng.choice(ops)), part(), part()]))
    lines = S.balanced("Union", leaves)
    if wrap:
        lines = [wrap, S.cube((0, 0, 0), "E0E0E0", 2.0)] + lines
    return "\n".join(lines) + "\n"


def _flush(extra):
    """A cube cut by a neighbour that touches its far face, and 23 spheres out of the way, `extra` among them."""
    rng = np.random.default_rng(5)
    spheres = [extra] + [S.sphere((6.0 + 0.5 * i, 5.0, rng.uniform(-1, 1)), "5AC85A", 0.2) for i in range(22)]
    member = "\n".join(["Difference", S.cube((0, 0, 0), "C85A5A", 1.0), S.cube((0, 0, -1), "5A5AC8", 1.0)])
    return "\n".join(S.balanced("Union", [member] + spheres)) + "\n"


SCENES = {
    "flush, a sphere behind": lambda: _flush(S.sphere((0, 0, -4), "5AC85A", 0.5)),
    "flush, a sphere in front": lambda: _flush(S.sphere((0, 0, 1.5), "5AC85A", 0.1)),
    # members: operators over cubes and spheres (all in their boxes), 24 and 25 (the smallest
    # group taken whole and one more), 65 (a second round of members), 300 (a second round of chunks)
    **{f"members{n}": lambda n=n: _group(n, n, ["cube", "sphere", "upright"]) for n in (24, 25, 65, 300)},
    "spheres and cubes": lambda: _group(48, 2, ["cube", "sphere"], ops=("Difference",)),
    # cylinders that leave their boxes, alone and within members
    "tilted24": lambda: _group(24, 3, ["tilted", "sphere"]),
    "tilted96": lambda: _group(96, 4, ["tilted", "cube", "sphere"]),
    "tilted only": lambda: _group(40, 5, ["tilted"], ops=("Difference", "Union")),
    # lists that overflow, walked in stretches
    "cut by members": lambda: _group(200, 6, ["tilted", "cube", "sphere"], wrap="Difference"),
    "common with members": lambda: _group(80, 7, ["cube", "sphere", "upright"], wrap="Intersection"),
    "stress300": lambda: S.stress(300, seed=300),
    "stress440": lambda: S.stress(440, seed=440),
    "stress1100": lambda: S.stress(1100, seed=1100),
}
VIEWS = [((0.0, 0.0, 4.0), (0.0, 0.0, 0.0), 55), ((2.2, 1.3, 2.9), (0.0, 0.01, 0.0), 45),
         ((0.05, 0.02, 0.04), (0.3, 0.1, -1.0), 90)]  # along an axis, from a corner, from inside


def _frame(scene, view, w, h, **opts):
    eye, target, fov = view
    return scene.render(C.camera_look_at(eye, target, fov), C.light(LIGHT), C.phong(*PHONG), w, h, seed=5, **opts)


def _same(got, ref, what):
    torch.cuda.synchronize()
    for key in KEYS:
        a, b = got[key].cpu().numpy(), ref[key].cpu().numpy()
        assert a.tobytes() == b.tobytes(), (what, key, int((a != b).sum()))


@pytest.mark.parametrize("mode", [C.MODE_FAST, C.MODE_EXACT], ids=["fast", "exact"])
@pytest.mark.parametrize("name", list(SCENES))
def test_groups_equal_the_state_machine(gpu, name, mode):
    scene = C.Scene(SCENES[name]())
    for (w, h, samples), view in zip([(65, 33, 1), (160, 121, 2), (403, 333, 1), (403, 333, 1), (403, 333, 2)],
                                     VIEWS + VIEWS[:2]):
        print(f"[case] {name} {w}x{h} samples {samples}", flush=True)
        got = _frame(scene, view, w, h, samples=samples, mode=mode)
        ref = _frame(scene, view, w, h, samples=samples, mode=mode, coop=-1)
        _same(got, ref, (w, h))
    scene.close()


@pytest.mark.parametrize("mode", [C.MODE_FAST, C.MODE_EXACT], ids=["fast", "exact"])
def test_groups_in_a_batch_equal_the_state_machine(gpu, mode):
    specs, refs = [], []
    for i, name in enumerate(SCENES):
        scene = C.Scene(SCENES[name]())
        eye, target, fov = VIEWS[i % 3]
        w, h = 121 + 8 * i, 96 + i
        specs.append((scene, C.camera_look_at(eye, target, fov), C.light(LIGHT), C.phong(*PHONG), w, h,
                      C.alloc_outputs(w, h)))
        refs.append(_frame(scene, VIEWS[i % 3], w, h, mode=mode, coop=-1))
    print(f"[case] batch of {len(specs)}", flush=True)
    C.render_batch(C.make_jobs(specs), mode=mode)
    for spec, ref, name in zip(specs, refs, SCENES):
        _same(spec[6], ref, name)


def test_the_first_crossing_before_a_flush_cut(gpu):
    """The ray along -z meets the cut cube's near face (primitive 0) at 3.5 with a sphere behind it."""
    scene = C.Scene(SCENES["flush, a sphere behind"]())
    out = _frame(scene, VIEWS[0], 33, 33)
    torch.cuda.synchronize()
    assert int(out["prim_id"][16, 16]) == 0
    assert abs(float(out["depth"][16, 16]) - 3.5) < 0.01
    scene.close()


def _flush_cubes(n, seed, cut=False):
    """A Union of n cubes on a grid, many with faces in one plane; `cut`: each with a flush piece cut off."""
    rng = np.random.default_rng(seed)
    leaves = []
    for _ in range(n):
        c = list(_grid(rng, 0.25))
        leaf = S.cube(c, "C85A5A", 0.5 if cut else float(rng.integers(1, 5)) * 0.25)
        if cut:
            c[int(rng.integers(0, 3))] += 0.25
            leaf = "\n".join(["Difference", leaf, S.cube(c, "5A5AC8", 0.5)])
        leaves.append(leaf)
    return "\n".join(S.balanced("Union", leaves)) + "\n"


# Unions of flush parts: too few members for a group, a group of few, 31 and 32 operators (32 and 16
# steps in a failed ray's lane), groups kept up to 3000 tiles (432x432 has 2916, 440x440 3025), and by
# the per-lane kernel: in fast mode from 48 operators and 6144 tiles on (624x624 has 6084, 632x632
# 6241), from 400 operators and 3000 tiles in both modes
@pytest.mark.parametrize("mode", [C.MODE_FAST, C.MODE_EXACT], ids=["fast", "exact"])
@pytest.mark.parametrize("n,cut", [(23, False), (24, False), (24, True), (32, False), (33, False), (48, False),
                                   (49, False), (200, True), (400, False), (401, False)])
def test_flush_unions_equal_the_state_machine(gpu, n, cut, mode):
    scene = C.Scene(_flush_cubes(n, n, cut))
    specs, refs = [], []
    for size, view in zip([97, 432, 440, 624, 632], VIEWS + VIEWS[:2]):
        print(f"[case] {n} cubes, cut {cut}, {size}x{size}", flush=True)
        got = _frame(scene, view, size, size, mode=mode)
        ref = _frame(scene, view, size, size, mode=mode, coop=-1)
        _same(got, ref, size)
        eye, target, fov = view
        specs.append((scene, C.camera_look_at(eye, target, fov), C.light(LIGHT), C.phong(*PHONG), size, size,
                      C.alloc_outputs(size, size)))
        refs.append(ref)
    small = C.Scene(S.WIKIPEDIA)
    eye, target, fov = VIEWS[1]
    specs.append((small, C.camera_look_at(eye, target, fov), C.light(LIGHT), C.phong(*PHONG), 300, 200,
                  C.alloc_outputs(300, 200)))
    refs.append(_frame(small, VIEWS[1], 300, 200, mode=mode, coop=-1))
    C.render_batch(C.make_jobs(specs), mode=mode)
    batch = C.Batch(C.make_jobs(specs), mode=mode)
    for spec, ref in zip(specs, refs):
        _same(spec[6], ref, "batch")
        for t in spec[6].values():
            t.fill_(0)
    batch.launch()
    for spec, ref in zip(specs, refs):
        _same(spec[6], ref, "captured batch")
    batch.close()
    scene.close()
    small.close()
