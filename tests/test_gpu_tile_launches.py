"""Batches of several launches (1024 jobs each) through the tile kernel: a
launch whose trees need no cooperative kernel hands no rays over, whatever the
launch before it did."""
import numpy as np
import pytest
import torch
import csgray as C
from csgray import scenes as S

pytestmark = pytest.mark.gpu

KEYS = ("rgba", "depth", "prim_id", "flags")
LIGHT, PHONG = (0.4, 0.7, 0.6), (0.2, 0.7, 0.3, 16.0)


def _flush_cubes(seed=174):
    """Eight cubes with many flush faces under seven operators: some rays meet ties they must trace to the end."""
    rng = np.random.default_rng(seed)
    cubes = [S.cube(tuple(float(v) * 0.5 for v in rng.integers(-2, 3, 3)), "C85A5A", float(rng.integers(1, 4)) * 0.5)
             for _ in range(8)]
    return "\n".join(S.random_ops_balanced(rng, cubes)) + "\n"


def test_a_later_launch_of_small_trees_finishes_its_rays(gpu):
    small = C.Scene(_flush_cubes())
    # 33 primitives, out of sight: a launch with this tree has a cooperative kernel, which its failed
    # rays go to after 16 steps, and gives it no rays itself
    other = C.Scene("\n".join(S.balanced("Union", [S.sphere((30 + i, 0, 0), "5AC85A", 0.2) for i in range(33)])) + "\n")
    cam, light, phong = C.camera_look_at((2.2, 1.3, 2.9), (0, 0, 0), 45), C.light(LIGHT), C.phong(*PHONG)
    ref = small.render(cam, light, phong, 48, 48, coop=-1)
    far = other.render(cam, light, phong, 8, 8, coop=-1)
    out, rest = C.alloc_outputs(48, 48), [C.alloc_outputs(8, 8) for _ in range(1024)]

    def clear():
        for o in [out] + rest:
            for t in o.values():
                t.fill_(77)

    # in one launch the small tree's rays do go to the cooperative kernel
    clear()
    before = C.coop_rays()
    C.render_batch(C.make_jobs([(small, cam, light, phong, 48, 48, out), (other, cam, light, phong, 8, 8, rest[0])]))
    assert C.coop_rays() > before
    for key in KEYS:
        assert torch.equal(out[key].view(torch.uint8), ref[key].view(torch.uint8)), key
    # in the second of two launches, the first of which has a cooperative kernel, they end in their lanes
    clear()
    before = C.coop_rays()
    print("[case] 1024 + 1 jobs", flush=True)
    C.render_batch(C.make_jobs([(other, cam, light, phong, 8, 8, o) for o in rest] +
                               [(small, cam, light, phong, 48, 48, out)]))
    assert C.coop_rays() == before
    for key in KEYS:
        assert torch.equal(out[key].view(torch.uint8), ref[key].view(torch.uint8)), key
        for o in rest:
            assert torch.equal(o[key].view(torch.uint8), far[key].view(torch.uint8)), key
    # and the stream's next hand-over finds an empty list
    clear()
    C.render_batch(C.make_jobs([(small, cam, light, phong, 48, 48, out), (other, cam, light, phong, 8, 8, rest[0])]))
    torch.cuda.synchronize()
    for key in KEYS:
        assert torch.equal(out[key].view(torch.uint8), ref[key].view(torch.uint8)), key
    small.close()
    other.close()


# A launch keeps the per-lane kernel for large trees with groups in few tiles (64x64: 64 tiles; 1000
# spheres to 327 tiles, 144x144 324 and 152x152 361) unless its other jobs, small trees or large ones, outweigh them
@pytest.mark.parametrize("mode", [C.MODE_FAST, C.MODE_EXACT], ids=["fast", "exact"])
@pytest.mark.parametrize("others", ["none", "small", "large"])
@pytest.mark.parametrize("n,size", [(447, 64), (448, 64), (1000, 144), (1000, 152)])
def test_large_trees_in_few_tiles(gpu, n, size, others, mode):
    light, phong = C.light(LIGHT), C.phong(*PHONG)
    cam = C.camera_look_at((2.2, 1.3, 2.9), (0, 0, 0), 55)
    big, wiki = C.Scene(S.cheese(n, seed=n)), C.Scene(S.WIKIPEDIA)
    mixed = C.Scene("\n".join(S.random_ops_balanced(np.random.default_rng(3), [
        S.cube(tuple(np.random.default_rng(i).uniform(-1, 1, 3)), "3CC850", 0.8) for i in range(80)])) + "\n")
    scenes = {"none": [(big, size)] * 34, "small": [(big, size)] + [(wiki, 400)] * 3,
              "large": [(big, size)] + [(mixed, 400)] * 3}[others]
    specs = [(sc, cam, light, phong, s, s, C.alloc_outputs(s, s)) for sc, s in scenes]
    refs = {sc: sc.render(cam, light, phong, s, s, mode=mode, coop=-1) for sc, s in scenes}
    jobs = C.make_jobs(specs)
    print(f"[case] {n} spheres {size}x{size}, others {others}", flush=True)
    batch = C.Batch(jobs, mode=mode)
    for launch in (lambda: C.render_batch(jobs, mode=mode), batch.launch):
        for spec in specs:
            for t in spec[6].values():
                t.fill_(77)
        launch()
        torch.cuda.synchronize()
        for spec in specs:
            for key in KEYS:
                assert torch.equal(spec[6][key].view(torch.uint8), refs[spec[0]][key].view(torch.uint8)), key
    batch.close()
    for sc in (big, wiki, mixed):
        sc.close()


def test_the_tuner_says_which_kernel_it_kept(gpu):
    """What autotune reports gives the same choice again: block 0 where whole tiles were
    faster, else the reported block (which turns whole tiles off)."""
    light, phong = C.light(LIGHT), C.phong(*PHONG)
    specs = [(C.Scene(text), C.camera_look_at(eye, (0, 0, 0), 60), light, phong, size, size,
              C.alloc_outputs(size, size)) for text, eye, size in S.batch_mix(12, seed=5, resolutions=(128, 256))]
    jobs = C.make_jobs(specs)
    for opts, tiles in [({}, True), ({"block": 256}, False), ({"coop": -1}, False)]:
        batch = C.Batch(jobs, **opts)
        assert batch.whole_tiles() == tiles, opts
        batch.close()
    batch = C.Batch(jobs)
    t = batch.autotune(reps=2)
    again = C.Batch(jobs, block=0 if batch.whole_tiles() else t.block, walk=t.tile_walk)
    assert again.whole_tiles() == batch.whole_tiles()
    got = []
    for b in (batch, again):
        b.launch()
        torch.cuda.synchronize()
        got.append([{k: spec[6][k].clone() for k in KEYS} for spec in specs])
        b.close()
    for x, y in zip(*got):
        for key in KEYS:
            assert torch.equal(x[key].view(torch.uint8), y[key].view(torch.uint8)), key
    with pytest.raises(C.CsgError):
        C._check(C.lib().csg_batch_whole_tiles(None, None))
