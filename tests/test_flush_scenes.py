"""Loading scenes whose parts share planes: the search for flush faces takes
any numbers the parser takes, and many parts in one plane."""
import time

import csgray as C
from csgray import scenes as S


def _union(leaves):
    return "\n".join(S.balanced("Union", leaves)) + "\n"


def test_faces_that_are_no_numbers():
    odd = [f"Cube {x} 0 0 C85A5A {e}" for x in ("nan", "inf", "-inf", "3e38", "0", "-0") for e in ("1", "0", "-1", "3e38", "nan")]
    odd += [f"Cylinder 0 {y} 0 C85A5A {r} {h} 0 0 0" for y in ("nan", "0", "3e38") for r in ("1", "inf") for h in ("1", "-2")]
    scene = C.Scene(_union(odd), upload=False)
    assert scene.info().primitives == len(odd) and scene.info().union_groups == 1
    scene.close()


def test_many_parts_in_one_plane_load_quickly():
    leaves = [S.cube((0.25 * (i % 90), 0.25 * (i // 90), 0), "C85A5A", 1.0) for i in range(8100)]
    leaves += [S.cube((0, 0, 0), "C85A5A", 1.0)] * 900
    t0 = time.perf_counter()
    scene = C.Scene(_union(leaves), upload=False)
    assert scene.info().primitives == 9000
    assert time.perf_counter() - t0 < 5.0
    scene.close()
