"""Render workloads timed from the outside: what a program that uses this
library asks of it, through the Python binding of its C ABI.

Each case is a frame, a set of frames or a stream of requests.  `kind` names
the entry point: "frame" (Scene.render), "batch" (render_batch), "graph" (a
captured Batch updated each pass) and "serve" (Server).  `scene`
names one of the library's own scene generators and `size` its primitive
count (the tree count for "batch", "graph" and "serve").
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "cuda-csg-tree-raycasting_amd"))
import csgray as C  # noqa: E402
from csgray import scenes as S  # noqa: E402

BACKGROUND = (0.08, 0.08, 0.11, 1.0)


def _frame(name, scene, size, width, height, mode="fast", samples=1, view="orbit"):
    return {"name": name, "kind": "frame", "scene": scene, "size": size, "width": width, "height": height,
            "mode": mode, "samples": samples, "view": view}


def _many(name, kind, size, resolutions):
    return {"name": name, "kind": kind, "scene": "mix", "size": size, "resolutions": resolutions, "mode": "fast",
            "samples": 1}


def listed():
    return [
        # a preview of a small model: the time is launches and latency
        _frame("preview_128x72", "wikipedia", 5, 128, 72),
        # the textbook model at the size the reference's CPU tests use
        _frame("wikipedia_640x360", "wikipedia", 5, 640, 360),
        # the interactive window of the reference (ragged: 871 x 601, its default camera)
        _frame("window_871x601", "cheese", 256, 871, 601, view="default"),
        # the headline frame
        _frame("cheese512_1080p", "cheese", 512, 1920, 1080),
        # reproducible pictures: the mode whose bits are the reference's
        _frame("exact_640x360", "cheese", 512, 640, 360, mode="exact"),
        # an antialiased still
        _frame("still_1080p_4spp", "wikipedia", 5, 1920, 1080, samples=4),
        # one mixed tree of spheres, tilted cylinders and cubes
        _frame("tree_1023", "tree", 200, 1023, 1023),
        # a part that was cut one operation after another: a deep, narrow tree
        _frame("chain_800x600", "chain", 41, 800, 600),
        # a large model, antialiased: too large for on-chip memory
        _frame("large_1080p_4spp", "stress", 4095, 1920, 1080, samples=4),
        # thumbnails and previews of many models in one call
        _many("batch_48", "batch", 48, "128 256 512 1024"),
        # the same scenes frame after frame, cameras moving, as a captured graph
        _many("graph_24", "graph", 24, "256 512"),
        # requests against resident models
        _many("serve_32", "serve", 32, "256 512 1024"),
    ]


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "frame", "batch", "graph", "serve"])
    if kind != "frame":
        n = int(round(math.exp(rng.uniform(math.log(2), math.log(48)))))
        sizes = sorted(rng.sample([97, 128, 200, 256, 333, 512, 640], 3))
        return {"kind": kind, "scene": "mix", "size": n, "resolutions": " ".join(str(s) for s in sizes),
                "mode": rng.choice(["fast", "fast", "exact"]) if kind == "batch" and n <= 8 else "fast",
                "samples": 1}
    scene = rng.choice(["wikipedia", "cheese", "cheese", "tree", "tree", "chain", "stress"])
    lo, hi = {"wikipedia": (5, 5), "cheese": (8, 1500), "tree": (2, 900), "chain": (3, 60),
              "stress": (300, 4095)}[scene]
    size = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    mode = rng.choice(["fast", "fast", "fast", "exact"])
    samples = rng.choice([1, 1, 1, 2, 4])
    width = int(round(math.exp(rng.uniform(math.log(64), math.log(1920)))))
    # the machine that reproduces the reference's bits walks every ray: smaller frames
    if mode == "exact" and scene in ("tree", "stress"):
        width, samples = min(width, 640), 1
    height = max(2, int(round(width * rng.choice([0.5625, 0.75, 1.0]))))
    return {"kind": "frame", "scene": scene, "size": size, "width": width, "height": height, "mode": mode,
            "samples": samples, "view": rng.choice(["orbit", "orbit", "default"])}


# ---- inputs -----------------------------------------------------------------

def _colour(rng):
    return "%02X%02X%02X" % tuple(int(v) for v in rng.integers(40, 256, size=3))


def _tree(n, rng):
    """A balanced tree over n spheres, tilted cylinders and cubes: half Unions (the top two
    levels all), the rest Differences and Intersections."""
    leaves = []
    for _ in range(n):
        c = rng.uniform(-1.0, 1.0, size=3)
        kind = int(rng.integers(0, 3))
        if kind == 0:
            leaves.append(S.sphere(c, _colour(rng), rng.uniform(0.1, 0.8)))
        elif kind == 1:
            leaves.append(S.cylinder(c, _colour(rng), rng.uniform(0.1, 0.6), rng.uniform(0.5, 2.0),
                                     rng.uniform(0.0, 180.0, size=3)))
        else:
            leaves.append(S.cube(c, _colour(rng), rng.uniform(0.2, 1.5)))
    out = []

    def rec(lo, hi, level):
        if hi - lo == 1:
            out.append(leaves[lo])
            return
        mid = lo + (hi - lo + 1) // 2
        out.append("Union" if level < 2 else str(rng.choice(["Union", "Union", "Difference", "Intersection"])))
        rec(lo, mid, level + 1)
        rec(mid, hi, level + 1)

    rec(0, n, 0)
    return "\n".join(out) + "\n"


def _chain(n, rng):
    """A cube cut by n - 1 spheres and tilted drill holes, one Difference after another."""
    cuts = []
    for i in range(n - 1):
        c = rng.uniform(-1.0, 1.0, size=3)
        if i % 3 == 2:
            cuts.append(S.cylinder(c, _colour(rng), rng.uniform(0.05, 0.15), rng.uniform(1.0, 2.5),
                                   rng.uniform(0.0, 180.0, size=3)))
        else:
            cuts.append(S.sphere(c, _colour(rng), rng.uniform(0.15, 0.35)))
    return "\n".join(["Difference"] * (n - 1) + [S.cube((0, 0, 0), "E0E0E0", 2.0)] + cuts) + "\n"


def _jobs(case, seed):
    """[(scene text, (eye, target, vfov in degrees), width, height)] of a case."""
    rng = np.random.default_rng([seed, 0xC5C])
    if case["scene"] == "mix":
        mix = S.batch_mix(case["size"], seed=int(rng.integers(1 << 31)))
        return [(text, (eye, (0.0, 0.0, 0.0), 60.0), size, size)
                for (text, eye, _), size in zip(mix, _mix_sizes(case))]
    n, sub = case["size"], int(rng.integers(1 << 31))
    text = {"wikipedia": lambda: S.WIKIPEDIA, "cheese": lambda: S.cheese(n, seed=sub),
            "stress": lambda: S.stress(n, seed=sub), "tree": lambda: _tree(n, np.random.default_rng(sub)),
            "chain": lambda: _chain(n, np.random.default_rng(sub))}[case["scene"]]()
    if case["view"] == "default":  # the reference's camera, moved a little
        eye = tuple(np.array([0.0, 0.0, 5.0]) + rng.uniform(-0.05, 0.05, size=3))
        view = (eye, (eye[0], eye[1], 0.0), 90.0)
    else:  # about the named view (3, 2.5, 4)
        eye = tuple(np.array(S.VIEW_EYE) * rng.uniform(0.95, 1.05, size=3))
        view = (eye, (0.0, 0.0, 0.0), 60.0)
    return [(text, view, case["width"], case["height"])]


def _mix_sizes(case):
    res = [int(s) for s in case["resolutions"].split()]
    return [res[i % len(res)] for i in range(case["size"])]


def _cam(view):
    return C.camera_look_at(view[0], view[1], view[2])


def prepare(case, seed):
    jobs = _jobs(case, seed)
    st = {"case": case, "seed": seed & 0xFFFF, "light": C.light(S.LIGHT_TOWARD), "phong": C.phong(*S.PHONG),
          "mode": C.MODE_EXACT if case["mode"] == "exact" else C.MODE_FAST}
    st["scenes"] = [C.Scene(text) for text, _, _, _ in jobs]
    st["cams"] = [_cam(v) for _, v, _, _ in jobs]
    st["sizes"] = [(w, h) for _, _, w, h in jobs]
    if case["kind"] == "frame":
        st["all"] = C.alloc_outputs(*st["sizes"][0], case["samples"])
        st["outs"] = [st["all"]]
    else:  # one buffer per output, the jobs' pictures one after another
        total = sum(w * h for w, h in st["sizes"])
        st["all"] = {k: v.reshape(total, -1) for k, v in C.alloc_outputs(total, 1).items()}
        st["outs"], first = [], 0
        for w, h in st["sizes"]:
            st["outs"].append({k: v[first:first + w * h] for k, v in st["all"].items()})
            first += w * h
    if case["kind"] in ("batch", "graph"):
        specs = [(sc, cam, st["light"], st["phong"], w, h, o)
                 for sc, cam, (w, h), o in zip(st["scenes"], st["cams"], st["sizes"], st["outs"])]
        st["jobs"] = C.make_jobs(specs)
        if case["kind"] == "graph":
            st["batch"] = C.Batch(st["jobs"])
    elif case["kind"] == "serve":
        st["server"] = C.Server(streams=2, max_batch_jobs=64)
        st["ids"] = [st["server"].add_scene(sc) for sc in st["scenes"]]
    return st


def run(st):
    case = st["case"]
    if case["kind"] == "frame":
        w, h = st["sizes"][0]
        return st["scenes"][0].render(st["cams"][0], st["light"], st["phong"], w, h, mode=st["mode"],
                                      outputs=st["outs"][0], samples=case["samples"], seed=st["seed"])
    if case["kind"] == "batch":
        C.render_batch(st["jobs"], mode=st["mode"])
        return st["all"]
    if case["kind"] == "graph":
        st["batch"].update(st["jobs"])  # this frame's cameras
        st["batch"].launch()
        return st["all"]
    server = st["server"]
    tickets = [server.submit(i, cam, st["light"], st["phong"], w, h)
               for i, cam, (w, h) in zip(st["ids"], st["cams"], st["sizes"])]
    for t, o in zip(tickets, st["outs"]):
        server.wait(t)
        server.copy(t, o)
        server.release(t)
    return st["all"]


def work(case):
    """One pass: every output written once (RGBA 16 B, depth 4 B, id 4 B,
    flags 1 B a ray) and the scenes read once; a ray's generation, the test
    of the model's box, and for the quarter of the rays that hit one
    primitive's intersection, hit details and shading."""
    if case["scene"] == "mix":
        rays = sum(r * r for r in _mix_sizes(case))
        prims = case["size"] * 164  # the mean of exp(U[ln 2, ln 1024])
    else:
        rays = case["width"] * case["height"] * case["samples"]
        prims = case["size"]
    return {"bytes": rays * 25 + prims * (32 + 16 + 24), "flops": rays * (50 + 26 + (37 + 112) // 4)}


# ---- the same picture in 64 bits --------------------------------------------

_EXACT_LIMIT = 2_400_000_000  # rays x nodes that take well under 20 s


def _parse(text):
    """(tree, primitives): a tree node is an int (a primitive) or (operator, children)."""
    tok = text.split()
    prims, pos = [], 0

    def node():
        nonlocal pos
        key = tok[pos]
        pos += 1
        if key in ("Union", "Difference", "Intersection"):
            a, b = node(), node()
            if key == "Union":  # one node for a run of Unions
                kids = []
                for c in (a, b):
                    kids += c[1] if isinstance(c, tuple) and c[0] == "Union" else [c]
                return (key, kids)
            return (key, [a, b])
        n = {"Sphere": 5, "Cube": 5, "Cylinder": 9}[key]
        f = tok[pos:pos + n]
        pos += n
        p = {"type": key, "c": [float(np.float32(v)) for v in f[:3]],
             "rgb": [int(f[3][i:i + 2], 16) / 255.0 for i in (0, 2, 4)],
             "s": float(np.float32(f[4]))}
        if key == "Cylinder":
            p["h"] = float(np.float32(f[5]))
            rx, ry, rz = (math.radians(float(v)) for v in f[6:])
            v = np.array([-math.sin(rz) * math.cos(ry) + math.sin(ry) * math.sin(rx) * math.cos(rz),
                          math.cos(rx) * math.cos(rz),
                          math.sin(ry) * math.sin(rz) + math.sin(rx) * math.cos(ry) * math.cos(rz)])
            p["axis"] = list(v / np.linalg.norm(v))
        prims.append(p)
        return len(prims) - 1

    sys.setrecursionlimit(max(sys.getrecursionlimit(), 4000))
    return node(), prims


def _slab(o, d, lo, hi):
    a, b = (lo - o) / d, (hi - o) / d
    return torch.minimum(a, b), torch.maximum(a, b)


def _interval(p, o, d):
    """Entry and exit distances (inf, -inf: none) of one primitive along rays d [R, 3] from o [3]."""
    c = torch.tensor(p["c"], dtype=torch.float64, device=d.device)
    inf = math.inf
    if p["type"] == "Sphere":
        oc = o - c
        b = d @ oc
        f = oc - b[:, None] * d
        disc = p["s"] ** 2 - (f * f).sum(1)
        sq = disc.clamp(min=0).sqrt()
        e, x, ok = -b - sq, -b + sq, disc >= 0
    elif p["type"] == "Cube":
        n, m = _slab(o, d, c - p["s"] / 2, c + p["s"] / 2)
        e, x = n.amax(1), m.amin(1)
        ok = e <= x
    else:
        v = torch.tensor(p["axis"], dtype=torch.float64, device=d.device)
        oc = o - c
        dv, ov = d @ v, oc @ v
        dp, op = d - dv[:, None] * v, oc - ov * v
        qa, qb = (dp * dp).sum(1), dp @ op
        disc = qb * qb - qa * (op @ op - p["s"] ** 2)
        sq = disc.clamp(min=0).sqrt()
        n, m = _slab(ov, dv, torch.tensor(-p["h"] / 2, device=d.device), torch.tensor(p["h"] / 2, device=d.device))
        e, x = torch.maximum((-qb - sq) / qa, n), torch.minimum((-qb + sq) / qa, m)
        # the reference tests a box of max(h/2, r) about the centre first
        half = max(p["h"] / 2, p["s"])
        bn, bm = _slab(o, d, c - half, c + half)
        ok = (disc >= 0) & (e <= x) & (bn.amax(1) <= bm.amin(1)) & (bm.amin(1) > 0)
    return torch.where(ok, e, torch.full_like(e, inf)), torch.where(ok, x, torch.full_like(x, -inf))


def _inside(tree, e, x, t):
    def ev(n):
        if isinstance(n, int):
            return (e[n] <= t) & (t < x[n])
        if n[0] == "Union":
            leaves = [c for c in n[1] if isinstance(c, int)]
            out = None
            if leaves:
                if len(leaves) == leaves[-1] - leaves[0] + 1:
                    le, lx = e[leaves[0]:leaves[-1] + 1], x[leaves[0]:leaves[-1] + 1]
                else:
                    le, lx = e[leaves], x[leaves]
                out = ((le <= t) & (t < lx)).any(0)
            for c in n[1]:
                if not isinstance(c, int):
                    out = ev(c) if out is None else out | ev(c)
            return out
        a, b = ev(n[1][0]), ev(n[1][1])
        return a & ~b if n[0] == "Difference" else a & b

    return ev(tree)


def _normal(p, pts):
    c = torch.tensor(p["c"], dtype=torch.float64, device=pts.device)
    q = pts - c
    if p["type"] == "Sphere":
        n = q
    elif p["type"] == "Cube":
        a = q.abs() / (p["s"] / 2)
        n = torch.where(a > 1 - 1e-5, q.sign(), torch.zeros_like(q))
    else:
        v = torch.tensor(p["axis"], dtype=torch.float64, device=pts.device)
        m = q @ v
        side = q - m[:, None] * v
        rim = ((side * side).sum(1).sqrt() - p["s"]).abs()
        cap = (m.abs() - p["h"] / 2).abs() < rim
        n = torch.where(cap[:, None], m.sign()[:, None] * v, side)
    return n / (n * n).sum(1, keepdim=True).sqrt().clamp(min=1e-300)


def _jitter(seed, pixel, sample, axis):
    m = 0xFFFFFFFF
    h = (seed ^ (pixel * 0x9E3779B1 & m) ^ (sample * 0x85EBCA77 & m) ^ (axis * 0xC2B2AE3D & m)) & m
    h = h ^ (h >> 16)
    h = h * 0x7FEB352D & m
    h = h ^ (h >> 15)
    h = h * 0x846CA68B & m
    h = h ^ (h >> 16)
    return (h >> 8).double() / 16777216.0


def _picture(text, view, w, h, spp, seed, dev):
    tree, prims = _parse(text)
    eye, target, deg = view
    o = np.array([float(np.float32(v)) for v in eye])
    f = np.array(target) - o
    f = f / np.linalg.norm(f)
    lim = 89.0 * 3.14159 / 180.0
    pitch, yaw = max(-lim, min(lim, math.asin(f[1]))), math.atan2(-f[0], -f[2])
    pitch, yaw = float(np.float32(pitch)), float(np.float32(yaw))
    fwd = np.array([-math.sin(yaw) * math.cos(pitch), math.sin(pitch), -math.cos(yaw) * math.cos(pitch)])
    right = np.array([math.cos(yaw), 0.0, -math.sin(yaw)])
    up = np.cross(fwd, right)
    tan = math.tan(float(np.float32(np.float32(deg) * np.float32(3.14159) / np.float32(180))) / 2)
    t64 = lambda a: torch.tensor(np.asarray(a), dtype=torch.float64, device=dev)  # noqa: E731
    o_t, fwd, right, up = t64(o), t64(fwd), t64(right), t64(up)
    light = t64(S.LIGHT_TOWARD)
    light = light / light.norm()
    ka, kd, ks, shin = S.PHONG
    depth = torch.full((h * w * spp,), math.inf, dtype=torch.float64, device=dev)
    rgba = t64(BACKGROUND).repeat(h * w * spp, 1)
    step = max(1, 48_000_000 // len(prims))
    for first in range(0, h * w * spp, step):
        idx = torch.arange(first, min(first + step, h * w * spp), device=dev)
        pixel, sample = idx // spp, idx % spp
        px, py = (pixel % w).double(), (pixel // w).double()
        if spp > 1:
            ox, oy = _jitter(seed, pixel, sample, 0), _jitter(seed, pixel, sample, 1)
        else:
            ox = oy = 0.5
        nx = (2 * (px + ox) / (w - 1) - 1) * (w / h) * tan
        ny = (1 - 2 * (py + oy) / (h - 1)) * tan
        d = nx[:, None] * right + ny[:, None] * up + fwd
        d = d / (d * d).sum(1, keepdim=True).sqrt()
        ev = [_interval(p, o_t, d) for p in prims]
        e, x = torch.stack([a for a, _ in ev]), torch.stack([b for _, b in ev])
        del ev
        live = torch.nonzero((x > 0).any(0)).flatten()
        e, x = e[:, live], x[:, live]
        t = torch.zeros(live.numel(), dtype=torch.float64, device=dev)
        was = _inside(tree, e, x, t)
        while live.numel():
            ne = torch.where(e > t, e, math.inf).min(0)
            nx_ = torch.where(x > t, x, math.inf).min(0)
            t = torch.minimum(ne.values, nx_.values)
            prim = torch.where(ne.values <= nx_.values, ne.indices, nx_.indices)
            # (surfaces that coincide change together)
            now = _inside(tree, e, x, t + 1e-9)
            changed = (now != was) & (t < math.inf)
            t = torch.where(changed, t, t + 1e-9)
            hit = torch.nonzero(changed).flatten()
            if hit.numel():
                r, th, pr = live[hit], t[hit], prim[hit]
                depth[idx[r]] = th
                for k in torch.unique(pr).tolist():
                    sel = pr == k
                    rr, dd = idx[r[sel]], d[r[sel]]
                    pts = o_t + th[sel][:, None] * dd
                    n = _normal(prims[k], pts)
                    n = torch.where(((n * dd).sum(1) > 0)[:, None], -n, n)  # the surface faces the viewer
                    refl = 2 * (n @ light)[:, None] * n - light
                    diff = (n @ light).clamp(min=0)
                    spec = (-(dd * refl).sum(1)).clamp(min=0) ** shin
                    lum = ka + kd * diff + ks * spec
                    rgba[rr, :3] = (t64(prims[k]["rgb"]) * lum[:, None]).clamp(0, 1)
                    rgba[rr, 3] = 1.0
            keep = torch.nonzero(~changed & (t < math.inf)).flatten()
            live, t, was = live[keep], t[keep], was[keep]
            e, x = e[:, keep], x[:, keep]
    return {"rgba": rgba.reshape(h, w * spp, 4), "depth": depth.reshape(h, w * spp), "prim_id": None, "flags": None}


def exact(case, seed):
    jobs = _jobs(case, seed)
    total = sum(text.count("\n") * w * h * case["samples"] for text, _, w, h in jobs)
    if total > _EXACT_LIMIT or len(jobs) > 4:
        return None
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    pics = [_picture(text, v, w, h, case["samples"], seed & 0xFFFF, dev) for text, v, w, h in jobs]
    if case["kind"] == "frame":
        return pics[0]
    return {"rgba": torch.cat([p["rgba"].reshape(-1, 4) for p in pics]),
            "depth": torch.cat([p["depth"].reshape(-1, 1) for p in pics]), "prim_id": None, "flags": None}
