"""Performance cases of the renderer: the calls a program makes, over the sizes it makes them at.

Four kinds of work, each through the package's public entry points:

* ``frame`` -- one scene through ``VGRasterizer``.  ``how`` says what the program does:
  ``still`` redraws a resident scene, ``view`` sets the camera before every frame, ``noalloc``
  renders into the caller's buffer without allocating, ``document`` uploads the scene, renders
  it and reads the image back to the host;
* ``animation`` -- a chord-diagram frame generated on the GPU and rendered;
* ``batch`` -- many small scenes rendered by one captured graph;
* ``diff`` -- a differentiable render, forward alone or with the gradients of the control
  points and colours.

Scenes are the package's seeded generators: closed cubic chains, mixed line / quadratic /
cubic paths, glyph-like contours, and mixed paths of which a third carry gradient paints.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "gpu-scanline-path-rendering_amd"))

import scanline  # noqa: E402
from scanline import animation, diff  # noqa: E402
from scanline.gradient import GradientTextures  # noqa: E402
from scanline.scene import (KIND_CUBIC_CHAINS, KIND_GLYPHS, KIND_MIXED, SEED_BASE,  # noqa: E402
                            SceneArrays)

KINDS = {"cubics": KIND_CUBIC_CHAINS, "mixed": KIND_MIXED, "glyphs": KIND_GLYPHS, "gradients": KIND_MIXED}


def _frame(scene, width, height, paths, spp, ms=False, srgb=True, how="still", camera="flat"):
    return {"kind": "frame", "scene": scene, "width": width, "height": height, "paths": paths, "spp": spp,
            "ms": ms, "srgb": srgb, "how": how, "camera": camera}


def listed():
    return [
        # a user-interface icon: a handful of shapes, redrawn whenever its placement changes
        dict(_frame("cubics", 64, 64, 12, 8, how="view"), name="icon_64"),
        # a thumbnail of a small drawing kept on screen (the package's small configuration)
        dict(_frame("cubics", 512, 512, 200, 8), name="drawing_512"),
        # a page of text in a serving loop that may not allocate device memory
        dict(_frame("glyphs", 1240, 1754, 3000, 16, how="noalloc"), name="page_1240x1754"),
        # the headline scene: a dense illustration, coverage output
        dict(_frame("mixed", 2048, 2048, 20000, 32), name="illustration_2048"),
        # the same with the reference's default output, every sample blended
        dict(_frame("mixed", 2048, 2048, 20000, 32, ms=True), name="illustration_2048_ms"),
        # a large sheet of glyphs: the widest canvas and the most curves
        dict(_frame("glyphs", 4096, 4096, 100000, 16), name="sheet_4096"),
        # a viewer window of an odd size under a moving perspective camera, linear colour
        dict(_frame("mixed", 1279, 719, 3000, 8, ms=True, srgb=False, how="view", camera="perspective"),
             name="viewer_1279x719_ms"),
        # a poster with linear and radial gradient paints among its fills
        dict(_frame("gradients", 1024, 768, 1500, 16, how="view", camera="affine"), name="poster_1024x768"),
        # a file opened once: upload, render, image back on the host
        dict(_frame("mixed", 1000, 777, 2000, 32, how="document"), name="document_1000x777"),
        # the animation mode: two chord diagrams of 150 nodes on its 1920x1080 window
        {"name": "animation_1080p", "kind": "animation", "nodes": 150, "links": 1500, "time_ms": 9100, "spp": 16},
        # a glyph and icon cache filled in one go: many small scenes of uneven size
        {"name": "batch_1024", "kind": "batch", "scenes": 1024, "max_side": 512, "max_paths": 200},
        # one step of fitting a drawing to an image: forward and both gradients
        {"name": "fit_256", "kind": "diff", "scene": "cubics", "width": 256, "height": 256, "paths": 64,
         "segments": 6, "rows": 16, "backward": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: canvas sides, path counts and rows log-uniform (odd ones among them),
    sample counts, output modes, colour encodings, cameras and call patterns at random, and
    never more work than the largest listed case of the kind."""
    u = rng.random()
    if u < 0.68:
        scene = rng.choice(["cubics", "mixed", "mixed", "glyphs", "gradients"])
        how = rng.choice(["still", "still", "view", "view", "noalloc", "document"])
        ms, spp = rng.random() < 0.35, rng.choice([8, 16, 32])
        top = {"noalloc": 1024, "document": 2048}.get(how, 4096 if scene == "glyphs" and not ms else 2048)
        w, h = _log(rng, 24, top), _log(rng, 24, top)
        share = math.sqrt(w * h) / 2048.0
        most = {"cubics": 400, "mixed": 16000, "glyphs": 30000, "gradients": 4000}[scene] * share
        if ms:
            most *= 0.5
        if how == "noalloc":  # the frames that fit the static scratch
            most = min(most, {"cubics": 40, "mixed": 150, "glyphs": 1500, "gradients": 150}[scene])
        return _frame(scene, w, h, _log(rng, 8, max(16, most)), spp, ms=ms, srgb=rng.random() < 0.75, how=how,
                      camera=rng.choice(["flat", "affine", "perspective"]))
    if u < 0.76:
        return {"kind": "animation", "nodes": rng.randint(8, 150), "links": _log(rng, 20, 1500),
                "time_ms": rng.randint(6001, 17999), "spp": rng.choice([8, 16, 32])}
    if u < 0.84:
        return {"kind": "batch", "scenes": _log(rng, 8, 1024), "max_side": _log(rng, 32, 512),
                "max_paths": _log(rng, 8, 200)}
    w, h = _log(rng, 32, 512), _log(rng, 32, 512)
    return {"kind": "diff", "scene": rng.choice(["cubics", "mixed"]), "width": w, "height": h,
            "paths": _log(rng, 2, min(128, max(4, 2 ** 22 / (w * h)))), "segments": rng.randint(3, 8),
            "rows": rng.choice([4, 8, 16]), "backward": rng.random() < 0.75}


def _gradients(a, w, h, seed, srgb):
    """The scene with linear and radial paints of 2 to 4 stops on about a third of its paths."""
    rng = np.random.default_rng(seed)
    g = GradientTextures(srgb=srgb)
    fill = a.fill_color.copy()
    # a palette of stops, as a drawing has: building a ramp costs host time per gradient
    for p in range(a.n_paths):
        if p >= 96 or rng.random() >= 0.35:
            g.add_solid()
            continue
        n = int(rng.integers(2, 5))
        offs = np.linspace(0.0, 1.0, n)
        stops = [(float(o),) + tuple(float(v) for v in rng.random(4)) for o in offs]
        x0, y0 = rng.uniform(0, w), rng.uniform(0, h)
        tr = [1.0 + rng.normal(0, 0.2), rng.normal(0, 0.2), rng.normal(0, 10),
              rng.normal(0, 0.2), 1.0 + rng.normal(0, 0.2), rng.normal(0, 10)]
        if rng.random() < 0.5:
            g.add("linear", x0, y0, x0 + rng.uniform(20, 200), y0 + rng.uniform(20, 200), 0, stops,
                  float(rng.uniform(0.3, 1)), tr)
        else:
            g.add("radial", x0, y0, x0 + rng.normal(0, 10), y0 + rng.normal(0, 10), rng.uniform(5, 150), stops,
                  float(rng.uniform(0.3, 1)), tr)
        fill[p] = p + 1
    # the remaining paths share the gradients of the first ones
    slots = np.flatnonzero(fill[:96] != a.fill_color[:96])
    for p in range(96, a.n_paths):
        if len(slots) and rng.random() < 0.35:
            fill[p] = int(slots[rng.integers(0, len(slots))]) + 1
    ramp, table = g.textures()
    return SceneArrays(a.vertex, a.curve_vertex_pos, a.curve_type, a.curve_path_id, a.curve_arc_w, a.fill_rule,
                       fill, ramp, table)


def _scene(case, seed, paint=True):
    w, h = case["width"], case["height"]
    segs = case.get("segments", 0)
    if case["kind"] == "diff":
        seed = 1  # one topology a case: the points and paints are the seed's
    a = scanline.generate(KINDS[case["scene"]], w, h, case["paths"], SEED_BASE ^ (int(seed) * 2654435761), segs, segs)
    if case["scene"] == "gradients" and paint:
        a = _gradients(a, w, h, seed, case["srgb"])
    return a


def _batch(case, seed):
    """Closed cubic chains on canvases of log-uniform sides, 8 or 16 samples: the sizes are
    the case's, the drawings the seed's."""
    rng = np.random.default_rng(SEED_BASE)
    n, lo, hi = case["scenes"], math.log(16), math.log(case["max_side"])
    sizes = np.rint(np.exp(rng.uniform(lo, hi, (n, 2)))).astype(int).tolist()
    paths = rng.integers(4, case["max_paths"] + 1, n).tolist()
    spp = rng.choice([8, 16], n).tolist()
    seeds = np.random.default_rng(int(seed)).integers(0, 2 ** 62, n).tolist()
    scenes = [scanline.generate(KIND_CUBIC_CHAINS, w, h, p, q) for (w, h), p, q in zip(sizes, paths, seeds)]
    return scenes, sizes, spp


def _camera(case, seed):
    """A column-major 4x4 matrix, varied a little by the seed."""
    w, h = case["width"], case["height"]
    d = (seed % 7) / 7.0
    m = np.eye(4, dtype=np.float32)
    if case["camera"] == "affine":
        m[0, 0], m[1, 1], m[1, 0], m[0, 1] = 0.97 + 0.02 * d, 0.95, 0.06, -0.04
        m[3, 0], m[3, 1] = 0.01 * w + d, 0.02 * h
    elif case["camera"] == "perspective":
        m[0, 0], m[1, 1], m[1, 0] = 1.05, 0.95, 0.08
        m[3, 0], m[3, 1] = -0.02 * w, 0.01 * h + d
        m[0, 3] = 0.15 / w
        m[3, 2] = 0.05 * min(w, h)  # depth: the vanishing point behind the canvas
    return m


class _View:
    """Device bytes of `owner` as torch takes them; the tensor keeps this object, and with it
    the owner, alive."""

    def __init__(self, owner, ptr, n):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "|u1", "data": (ptr, False), "version": 2}


def prepare(case, seed):
    stream = torch.cuda.current_stream().cuda_stream
    s = {"case": case, "stream": stream}
    if case["kind"] == "diff":
        a = _scene(case, seed)
        r = diff.DiffRenderer(a, case["width"], case["height"], samples=case["rows"])
        g = torch.Generator("cuda").manual_seed(int(seed))
        noise = 0.05 * torch.randn(r.colors0.shape, generator=g, device="cuda")
        # the drawing bent by a smooth field (shared ends of segments stay shared)
        phase = 6.2832 * torch.rand((2, 1, 2), generator=g, device="cuda")
        size = torch.tensor([[float(case["width"]), float(case["height"])]], device="cuda")
        bend = torch.sin(6.2832 * r.points0.flip(1) / size.flip(1) + phase[0]) + torch.sin(9.0 * r.points0 / size + phase[1])
        s["points"] = (r.points0 + 0.04 * size * bend).contiguous()
        s["colors"] = (r.colors0 + noise).clamp(0, 1).contiguous()
        s["grad"] = torch.randn((case["height"], case["width"], 4), generator=g, device="cuda")
        if case["backward"]:
            s["points"].requires_grad_(True)
            s["colors"].requires_grad_(True)
        s["r"] = r
        return s
    if case["kind"] == "batch":
        scenes, sizes, spp = _batch(case, seed)
        b = scanline.BatchRasterizer(scenes, sizes, spp)
        s["b"] = b
        # the images of one sample count lie in one allocation: a view of each, with the
        # bytes between images cleared once
        ptr, pitch, span = ctypes.c_void_p(), ctypes.c_int(), {}
        for i, ((w, h), n) in enumerate(zip(sizes, spp)):
            b._chk(b._L.sl_batch_output_device_ptr(b._b, i, ctypes.byref(ptr), ctypes.byref(pitch)))
            lo, hi = span.get(n, (ptr.value, 0))
            span[n] = (min(lo, ptr.value), max(hi, ptr.value + h * pitch.value))
        s["images"] = [torch.as_tensor(_View(b, lo, hi - lo), device="cuda") for _, (lo, hi) in sorted(span.items())]
        for v in s["images"]:
            v.zero_()
        return s
    r = scanline.VGRasterizer(0)
    r.setSamples(case["spp"])
    r.setMultisampleOutput(case.get("ms", False))
    r.enableSRGBCorrection(case.get("srgb", True))
    s["r"] = r
    if case["kind"] == "animation":
        w, h = animation.CANVAS
        ds = animation.refugee_diagrams(n_nodes=case["nodes"], n_years=4,
                                        links_per_year=min(case["links"], case["nodes"] * (case["nodes"] - 1) // 4),
                                        seed=int(seed))
        s["anim"] = animation.ChordAnimation(r, ds)
    else:
        w, h = case["width"], case["height"]
        s["scene"] = _scene(case, seed)
        s["camera"] = _camera(case, seed)
        r.setInputTransform(s["camera"])
    r.resizeOutputBuffer(w, h)
    if case["kind"] == "frame" and case["how"] != "document":
        r.addVg(s["scene"])
    s["image"] = torch.zeros((h, w, 4), dtype=torch.uint8, device="cuda")
    return s


def run(s):
    case, stream = s["case"], s["stream"]
    if case["kind"] == "diff":
        r, p, c = s["r"], s["points"], s["colors"]
        if not case["backward"]:
            return r.forward_raw(p, c, keep=False)
        img = r.render(p, c)
        gp, gc = torch.autograd.grad(img, (p, c), s["grad"])
        return img.detach(), gp, gc
    if case["kind"] == "batch":
        s["b"].render(stream)
        return s["images"]
    r, img = s["r"], s["image"]
    h, w = img.shape[0], img.shape[1]
    if case["kind"] == "animation":
        s["anim"].frame(case["time_ms"], stream)
    elif case["how"] == "noalloc":
        r.rasterizeNoAlloc(img.data_ptr(), 4 * w, stream)
        return img
    elif case["how"] == "document":
        r.addVg(s["scene"])
        r.rasterize(stream)
        return r.output()
    elif case["how"] == "view":
        r.setInputTransform(s["camera"])
    r.rasterize(stream)
    r.present(img.data_ptr(), 4 * w, w, h, stream)
    return img


def _scene_bytes(a):
    """Each vertex (8), curve (type, path, vertex position, weight: 13) and path (5) read once."""
    return 8 * a.n_vertices + 13 * a.n_curves + 5 * a.n_paths


def work(case):
    """The scene read once and the outputs written once.  The operations depend on how the
    paths cross and cover the canvas, not on the sizes alone, and are not counted."""
    if case["kind"] == "animation":
        w, h = animation.CANVAS
        paths = 2 * (case["nodes"] + min(case["links"], case["nodes"] * (case["nodes"] - 1) // 4))
        return {"bytes": paths * 64 + 4 * w * h, "flops": 0}
    if case["kind"] == "batch":
        # sides log-uniform in [16, max_side], 8 cubics a path
        side = (case["max_side"] - 16) / math.log(case["max_side"] / 16.0)
        paths = 0.5 * (4 + case["max_paths"])
        return {"bytes": case["scenes"] * (4 * side * side + paths * (8 * (32 + 13) + 5)), "flops": 0}
    a = _scene(case, 1, paint=False)
    px = case["width"] * case["height"]
    if case["kind"] == "diff":
        n = 16 * px + 8 * a.n_vertices + 16 * a.n_paths
        if case["backward"]:
            n += 16 * px + 8 * a.n_vertices + 16 * a.n_paths
        return {"bytes": n, "flops": 0}
    return {"bytes": _scene_bytes(a) + 4 * px, "flops": 0}


# ---- the differentiable model in 64 bits ------------------------------------------------


def _basis(n, t):
    s = 1 - t
    if n == 2:
        return torch.stack([s, t], 1)
    if n == 3:
        return torch.stack([s * s, 2 * s * t, t * t], 1)
    return torch.stack([s ** 3, 3 * s * s * t, 3 * s * t * t, t ** 3], 1)


def _slope(n, v, t):
    """d/dt of the Bezier curve with control values v [N, n]."""
    d = (n - 1) * (v[:, 1:] - v[:, :-1])
    return d[:, 0] if n == 2 else (_basis(n - 1, t) * d).sum(1)


def _extrema(n, y):
    """Parameters of the y-extrema in (0, 1), ascending, 1 where there is none."""
    one = torch.ones_like(y[:, 0])
    if n == 2:
        return []
    if n == 3:
        t = (y[:, 0] - y[:, 1]) / (y[:, 0] - 2 * y[:, 1] + y[:, 2])
        return [torch.where((t > 0) & (t < 1), t, one)]
    a = -y[:, 0] + 3 * y[:, 1] - 3 * y[:, 2] + y[:, 3]
    b = 2 * (y[:, 0] - 2 * y[:, 1] + y[:, 2])
    c = y[:, 1] - y[:, 0]
    q = torch.sqrt(b * b - 4 * a * c)  # NaN without a root
    r = torch.stack([(-b - q) / (2 * a), (-b + q) / (2 * a)], 1)
    r = torch.where((r > 0) & (r < 1), r, torch.ones_like(r)).sort(1).values
    return [r[:, 0], r[:, 1]]


def exact(case, seed):
    """The image, and the gradients where they are asked for: row-sampled coverage, exact
    along x, src-over onto white, and the boundary terms of its crossings."""
    if case["kind"] != "diff":
        return None
    a = _scene(case, seed)
    s = prepare(case, seed)
    dev, f8 = s["points"].device, torch.float64
    P, W, H, S = a.n_paths, case["width"], case["height"], case["rows"]
    J = H * S
    pts, col = s["points"].detach().to(f8), s["colors"].detach().to(f8)
    ctype = torch.tensor(a.curve_type.astype(np.int64) & 7, device=dev)
    cpos = torch.tensor(a.curve_vertex_pos.astype(np.int64), device=dev)
    cpath = torch.tensor(a.curve_path_id.astype(np.int64), device=dev)
    rule = torch.tensor(a.fill_rule.astype(np.int64), device=dev)
    found = []
    for n in (2, 3, 4):
        cs = torch.nonzero(ctype == n).reshape(-1)
        if not len(cs):
            continue
        v = pts[cpos[cs][:, None] + torch.arange(n, device=dev)]  # [N, n, 2]
        x, y = v[:, :, 0], v[:, :, 1]
        ts = [torch.zeros_like(y[:, 0])] + _extrema(n, y) + [torch.ones_like(y[:, 0])]
        ys = [(_basis(n, t) * y).sum(1) for t in ts]
        for t0, t1, y0, y1 in zip(ts, ts[1:], ys, ys[1:]):
            ja = torch.ceil(torch.minimum(y0, y1) * S - 0.5).clamp(0, J).to(torch.int64)
            jb = torch.ceil(torch.maximum(y0, y1) * S - 0.5).clamp(0, J).to(torch.int64)
            m = torch.where((t1 > t0) & (jb > ja), jb - ja, torch.zeros_like(ja))
            i = torch.repeat_interleave(torch.arange(len(cs), device=dev), m)
            if not len(i):
                continue
            j = ja[i] + torch.arange(len(i), device=dev) - (torch.cumsum(m, 0) - m)[i]
            up = (y1 > y0)[i]
            row = (j.to(f8) + 0.5) / S
            lo, hi = torch.where(up, t0[i], t1[i]), torch.where(up, t1[i], t0[i])
            yi, xi = y[i], x[i]
            for _ in range(50):
                mid = 0.5 * (lo + hi)
                below = (_basis(n, mid) * yi).sum(1) < row
                lo, hi = torch.where(below, mid, lo), torch.where(below, hi, mid)
            t = 0.5 * (lo + hi)
            b = _basis(n, t)
            dy = _slope(n, yi, t)
            dy = torch.where(dy.abs() < 1e-4, torch.where(dy < 0, -1e-4, 1e-4).to(f8), dy)
            pad = torch.zeros((len(i), 4), dtype=f8, device=dev)
            pad[:, :n] = b
            at = cpos[cs[i]][:, None] + torch.arange(4, device=dev).clamp(max=n - 1)
            found.append((cpath[cs[i]] * J + j, (b * xi).sum(1), torch.where(up, 1, -1), pad, at, _slope(n, xi, t) / dy))
    key, x, d, b, at, ratio = (torch.cat(v) for v in zip(*found)) if found else (torch.zeros(0, device=dev),) * 6
    cov = torch.zeros((P * H, W + 2), dtype=f8, device=dev)
    if found:
        o = torch.argsort(x)
        o = o[torch.argsort(key[o], stable=True)]
        key, x, d, b, at, ratio = key[o], x[o], d[o], b[o], at[o], ratio[o]
        run_sum = torch.cumsum(d, 0)
        first = torch.ones_like(key, dtype=torch.bool)
        first[1:] = key[1:] != key[:-1]
        start = torch.cummax(torch.where(first, torch.arange(len(key), device=dev), 0), 0).values
        w1 = run_sum - (run_sum - d)[start]
        w0 = w1 - d
        odd = rule[key // J] == 1
        inside = lambda w: torch.where(odd, w % 2 != 0, w != 0).to(f8)  # noqa: E731
        turn = inside(w1) - inside(w0)
        line = key // J * H + key % J // S
        u = x.clamp(0, W)
        p = torch.floor(u)
        flat = line * (W + 2) + p.to(torch.int64)
        step = torch.zeros((P * H * (W + 2),), dtype=f8, device=dev)
        step.index_add_(0, flat + 1, turn / S)
        cov = torch.cumsum(step.reshape(P * H, W + 2), 1)
        cov.view(-1).index_add_(0, flat, turn * (p + 1 - u) / S)
    cov = cov[:, :W].reshape(P, H, W)
    img = torch.ones((H, W, 4), dtype=f8, device=dev)
    before = []
    for k in range(P):
        before.append(img if case["backward"] else None)
        al = (col[k, 3] * cov[k])[:, :, None]
        src = torch.cat([col[k, :3].expand(H, W, 3) * al, al * al], 2)
        img = src + img * (1 - al)
    if not case["backward"]:
        return img
    g = s["grad"].to(f8)
    gcov = torch.zeros((P, H, W), dtype=f8, device=dev)
    gcol = torch.zeros((P, 4), dtype=f8, device=dev)
    for k in range(P - 1, -1, -1):
        al = col[k, 3] * cov[k]
        da = (g[:, :, :3] * (col[k, :3] - before[k][:, :, :3])).sum(2) + g[:, :, 3] * (2 * al - before[k][:, :, 3])
        gcov[k] = da * col[k, 3]
        gcol[k, :3] = (g[:, :, :3] * al[:, :, None]).sum((0, 1))
        gcol[k, 3] = (da * cov[k]).sum()
        g = g * (1 - al)[:, :, None]
    gpts = torch.zeros_like(pts)
    if found:
        on = (x >= 0) & (x < W) & (turn != 0)
        at, b, ratio = at[on], b[on], ratio[on]
        gx = gcov.view(-1)[line[on] * W + torch.floor(x[on]).to(torch.int64)] * -turn[on] / S
        for k in range(4):
            gpts[:, 0].index_add_(0, at[:, k], gx * b[:, k])
            gpts[:, 1].index_add_(0, at[:, k], -gx * ratio * b[:, k])
    return img, gpts, gcol
