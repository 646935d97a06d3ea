"""Timed cases of the raster path, from the smallest call to a whole 4096^2 frame.

A case is a dict of plain values.  ``kind`` is how the program calls the library:

  frame    a frame resident on the device, rendered again (Rasterizer.frame_render)
  animate  outlines of a new frame in host memory to a frame on the device
           (scene_upload_outlines, scene_bin, frame_render)
  still    a serialised scene in host memory to a frame in host memory (raster_scene)
  jobs     the per-job boundary, host buffers in and out (queue_jobs)
  batch    many scenes in one launch replayed from a captured graph, frames read back
  fit      one step of fitting a scene to an image: new parameters (where ``update``),
           forward and backward, loss, gradients and image on the device

``content`` is what is drawn: "rects" (panels and bars of a user interface, corners
on quarter pixels), "scribbles" (random self-crossing outlines, half of them filled
nonzero) or "blobs" (rounded shapes and glyph-like outlines with solid, gradient
and texture colours).
"""
import dataclasses
import math

import numpy as np
import torch

import gudni_amd as G
from gudni_amd import scenes as S

ACCURATE, REFERENCE = 0, 1


def listed():
    return [
        # an icon redrawn: the smallest call, where launches and latency count
        {"name": "icon_64", "kind": "frame", "content": "rects", "width": 64, "height": 64, "shapes": 12,
         "tile": 256, "radix": 0, "mode": ACCURATE, "filter": 0},
        # a window of an interface whose content changes every frame
        {"name": "window_641x479", "kind": "animate", "content": "rects", "width": 641, "height": 479,
         "shapes": 300, "tile": 256, "radix": 0, "mode": ACCURATE, "filter": 0},
        # dense self-crossing outlines with both fill rules at the default spec
        {"name": "scribbles_512", "kind": "frame", "content": "scribbles", "width": 512, "height": 512,
         "shapes": 1000, "tile": 256, "radix": 0, "mode": ACCURATE, "filter": 0},
        # an animation at the reference's real-time goal of ~10,000 shapes
        {"name": "animation_1080p", "kind": "animate", "content": "blobs", "width": 1920, "height": 1080,
         "shapes": 10000, "tile": 32, "radix": 0, "mode": ACCURATE, "filter": 1},
        # the benchmark's frame: 4096^2, 200,000 shapes, its tuned tile size
        {"name": "poster_4096", "kind": "frame", "content": "blobs", "width": 4096, "height": 4096,
         "shapes": 200000, "tile": 32, "radix": 0, "mode": ACCURATE, "filter": 1},
        # the reference's own arithmetic, sampling and tile size, on a ragged canvas
        {"name": "reference_mode_1000x701", "kind": "frame", "content": "blobs", "width": 1000, "height": 701,
         "shapes": 5000, "tile": 256, "radix": 0, "mode": REFERENCE, "filter": 0},
        # one still image, host memory to host memory
        {"name": "still_800x600", "kind": "still", "content": "blobs", "width": 800, "height": 600,
         "shapes": 3000, "tile": 256, "radix": 0, "mode": ACCURATE, "filter": 1},
        # the reference's per-job call structure
        {"name": "jobs_768", "kind": "jobs", "content": "blobs", "width": 768, "height": 768, "shapes": 8000,
         "tile": 256, "radix": 0, "mode": ACCURATE, "filter": 0},
        # serving: a batch of uneven scenes, frames read back
        {"name": "batch_24", "kind": "batch", "content": "blobs", "scenes": 24, "side_lo": 256, "side_hi": 1024,
         "shapes_lo": 100, "shapes_hi": 5000, "tile": 64, "radix": 0, "mode": ACCURATE, "filter": 1},
        # fitting a small picture: the shortest training step, parameters updated on the device
        {"name": "fit_250", "kind": "fit", "content": "blobs", "scenes": 1, "side": 250, "shapes_lo": 120,
         "shapes_hi": 120, "pictures": 0, "update": True, "tile": 16, "radix": 4, "filter": 1},
        # the benchmark's differentiable scene: forward and backward
        {"name": "fit_1024", "kind": "fit", "content": "blobs", "scenes": 1, "side": 1024, "shapes_lo": 2000,
         "shapes_hi": 2000, "pictures": 0, "update": False, "tile": 16, "radix": 4, "filter": 1},
        # a batch of textured scenes, every scene's parameters updated on the device
        {"name": "fit_8x512", "kind": "fit", "content": "blobs", "scenes": 8, "side": 512, "shapes_lo": 500,
         "shapes_hi": 5000, "pictures": 1, "update": True, "tile": 16, "radix": 4, "filter": 1},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(("frame", "frame", "frame", "animate", "still", "jobs", "batch", "fit"))
    base = {"kind": kind, "tile": rng.choice((32, 64, 128, 256)), "radix": rng.choice((0, 0, 3, 4)),
            "filter": rng.choice((0, 1))}
    if kind == "batch":
        lo, shapes = _log_uniform(rng, 128, 512), _log_uniform(rng, 50, 500)
        return dict(base, content="blobs", scenes=_log_uniform(rng, 2, 32), side_lo=lo, side_hi=2 * lo + rng.randint(0, 100),
                    shapes_lo=shapes, shapes_hi=8 * shapes, mode=ACCURATE)
    if kind == "fit":
        n = _log_uniform(rng, 1, 8)
        side = _log_uniform(rng, 64, 1024 if n < 3 else 400)
        shapes = max(10, min(1500, side * side // _log_uniform(rng, 80, 2000)))
        return dict(base, content="blobs", scenes=n, side=side, shapes_lo=shapes, shapes_hi=2 * shapes,
                    pictures=rng.choice((0, 1)), update=rng.choice((True, False)), tile=rng.choice((16, 32, 64)),
                    radix=rng.choice((0, 3, 4, 5)))
    mode = rng.choice((ACCURATE, ACCURATE, ACCURATE, REFERENCE))
    content = rng.choice(("blobs", "blobs", "rects", "scribbles"))
    if content == "scribbles":
        w, h = _log_uniform(rng, 48, 512), _log_uniform(rng, 48, 512)
        shapes = max(10, max(w, h) ** 2 // _log_uniform(rng, 250, 2500))
    elif content == "rects":
        w, h = _log_uniform(rng, 16, 1920), _log_uniform(rng, 16, 1080)
        shapes = _log_uniform(rng, 4, 100 if w * h < 100_000 else 400)
    else:
        most = {"frame": 3000, "animate": 2500, "still": 1500, "jobs": 1200}[kind]
        w = _log_uniform(rng, 48, most)
        h = max(16, int(w * rng.uniform(0.5, 1.2)))
        # up to the 4096^2 frame's density, one shape per 84 pixels
        shapes = max(8, int(max(w, h) ** 2 / _log_uniform(rng, 84, 2000)))
    return dict(base, content=content, width=w, height=h, shapes=shapes, mode=mode)


# ---- content -------------------------------------------------------------------

def _rects(width, height, n, seed):
    """Interface-like panels: corners on quarter pixels, the later ones larger (the
    first shape lies on top), solid and gradient colours, opaque background."""
    rng = np.random.default_rng(seed)
    side = np.sort(np.exp(rng.uniform(np.log(2.0), np.log(max(4.0, 0.6 * max(width, height))), n)))
    w = np.maximum(0.5, np.round(4 * side * rng.uniform(0.5, 1.5, n)) / 4)
    h = np.maximum(0.5, np.round(4 * side * rng.uniform(0.2, 0.8, n)) / 4)
    x = np.round(4 * rng.uniform(-0.05 * width, 0.95 * width, n)) / 4
    y = np.round(4 * rng.uniform(-0.05 * height, 0.95 * height, n)) / 4
    colors = (rng.integers(0, 256, (n, 4)) / 255.0).astype(np.float32)
    gradient = rng.random(n) < 0.2
    records, shapes = [], []
    for i in range(n):
        tag = S.solid_tag(i)
        if gradient[i]:
            stops = (rng.integers(0, 256, (2, 4)) / 255.0).astype(np.float32)
            records.append(S.gradient_record(0, (x[i], y[i]), (x[i] + w[i], y[i] + h[i]), [0.0, 1.0], stops))
            tag = S.gradient_tag(i)
            colors[i] = S.gradient_substance(len(records) - 1)
        shapes.append((tag, [S.rectangle_pairs(x[i], y[i], x[i] + w[i], y[i] + h[i])]))
    return S.build_scene(width, height, shapes, colors, gradients=np.array(records) if records else None,
                         name="rects"), (x, y, w, h)


def _blobs(width, height, n, seed, pictures=1, k_range=(4, 16), gradients=2, texture_side=256):
    """The benchmark's blob and glyph generator on any canvas, at the overdraw of
    its 4096^2 frame; shapes lie over the enclosing square."""
    size = max(width, height)
    radius = min(max(8.0 * (size / 4096.0) * math.sqrt(200_000.0 / n), 1.5), size / 8.0)
    glyphs = max(1, n // 10)
    sc = S.blobs_4096(n_blobs=max(1, n - glyphs), n_glyphs=glyphs, size=size, seed=seed, radius_median=radius,
                      em_scale=max(0.25, radius / 8.0), picture_share=pictures, k_range=k_range,
                      gradient_share=gradients, texture_side=1024 if size > 2048 else texture_side)
    return dataclasses.replace(sc, width=width, height=height)


def _scene(case, seed):
    w, h, n = case["width"], case["height"], case["shapes"]
    if case["content"] == "rects":
        return _rects(w, h, n, seed)[0]
    if case["content"] == "scribbles":
        return dataclasses.replace(S.uniform_512(n, max(w, h), seed), width=w, height=h)
    return _blobs(w, h, n, seed)


def _members(case, seed):
    """(side, shapes, seed) of the scenes of a batch: the sizes are the case's."""
    sizes, seeds = np.random.default_rng(case["shapes_hi"]), np.random.default_rng(seed)
    lo, hi = case["shapes_lo"], case["shapes_hi"]
    out = []
    for _ in range(case["scenes"]):
        side = case["side"] if "side" in case else int(sizes.integers(case["side_lo"], case["side_hi"] + 1))
        out.append((side, int(round(math.exp(sizes.uniform(math.log(lo), math.log(hi))))), int(seeds.integers(1 << 30))))
    return out


def _fit_scene(case, side, n, seed):
    """Blobs whose outlines have the case's numbers of curves, each shape at a place
    and in a colour of the seed's."""
    sc = _blobs(side, side, n, n, pictures=case["pictures"], k_range=(3, 8 if case["pictures"] else 12), gradients=0)
    rng = np.random.default_rng(seed)
    counts = np.diff(sc.outline_pair_offsets)
    starts = sc.outline_pair_offsets[:-1]
    centre = np.add.reduceat(sc.pairs[:, :2].astype(np.float64), starts, axis=0) / counts[:, None]
    move = np.repeat(rng.uniform(0, side, centre.shape) - centre, counts, axis=0)
    pairs = (sc.pairs + np.tile(move, 2)).astype(np.float32)
    colors = (rng.integers(0, 256, sc.substances.shape) / 255.0).astype(np.float32)
    solid = (sc.tags & np.uint64(S.TAG_GRADIENT)) == np.uint64(S.TAG_SOLID)
    return dataclasses.replace(sc, pairs=pairs, substances=np.where(solid[:, None], colors, sc.substances))


# ---- the calls -----------------------------------------------------------------

def _rasterizer(case):
    spec = G.default_spec(max_tile_size=case["tile"], sort_radix_bits=case["radix"], texture_filter=case["filter"],
                          coverage_mode=case.get("mode", ACCURATE))
    r = G.Rasterizer(spec)
    r.set_stream(torch.cuda.current_stream().cuda_stream)
    return r


def prepare(case, seed):
    kind = case["kind"]
    r = _rasterizer(case)
    state = {"kind": kind, "r": r}
    if kind == "batch":
        scenes = [_blobs(side, side, n, s) for side, n, s in _members(case, seed)]
        n = len(scenes)
        state["batch"] = G.Batch.from_outlines(r, scenes, [case["tile"]] * n, [case["radix"]] * n)
        return state
    if kind == "fit":
        return _prepare_fit(case, seed, state)
    scene = _scene(case, seed)
    state["scene"] = scene
    pixels = scene.width * scene.height
    if kind in ("frame", "animate"):
        state["bgra"] = torch.zeros(pixels, dtype=torch.int32, device="cuda")
        # interface windows and the reference's arithmetic also give the colours before quantisation
        if case["content"] == "rects" or case["mode"] == REFERENCE:
            state["rgba"] = torch.zeros(pixels * 4, dtype=torch.float32, device="cuda")
    if kind == "animate":
        return state
    geometry = G.Geometry(scene)
    if kind == "still":
        state["geometry"] = geometry
        return state
    jobs = G.RasterJobs(r.spec, geometry, scene.width, scene.height)
    r.upload_common(geometry.geo, scene)
    if kind == "frame":
        r.frame_upload(jobs, scene)
    else:
        state["jobs"] = jobs
        state["out"] = np.zeros(pixels, np.uint32)
    return state


def _prepare_fit(case, seed, state):
    """Targets are renders of the scenes; the parameters are perturbed copies."""
    r = state["r"]
    items = []
    for side, n, s in _members(case, seed):
        base = _fit_scene(case, side, n, s)
        _, geometry, jobs = G.prepare(base, r.spec)
        r.upload_common(geometry.geo, base)
        r.frame_upload(jobs, base)
        bgra = torch.zeros(side * side, dtype=torch.int32, device="cuda")
        rgba = torch.zeros(side * side * 4, dtype=torch.float32, device="cuda")
        r.frame_render(bgra.data_ptr(), rgba.data_ptr())
        r.frame_check()
        items.append((S.perturb(base, s + 1), rgba.cpu().numpy().reshape(side, side, 4)))
    state["adjoint"] = G.Adjoint(r, items)
    pairs = np.concatenate([sc.pairs.reshape(-1) for sc, _ in items])
    rgba = np.concatenate([sc.substances.reshape(-1) for sc, _ in items])
    state["update"] = case["update"]
    state["pairs"] = torch.from_numpy(pairs).cuda()
    state["colors"] = torch.from_numpy(rgba).cuda()
    state["loss"] = torch.zeros(len(items), dtype=torch.float64, device="cuda")
    state["d_pairs"] = torch.zeros_like(state["pairs"])
    state["d_colors"] = torch.zeros_like(state["colors"])
    state["image"] = torch.zeros(sum(4 * sc.width * sc.height for sc, _ in items), dtype=torch.float32, device="cuda")
    return state


def run(state):
    kind, r = state["kind"], state["r"]
    if kind == "batch":
        b = state["batch"]
        b.render(use_graph=True)
        return [b.frame(i) for i in range(len(b.sizes))]
    if kind == "fit":
        a = state["adjoint"]
        if state["update"]:
            a.update_device(-1, state["pairs"].data_ptr(), state["colors"].data_ptr())
        a.run()
        a.result_device(-1, *[state[k].data_ptr() for k in ("loss", "d_pairs", "d_colors", "image")])
        return {k: state[k] for k in ("loss", "d_pairs", "d_colors", "image")}
    scene = state["scene"]
    if kind == "still":
        return {"bgra": r.raster_scene(state["geometry"], scene)}
    if kind == "jobs":
        return {"bgra": r.queue_jobs(state["jobs"], scene, state["out"])}
    if kind == "animate":
        r.scene_upload_outlines(scene)
        r.scene_bin()
    rgba = state.get("rgba")
    r.frame_render(state["bgra"].data_ptr(), rgba.data_ptr() if rgba is not None else None)
    return {"bgra": state["bgra"]} if rgba is None else {"bgra": state["bgra"], "rgba": rgba}


def work(case):
    """Outlines (animate, fit) or strands in, colours in, pixels out, each once; a
    few operations for a curve's two column borders and for a layer of a pixel."""
    if "scenes" in case:
        n = case["scenes"]
        side = case.get("side") or (case["side_lo"] + case["side_hi"]) / 2.0
        pixels = n * side * side
        lo, hi = case["shapes_lo"], case["shapes_hi"]
        shapes = n * (hi - lo) / math.log(hi / lo) if hi > lo else n * lo
    else:
        pixels, shapes = case["width"] * case["height"], case["shapes"]
    curves = shapes * {"rects": 4, "scribbles": 7.5, "blobs": 10.7}[case["content"]]
    if case["content"] == "blobs" and case["kind"] == "fit":
        curves = shapes * (6.7 if case["pictures"] else 8.4)
    read = 16 * curves + 32 * shapes + (0 if case["content"] != "blobs" else 4 * 256 * 256)
    layers = {"rects": 4, "scribbles": 60, "blobs": 17}[case["content"]]
    flops = 40 * curves + pixels * layers * 8
    if case["kind"] == "fit":
        # the target read, the image written; the gradients written; backward about twice the forward
        return {"bytes": read + 32 * pixels + 16 * curves + 16 * shapes, "flops": 3 * flops}
    wide = case["content"] == "rects" or case["mode"] == REFERENCE
    wide = wide and case["kind"] in ("frame", "animate")
    return {"bytes": read + (20 if wide else 4) * pixels, "flops": flops}


def exact(case, seed):
    """The colours of interface windows in 64 bits: every edge lies on a quarter
    pixel, so the mean over 4 x 4 sub-pixels is a pixel's exact coverage."""
    if case["content"] != "rects" or case["kind"] not in ("frame", "animate"):
        return None
    width, height = case["width"], case["height"]
    scene, (x, y, w, h) = _rects(width, height, case["shapes"], seed)
    img = np.ones((4 * height, 4 * width, 3))
    px, py = np.arange(4 * width) // 4, np.arange(4 * height) // 4
    for i in reversed(range(case["shapes"])):
        x0, x1 = (int(max(0, min(4 * width, 4 * v))) for v in (x[i], x[i] + w[i]))
        y0, y1 = (int(max(0, min(4 * height, 4 * v))) for v in (y[i], y[i] + h[i]))
        if x0 >= x1 or y0 >= y1:
            continue
        if (int(scene.tags[i]) & S.TAG_GRADIENT) == S.TAG_GRADIENT:
            rec = scene.gradients[int(scene.substances[i].view(np.uint32)[0])].astype(np.float64)
            ax, ay, bx, by = rec[2:6]
            dx, dy = bx - ax, by - ay
            t = ((px[None, x0:x1] - ax) * dx + (py[y0:y1, None] - ay) * dy) / (dx * dx + dy * dy)
            t = np.clip(t, 0.0, 1.0)[..., None]
            color = rec[12:16] + (rec[16:20] - rec[12:16]) * t
        else:
            color = scene.substances[i].astype(np.float64)[None, None]
        a = color[..., 3:]
        img[y0:y1, x0:x1] = img[y0:y1, x0:x1] * (1.0 - a) + color[..., :3] * a
    rgb = img.reshape(height, 4, width, 4, 3).mean(axis=(1, 3))
    rgba = np.concatenate([rgb, np.ones((height, width, 1))], axis=2)
    return {"bgra": None, "rgba": rgba.reshape(-1)}
