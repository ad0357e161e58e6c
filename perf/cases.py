"""The work that is timed: calls a user's program makes through slimtracin_amd.

One case is one call pattern of the public entry points at one size:

  pick      what the editor does on a mouse press: st.pick at a few window points
  frame     one frame of one resident scene, as a viewer asks for it: FloatPixels with or without hit
            records (render, render_noalloc, render_batch with a replayed graph) or the BGRA8 window image
  moving    an animation frame: primitives moved, scene BVH rebuilt on the device, frame rendered
  rebuild   a crowd of implicit primitives moved and its scene BVH rebuilt and read back
  batch     many requests of mixed sizes, depths and modes over several scenes in one launch
  served    a burst of such requests through the server, every image taken back
  admit     a scene with a large mesh brought in (device build), its first preview frame, and out again

Scenes are the library's seeded ones at the sizes that its tests and benchmark use or smaller, so that inputs are
quickly made: 16 implicit primitives; one noise-displaced icosphere of 20 k^2 triangles with glass, mirror, floor, 4
point lights and 2 emissive quads; instances of three textured meshes sampled with ray cones. Meshes get each of the
three builders. Frames go to page-locked arrays where a program that renders in a loop would keep them.
"""
from __future__ import annotations

import math
import struct

import numpy as np
import torch

import slimtracin_amd as st
from slimtracin_amd.scene import (BRDF_BLINN, BRDF_COOK_TORRANCE, HIT_DTYPE, MODE_BEAUTY, MODE_DEPTH, MODE_NORMALS,
                                  MODE_UVS, PIXEL_DTYPE, PRIM_BOX, PRIM_DTYPE, PRIM_MESH, PRIM_QUAD, PRIM_SPHERE,
                                  PRIM_TETRAHEDRON, Light, Material, Primitive, Scene, blob_prims, make_view)
from slimtracin_amd.server import OUTPUT_BGRA8, Server

MODES = {"beauty": MODE_BEAUTY, "depth": MODE_DEPTH, "normals": MODE_NORMALS, "uvs": MODE_UVS}
BUILDERS = {"sah": {}, "lbvh": {"mesh_lbvh": True}, "binned": {"mesh_binned": True}}
CONE = 0.001                    # ray-cone angle of requests on textured scenes
TEXTURE = 256


# ---- the cases ---------------------------------------------------------------

def listed():
    return [
        # one mouse press over a scene with a 200k-triangle mesh: nothing but latency
        dict(name="pick_press", kind="pick", scene="pbr", k=100, builder="lbvh", points=1),
        # a thumbnail in a program that may not allocate; the smallest frame, launches and copies only
        dict(name="thumb_noalloc", kind="frame", api="noalloc", scene="implicit", k=0, builder="sah", mode="depth",
             depth=2, width=128, height=96, hits=True),
        # the 640x480 frame of implicit primitives, FloatPixels brought to the host as the reference does
        dict(name="implicit_640x480", kind="frame", api="render", scene="implicit", k=0, builder="sah", mode="beauty",
             depth=2, width=640, height=480, hits=False),
        # a normals pass with hit records at an odd size, for a program that shades by itself
        dict(name="normals_hits_1283x719", kind="frame", api="render", scene="pbr", k=100, builder="lbvh",
             mode="normals", depth=1, width=1283, height=719, hits=True),
        # the default builder's mesh (leaves of up to four), depth 3, at an odd size
        dict(name="pbr_sah_799x601", kind="frame", api="render", scene="pbr", k=32, builder="sah", mode="beauty",
             depth=3, width=799, height=601, hits=False),
        # the full-HD frame of the 200k-triangle scene, depth 4, as a window image
        dict(name="pbr_1920x1080", kind="frame", api="bgra8", scene="pbr", k=100, builder="binned", mode="beauty",
             depth=4, width=1920, height=1080, hits=False),
        # an animation frame: 64 textured instances moved, tree rebuilt, 1280x720, depth 3
        dict(name="moving_1280x720", kind="moving", instances=64, triangles=50000, builder="binned", depth=3,
             width=1280, height=720),
        # a crowd of 20,000 primitives moved, its tree rebuilt on the device and read back
        dict(name="rebuild_20000", kind="rebuild", prims=20000),
        # a strip of previews: 24 small mixed requests in one launch
        dict(name="batch_24_previews", kind="batch", scenes=3, k=60, requests=24, min_side=64, max_side=257),
        # the mixed batch: 160 requests from 128x128 to 1920x1080, all modes, depths 1 to 6, in one launch
        dict(name="batch_160_mixed", kind="batch", scenes=4, k=120, requests=160, min_side=128, max_side=1920),
        # a burst of 48 requests at a server with four scenes built on the device
        dict(name="served_48", kind="served", scenes=4, k=150, requests=48, min_side=96, max_side=1280),
        # a scene of a million triangles admitted: parsed, copied, built on the device, previewed, released
        dict(name="admit_1m", kind="admit", k=224, builder="lbvh", width=320, height=200),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pick", "frame", "frame", "frame", "moving", "rebuild", "batch", "served", "admit"])
    if kind == "pick":
        return dict(kind=kind, scene="pbr", k=_log(rng, 5, 150), builder=rng.choice(["lbvh", "binned"]),
                    points=_log(rng, 1, 4096))
    if kind == "frame":
        scene = rng.choice(["implicit", "pbr", "pbr", "instanced"])
        builder = rng.choice(["lbvh", "binned", "sah"])
        k = _log(rng, 3, 30 if builder == "sah" else 160)
        api = rng.choice(["render", "noalloc", "graph", "bgra8"])
        most = 560 if api == "noalloc" else 1920
        return dict(kind=kind, api=api, scene=scene, k=0 if scene == "implicit" else k, builder=builder,
                    mode=rng.choice(["beauty", "beauty", "depth", "normals", "uvs"]), depth=rng.randint(1, 6),
                    width=_log(rng, 33, most), height=_log(rng, 33, most * 9 // 16),
                    hits=api in ("render", "noalloc") and rng.random() < 0.5)
    if kind == "moving":
        return dict(kind=kind, instances=_log(rng, 4, 100), triangles=_log(rng, 500, 60000),
                    builder=rng.choice(["lbvh", "binned"]), depth=rng.randint(1, 4), width=_log(rng, 120, 1920),
                    height=_log(rng, 80, 1080))
    if kind == "rebuild":
        return dict(kind=kind, prims=_log(rng, 3, 20000))
    if kind == "batch":
        return dict(kind=kind, scenes=rng.randint(1, 4), k=_log(rng, 10, 120), requests=_log(rng, 2, 120),
                    min_side=64, max_side=_log(rng, 130, 1600))
    if kind == "served":
        return dict(kind=kind, scenes=rng.randint(1, 4), k=_log(rng, 10, 150), requests=_log(rng, 1, 48),
                    min_side=64, max_side=_log(rng, 130, 1280))
    return dict(kind=kind, k=_log(rng, 10, 224), builder=rng.choice(["lbvh", "binned"]), width=_log(rng, 64, 640),
                height=_log(rng, 48, 400))


# ---- what a program has in hand ------------------------------------------------

def _scene_blob(case, seed):
    if case["scene"] == "implicit":
        return st.gen_implicit(seed)
    if case["scene"] == "pbr":
        return st.gen_pbr(seed, case["k"])
    return st.gen_instanced(seed, 24, _three(20 * case["k"] ** 2 // 4), TEXTURE)


def _three(triangles):
    """Triangle counts of an instanced scene's three meshes, the largest about `triangles`."""
    return [max(20, triangles // 10), max(20, triangles // 3), max(20, triangles)]


def _orbit(rng, width, height, mode, depth, cone=0.0, dist=14.0, target_y=1.5):
    """A camera on a sphere around the scene that looks at its centre."""
    azim = float(rng.uniform(-np.pi / 2, np.pi / 2))
    elev = float(np.radians(rng.uniform(8.0, 50.0)))
    pos = (float(dist * np.cos(elev) * np.sin(azim)), float(target_y + dist * np.sin(elev)),
           float(-dist * np.cos(elev) * np.cos(azim)))
    return make_view(width=width, height=height, mode=mode, depth=depth, cone_angle=cone, position=pos,
                     yaw=float(np.tan(azim / 2)), pitch=float(np.tan(-elev / 2)))


def _mix(rng, case, scene_count, textured):
    """Requests with sides log-uniform in the case's range (the same sizes for every seed), the rest from rng."""
    views, ids = [], []
    sizes = np.random.default_rng(7)
    for _ in range(case["requests"]):
        side = [int(round(np.exp(sizes.uniform(np.log(case["min_side"]), np.log(m)))))
                for m in (case["max_side"], max(case["min_side"] + 1, case["max_side"] * 9 // 16))]
        s = int(rng.integers(0, scene_count))
        views.append(_orbit(rng, side[0], side[1],
                            int(rng.choice([MODE_BEAUTY, MODE_DEPTH, MODE_NORMALS, MODE_UVS])),
                            int(rng.integers(1, 7)), CONE if textured(s) else 0.0))
        ids.append(s)
    return np.concatenate(views), ids


def _several(case, seed):
    """Blobs of a batch's or server's scenes: icospheres, every second one a textured instanced scene."""
    return [st.gen_pbr(seed + i, max(2, case["k"] - 7 * i)) if i % 2 == 0 else
            st.gen_instanced(seed + i, 32, _three(20 * case["k"] ** 2 // 4), TEXTURE) for i in range(case["scenes"])]


def _windows(views):
    """A page-locked block and its slices, one BGRA8 window image for each view."""
    sizes = [int(v["width"]) * int(v["height"]) for v in views]
    block = st.pinned_empty(sum(sizes), np.uint32)
    at = np.concatenate([[0], np.cumsum(sizes)])
    return block, [block[at[i]:at[i + 1]] for i in range(len(sizes))]


def _moved(rng, prims):
    """The instances somewhere else with another rotation; the last primitive is the floor."""
    p = prims.copy()
    n = len(p) - 1
    p["position"][:n] = rng.uniform((-12, 1.5, -8), (12, 6, 16), (n, 3)).astype(np.float32)
    q = rng.normal(size=(n, 4))
    p["rotation"][:n] = (q / np.linalg.norm(q, axis=1, keepdims=True)).astype(np.float32)
    return p


def _crowd(rng, n):
    """n boxes, spheres, quads and tetrahedra of different sizes, strewn as a level's props are."""
    s = Scene(ambient=(0.01, 0.01, 0.01))
    s.lights = [Light((10, 10, -5), (1.0, 1.0, 0.65), 44.0)]
    s.materials = [Material(brdf=BRDF_BLINN, roughness=0.5), Material(brdf=BRDF_COOK_TORRANCE, roughness=0.3)]
    s.primitives = [Primitive(PRIM_BOX)]
    p = np.repeat(blob_prims(s.to_blob()), n)
    p["type"] = rng.choice([PRIM_BOX, PRIM_SPHERE, PRIM_QUAD, PRIM_TETRAHEDRON], n)
    p["material_id"] = rng.integers(0, 2, n)
    _strew(rng, p)
    blob = bytearray(s.to_blob())
    head, one = blob[:56], PRIM_DTYPE.itemsize
    struct.pack_into("<I", head, 8, n)
    return bytes(head) + p.tobytes() + bytes(blob[56 + one:]), p


def _strew(rng, p):
    n = len(p)
    p["position"] = rng.normal(0, (40, 4, 40), (n, 3)).astype(np.float32)
    q = rng.normal(size=(n, 4))
    p["rotation"] = (q / np.linalg.norm(q, axis=1, keepdims=True)).astype(np.float32)
    p["scale"] = np.exp(rng.uniform(np.log(0.05), np.log(2.0), (n, 1))).astype(np.float32)


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "pick":
        s["scene"] = st.DeviceScene(_scene_blob(case, seed), **BUILDERS[case["builder"]])
        s["view"] = _orbit(rng, 1280, 720, MODE_BEAUTY, 2)
        s["xy"] = _points(rng, case)
    elif kind == "frame":
        s["scene"] = st.DeviceScene(_scene_blob(case, seed), **BUILDERS[case["builder"]])
        s["view"] = _frame_view(rng, case)
        n = (case["width"] + 1) * (case["height"] + 1)
        if case["api"] == "bgra8":
            s["block"], s["outs"] = _windows(s["view"])
        else:
            s["out"] = st.pinned_empty(n, PIXEL_DTYPE)
    elif kind == "moving":
        blob = st.gen_instanced(seed, case["instances"], _three(case["triangles"]), TEXTURE)
        s["scene"] = st.DeviceScene(blob, **BUILDERS[case["builder"]])
        s["prims"] = np.ascontiguousarray(_moved(rng, blob_prims(blob)), dtype=PRIM_DTYPE)
        s["view"] = make_view(width=case["width"], height=case["height"], mode=MODE_BEAUTY, depth=case["depth"],
                              cone_angle=CONE, position=(float(rng.uniform(-2, 2)), 9.0, -22.0), pitch=-0.2)
        s["block"], s["outs"] = _windows(s["view"])
    elif kind == "rebuild":
        blob, p = _crowd(rng, case["prims"])
        s["scene"] = st.DeviceScene(blob)
        _strew(rng, p)
        s["prims"] = np.ascontiguousarray(p, dtype=PRIM_DTYPE)
    elif kind == "batch":
        s["scenes"] = [st.DeviceScene(b, **BUILDERS["binned"]) for b in _several(case, seed)]
        s["views"], ids = _mix(rng, case, case["scenes"], lambda i: i % 2 == 1)
        s["which"] = [s["scenes"][i] for i in ids]
        s["block"], s["outs"] = _windows(s["views"])
    elif kind == "served":
        s["server"] = Server(output=OUTPUT_BGRA8)
        s["ids"] = [s["server"].add_scene(b, mesh_lbvh=True) for b in _several(case, seed)]
        s["views"], which = _mix(rng, case, case["scenes"], lambda i: i % 2 == 1)
        s["which"] = [s["ids"][i] for i in which]
    else:
        s["blob"] = st.gen_pbr(seed, case["k"])
        s["view"] = _orbit(rng, case["width"], case["height"], MODE_BEAUTY, 2)
        s["block"], s["outs"] = _windows(s["view"])
    return s


def _points(rng, case):
    """Window points as a user presses them: around the middle, where the objects are."""
    x = np.clip(rng.normal(640, 200, case["points"]), 0, 1279)
    y = np.clip(rng.normal(360, 120, case["points"]), 0, 719)
    return np.stack([x, y], 1).astype(np.uint32)


def _frame_view(rng, case):
    if case["scene"] == "implicit":
        return make_view(width=case["width"], height=case["height"], mode=MODES[case["mode"]], depth=case["depth"],
                         position=(float(rng.uniform(-1, 1)), 7.0, -11.0), pitch=-0.2)
    return _orbit(rng, case["width"], case["height"], MODES[case["mode"]], case["depth"],
                  CONE if case["scene"] == "instanced" else 0.0)


# ---- one pass --------------------------------------------------------------------

def _pixels(p):
    """FloatPixel records as an array of r, g, b, opacity and one of depths (views)."""
    return {"rgba": p.view(np.float32).reshape(len(p), 6)[:, :4], "z": p["depth"]}


def _hits(h):
    return {"ids": h.view(np.int32).reshape(len(h), 4)[:, :3], "t": h["distance"]}


def _counts(counts):
    return [int(v) for c in counts for v in (c.primary, c.shadow, c.bounce)]


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "pick":
        p = st.pick(s["scene"], s["view"], s["xy"])
        return {"type": p["object_type"], "id": p["object_id"].astype(np.int64), "position": p["position"],
                "z": p["object_distance"]}
    if kind == "frame":
        if case["api"] == "bgra8":
            _, counts = st.render_batch_bgra8([s["scene"]], s["view"], outs=s["outs"])
            return [s["block"].view(np.uint8), np.array(_counts(counts))]
        if case["api"] == "graph":
            _, _, counts = st.render_batch([s["scene"]], s["view"], outs=[s["out"]], graph=True)
            return {"pixels": _pixels(s["out"]), "rays": np.array(_counts(counts))}
        call = st.render_noalloc if case["api"] == "noalloc" else st.render
        _, hits, counts = call(s["scene"], s["view"], hits=case["hits"], out=s["out"])
        got = {"pixels": _pixels(s["out"]), "rays": np.array(_counts([counts]))}
        if hits is not None:
            got["hits"] = _hits(hits)
        return got
    if kind == "moving":
        s["scene"].set_prims(s["prims"])
        s["scene"].rebuild(st.ST_REBUILD_LBVH)
        _, counts = st.render_batch_bgra8([s["scene"]], s["view"], outs=s["outs"])
        return [s["block"].view(np.uint8), np.array(_counts(counts))]
    if kind == "rebuild":
        s["scene"].set_prims(s["prims"])
        s["scene"].rebuild(st.ST_REBUILD_LBVH)
        nodes, leaf, height = s["scene"].bvh()
        words = nodes.view(np.int32).reshape(len(nodes), 8)
        return {"boxes": words[:, :6], "links": words[:, 6:], "leaf": leaf.astype(np.int64), "height": int(height)}
    if kind == "batch":
        _, counts = st.render_batch_bgra8(s["which"], s["views"], outs=s["outs"])
        return [s["block"].view(np.uint8), np.array(_counts(counts))]
    if kind == "served":
        srv = s["server"]
        tickets = [srv.submit(sid, s["views"][i:i + 1]) for i, sid in enumerate(s["which"])]
        images, counts = [], []
        for t in tickets:
            image, c, _ = srv.wait(t)
            srv.release(t)
            images.append(image.view(np.uint8))
            counts.append(c)
        return images + [np.array(_counts(counts))]
    scene = st.DeviceScene(s["blob"], **BUILDERS[case["builder"]])
    info = scene.info()
    _, counts = st.render_batch_bgra8([scene], s["view"], outs=s["outs"])
    scene.close()
    return [s["block"].view(np.uint8), np.array(_counts(counts) + [info.triangle_count, info.mesh_node_count])]


# ---- what a pass cannot do without -------------------------------------------------

def _tree_bytes(triangles):
    """Two 32-byte nodes and a 64-byte record for each triangle."""
    return 128.0 * triangles


def _ray_flops(triangles):
    """One ray's way down a tree: two boxes of about 20 operations on each level, and a triangle."""
    return 40.0 * max(1.0, math.log2(max(2, triangles))) + 60.0


def _frames_work(pixels, triangles, bytes_per_pixel, mode_beauty):
    rays = pixels * (3.0 if mode_beauty else 1.0)
    # a frame reads at most as many nodes and records as its rays' ways hold, and the tree once at most
    read = min(_tree_bytes(triangles), rays * (64.0 * math.log2(max(2, triangles)) + 64.0))
    return {"bytes": read + pixels * bytes_per_pixel,
            "flops": rays * (_ray_flops(triangles) + (300.0 if mode_beauty else 50.0))}


def work(case):
    kind = case["kind"]
    if kind == "pick":
        n = case["points"]
        t = 20 * case["k"] ** 2
        return {"bytes": 32.0 * n + min(_tree_bytes(t), 64.0 * n * math.log2(max(2, t))), "flops": n * _ray_flops(t)}
    if kind == "frame":
        t = 16 if case["scene"] == "implicit" else 20 * case["k"] ** 2
        n = (case["width"] + 1) * (case["height"] + 1)
        return _frames_work(n, t, 4.0 if case["api"] == "bgra8" else 24.0 + (16.0 if case["hits"] else 0.0),
                            case["mode"] == "beauty")
    if kind == "moving":
        n = (case["width"] + 1) * (case["height"] + 1)
        return _frames_work(n, case["instances"] * case["triangles"] // 2, 4.0, True)
    if kind == "rebuild":
        n = case["prims"]
        return {"bytes": n * (56.0 + 64.0 + 4.0), "flops": n * (200.0 + 30.0 * math.log2(max(2, n)))}
    if kind in ("batch", "served"):
        lo, hi = math.log(case["min_side"]), math.log(case["max_side"])
        hj = math.log(max(case["min_side"] + 1, case["max_side"] * 9 // 16))
        mean = [(math.exp(b) - math.exp(lo)) / max(1e-9, b - lo) for b in (hi, hj)]
        n = case["requests"] * mean[0] * mean[1]
        t = 20 * case["k"] ** 2
        w = _frames_work(n, t, 4.0, False)
        return {"bytes": w["bytes"] + (case["scenes"] - 1) * min(_tree_bytes(t), w["bytes"]), "flops": 1.5 * w["flops"]}
    t = 20 * case["k"] ** 2
    w = _frames_work((case["width"] + 1) * (case["height"] + 1), t, 4.0, True)
    # vertices, indices and their normals read once; tree and records written once
    return {"bytes": w["bytes"] + t * (52.0 + 64.0 + 144.0), "flops": w["flops"] + t * 400.0}


def tolerance(case):
    """Hits, geometry and trees are decided in the reference's fp32 operations and are the same in every correct
    implementation. Radiance goes through powf and acosf, which differ in their last places between math libraries: the
    CPU oracle's frames of these scenes differ from the GPU's by up to 8e-8 (2-norm), in a channel by up to 8e-7, and
    one byte in a million of the window images, the floors of square roots, is another where that crosses a whole
    value."""
    kind = case["kind"]
    if kind in ("pick", "rebuild") or (kind == "frame" and case["mode"] != "beauty"):
        return "exact"
    if kind == "frame" and case["api"] != "bgra8":
        return {"rel": 4e-7, "max": 4e-6, "differ": 0.0}
    return {"differ": 4e-6}


# ---- the same in 64 bits --------------------------------------------------------------

def exact(case, seed):
    """Picks, and depth frames of the implicit scenes: rays, intersections and transforms in 64 bits, every primitive
    and triangle tried. None otherwise: window images are whole numbers, a mesh frame by brute force takes minutes, and
    beauty follows bounce rays whose 64-bit hits are other surfaces' at every edge."""
    rng = np.random.default_rng(seed)
    if case["kind"] == "pick":
        blob = _scene_blob(case, seed)
        view = _orbit(rng, 1280, 720, MODE_BEAUTY, 2)
        xy = _points(rng, case)
        if case["points"] * 20 * case["k"] ** 2 > 4e8:
            return None
        cam, d, forward = _rays(view, xy[:, 0].astype(np.float64), xy[:, 1].astype(np.float64))
        t = _closest(blob, cam, d, view, xy[:, 0], xy[:, 1])
        t = np.minimum(t, _glow(blob, cam, d))
        pos = np.where(np.isfinite(t)[:, None], cam + d * np.where(np.isfinite(t), t, 0)[:, None], 0.0)
        z = np.where(np.isfinite(t), (pos - cam) @ forward, 0.0)
        return {"type": None, "id": None, "position": pos, "z": z}
    if case["kind"] == "frame" and case["scene"] == "implicit" and case["mode"] == "depth" and \
            case["api"] != "bgra8":
        view = _frame_view(rng, case)
        w, h = case["width"] + 1, case["height"] + 1
        y, x = np.divmod(np.arange(w * h), w)
        cam, d, forward = _rays(view, x.astype(np.float64), y.astype(np.float64))
        t = _closest(_scene_blob(case, seed), cam, d, view, x, y)
        hit = np.isfinite(t)
        shade = np.where(hit, (255.0 * 4.0 / np.where(hit, t, 1.0)) ** 2, 0.0)
        rgba = np.stack([shade, shade, shade, hit.astype(np.float64)], 1)
        got = {"pixels": {"rgba": rgba, "z": np.where(hit, t * (d @ forward), np.inf)}, "rays": None}
        if case["hits"]:
            got["hits"] = {"ids": None, "t": t}
        return got
    return None


def _rays(view, x, y):
    """Camera position, unit directions of window points and the camera's forward direction."""
    v = view[0]
    right, up, forward = _axes(v)
    w, h = int(v["width"]) + 1.0, int(v["height"]) + 1.0
    start = forward * h * float(v["focal_length"]) - right * w + up * h
    d = start + 2 * np.outer(x, right) - 2 * np.outer(y, up)
    return v["position"].astype(np.float64), d / np.linalg.norm(d, axis=1, keepdims=True), forward


def _axes(v):
    """The camera's right, up and forward directions."""
    def turn(amount):
        a = float(amount)
        return (1 - a * a) / (1 + a * a), 2 * a / (1 + a * a)

    (cy, sy), (cp, sp) = turn(v["yaw"]), turn(v["pitch"])
    yaw = np.array([[cy, 0, sy], [0, 1, 0], [-sy, 0, cy]])
    pitch = np.array([[1, 0, 0], [0, cp, -sp], [0, sp, cp]])
    return pitch @ yaw


def _inside(v, centre, radius, x, y):
    """The window points inside a bounding sphere's rectangle on the screen, in whole pixels cut off as the renderer
    cuts them: it tries a primitive at those points only."""
    w, h = int(v["width"]) + 1.0, int(v["height"]) + 1.0
    a, b, z = _axes(v) @ (centre - v["position"].astype(np.float64))
    if z <= -radius:
        return np.zeros(len(x), bool)
    if z <= radius:
        return np.ones(len(x), bool)
    den = z * z - radius * radius
    f = float(v["focal_length"]) / den
    sides = []
    for at, factor, half, turned in ((a, f * h / w, w / 2, 1), (b, f, h / 2, -1)):
        root = radius * math.sqrt(at * at + den)
        lo, hi = sorted(turned * factor * (at * z + s * root) for s in (-1, 1))
        if lo >= 1 or hi <= -1:
            return np.zeros(len(x), bool)
        sides += [int(half * (max(lo, -1) + 1)), int(half * (min(hi, 1) + 1))]
    return (x >= sides[0]) & (x < sides[1]) & (y >= sides[2]) & (y < sides[3])


def _bound(p, blob, counts):
    """Radius of the sphere that bounds a primitive on the screen."""
    s = p["scale"].astype(np.float64)
    if p["type"] == PRIM_MESH:
        faces = _mesh_faces(blob, counts, int(p["mesh_id"])).numpy().reshape(-1, 3)
        return max(np.linalg.norm(s * faces.min(0)), np.linalg.norm(s * faces.max(0)))
    return {PRIM_SPHERE: s.max(), PRIM_TETRAHEDRON: math.sqrt(2.0) * s.max()}.get(int(p["type"]), np.linalg.norm(s))


def _turned(v, q):
    a, w = q[:3], q[3]
    c = np.cross(a, v)
    return v + 2 * (w * c + np.cross(a, c))


def _closest(blob, cam, d, view, x, y):
    """Distance along each window point's ray to the nearest surface (inf: none)."""
    counts = struct.unpack_from("<7I", blob, 0)
    prims = np.frombuffer(blob, dtype=PRIM_DTYPE, count=counts[2], offset=56)
    best = np.full(len(d), np.inf)
    for p in prims:
        q = p["rotation"].astype(np.float64) * np.array([-1, -1, -1, 1])
        o = _turned(cam - p["position"].astype(np.float64), q) / p["scale"].astype(np.float64)
        r = _turned(d, q) / p["scale"].astype(np.float64)
        with np.errstate(all="ignore"):
            if p["type"] == PRIM_QUAD:
                t = -o[1] / r[:, 1]
                at = o + r * t[:, None]
                t = np.where((np.abs(at[:, 0]) <= 1) & (np.abs(at[:, 2]) <= 1), t, np.inf)
            elif p["type"] == PRIM_BOX:
                a, b = (-1 - o) / r, (1 - o) / r
                near, far = np.minimum(a, b).max(1), np.maximum(a, b).min(1)
                t = np.where(far >= np.maximum(near, 0), np.where(near > 0, near, far), np.inf)
            elif p["type"] == PRIM_SPHERE:
                rr, b = (r * r).sum(1), r @ o
                disc = b * b - rr * (o @ o - 1)
                root = np.sqrt(np.maximum(disc, 0))
                t = np.where((-b - root) > 0, (-b - root) / rr, (-b + root) / rr)
                t = np.where((disc > 0) & (b < 0), t, np.inf)
            elif p["type"] == PRIM_TETRAHEDRON:
                corners = np.array([[-1, -1, -1], [-1, 1, 1], [1, -1, 1], [1, 1, -1]]) / math.sqrt(3.0)
                t = _triangles(torch.from_numpy(corners[[[1, 2, 3], [0, 2, 3], [0, 1, 3], [0, 1, 2]]]), o, r)
            elif p["type"] == PRIM_MESH:
                t = _triangles(_mesh_faces(blob, counts, int(p["mesh_id"])), o, r)
            else:
                continue
        seen = _inside(view[0], p["position"].astype(np.float64), _bound(p, blob, counts), x, y)
        best = np.minimum(best, np.where((t > 0) & seen, t, np.inf))
    return best


def _mesh_faces(blob, counts, mesh):
    """Corner positions (triangles, 3, 3) of a mesh of the blob."""
    at = 56 + 56 * counts[2] + 84 * counts[3] + 28 * counts[4]
    for m in range(mesh + 1):
        v, t, n, u = struct.unpack_from("<4I", blob, at)
        pos = np.frombuffer(blob, np.float32, 3 * v, at + 56).reshape(v, 3)
        idx = np.frombuffer(blob, np.uint32, 3 * t, at + 56 + 12 * v).reshape(t, 3)
        at += 56 + 12 * v + 12 * t + (12 * n + 12 * t if n else 0) + (8 * u + 12 * t if u else 0)
    return torch.from_numpy(pos[idx].astype(np.float64))


def _triangles(faces, o, r):
    """Nearest hit of rays o + t r with triangles (either side), every ray against every triangle."""
    dev = "cuda" if torch.cuda.is_available() and len(faces) > 1000 else "cpu"
    faces, r = faces.to(dev), torch.from_numpy(np.ascontiguousarray(r)).to(dev)
    o = torch.from_numpy(np.ascontiguousarray(o)).to(dev)
    a, e1, e2 = faces[:, 0], faces[:, 1] - faces[:, 0], faces[:, 2] - faces[:, 0]
    n = torch.linalg.cross(e1, e2)
    s = o - a
    q = torch.linalg.cross(s, e1)
    sn = (s * n).sum(1)
    best = torch.full((len(r),), math.inf, dtype=torch.float64, device=dev)
    step = max(1, int(2e7) // max(1, len(r)))
    for i in range(0, len(faces), step):
        k = slice(i, i + step)
        det = -(r @ n[k].T)
        u = (r @ torch.linalg.cross(e2[k], s[k]).T) / det
        v = (r @ q[k].T) / det
        t = sn[k] / det
        ok = (det != 0) & (u >= 0) & (v >= 0) & (u + v <= 1) & (t > 0)
        best = torch.minimum(best, torch.where(ok, t, math.inf).min(1).values)
    return best.cpu().numpy()


def _glow(blob, cam, d):
    """Distance to the nearest light's glow sphere, of a 128th of its intensity."""
    counts = struct.unpack_from("<7I", blob, 0)
    best = np.full(len(d), np.inf)
    for i in range(counts[4]):
        l = struct.unpack_from("<7f", blob, 56 + 56 * counts[2] + 84 * counts[3] + 28 * i)
        c, radius = np.array(l[:3], np.float64) - cam, l[6] / 128.0
        b = d @ c
        disc = b * b - (c @ c - radius * radius)
        root = np.sqrt(np.maximum(disc, 0))
        best = np.minimum(best, np.where((disc >= 0) & (b + root > 0), b - root, np.inf))
    return best
