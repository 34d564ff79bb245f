"""Timed cases of the framework: what a program that renders volumes has it do.

A program loads a grid or an octree, converts a grid to an octree, and renders
frames: one at a time (the headless renderer), many in one launch (the batched
form), from a tight loop that may not allocate (the static form), or as
requests to a server.  Every case is one such use, through the package's public
entry points, on seeded volumes of the kinds that the benchmark and the tests
use: shells (thin coloured shells and noise), ct (a body with a soft interior
in a ragged box) and gas (a log-normal field).

The outputs are 8-bit frames, node words and counts.  They are fully specified
(the shaders' FP32 operations in order, and the converter's integers), so they
are whole numbers that have to stay equal, and there is no 64-bit value to
measure them against.
"""
import itertools
import math

import numpy as np
import torch

from xenodon_amd import abi, synth, workloads

SHADERS = ("dda", "svo-naive", "esvo", "svo-df", "svo-rope")
ALL = ",".join(SHADERS)
OCTREE = ",".join(SHADERS[1:])
EMISSION = {"shells": 4.0, "ct": 1.6, "gas": 1.0}  # at most about 1 % of the pixels saturate
TREES = {"sparse": abi.TREE_SPARSE, "dag": abi.TREE_DAG, "rope": abi.TREE_ROPE}


def listed():
    return [
        # a thumbnail or an interactive step on a small volume: the latency of one launch
        {"name": "plain-dda-256", "form": "plain", "volume": "shells", "x": 128, "y": 128, "z": 128, "w": 256, "h": 256,
         "shaders": "dda", "frames": 1, "save": False},
        # one small odd-sized frame by each octree shader, kept: render and download, the headless renderer's loop
        {"name": "plain-octrees-small", "form": "plain", "volume": "shells", "x": 128, "y": 128, "z": 128, "w": 199,
         "h": 143, "shaders": OCTREE, "frames": 1, "save": True},
        # the benchmark's own step: frames of the camera path at 1080p by all five shaders, one launch each
        {"name": "plain-path-1080p", "form": "plain", "volume": "ct", "x": 512, "y": 361, "z": 512, "w": 1920,
         "h": 1080, "shaders": ALL, "frames": 3, "save": False},
        # the largest image: a 4K frame of a large grid, saved
        {"name": "plain-dda-2160p", "form": "plain", "volume": "gas", "x": 512, "y": 512, "z": 512, "w": 3840,
         "h": 2160, "shaders": "dda", "frames": 1, "save": True},
        # the benchmark's batched step: new camera frames x five shaders into one launch
        {"name": "batch-path-1080p", "form": "batch", "volume": "ct", "x": 256, "y": 181, "z": 256, "w": 1920,
         "h": 1080, "shaders": ALL, "frames": 8, "save": False},
        # many views of several sizes over two volumes in one launch
        {"name": "batch-mixed-views", "form": "mixed", "volume": "ct", "x": 256, "y": 181, "z": 256, "views": 24},
        # the allocation-free form in a tight loop: a few small views at a time
        {"name": "static-small-views", "form": "static", "volume": "shells", "x": 128, "y": 128, "z": 128, "w": 160,
         "h": 120, "shaders": "dda,esvo,svo-rope", "frames": 4, "save": False},
        # a burst of requests to a server, from submission to frames in host memory
        {"name": "served-burst", "form": "serve", "volume": "ct", "x": 256, "y": 181, "z": 256, "requests": 32},
        # start-up on a grid: upload from host memory, first frame, release
        {"name": "load-grid", "form": "load", "volume": "ct", "x": 384, "y": 271, "z": 353, "w": 640, "h": 360,
         "shaders": "dda", "tree": "none"},
        # start-up on an octree file's nodes: upload, first frame, release
        {"name": "load-octree", "form": "load", "volume": "ct", "x": 192, "y": 137, "z": 192, "w": 640, "h": 360,
         "shaders": "svo-rope", "tree": "rope"},
        # lossless conversion of a resident grid to a rope octree, in host memory
        {"name": "convert-rope", "form": "convert", "volume": "ct", "x": 300, "y": 217, "z": 283, "tree": "rope",
         "chan_diff": 0, "std_dev": -1.0},
        # lossy conversion to a DAG under the standard-deviation heuristic
        {"name": "convert-dag-stddev", "form": "convert", "volume": "shells", "x": 128, "y": 128, "z": 128,
         "tree": "dag", "chan_diff": 0, "std_dev": 6.0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_volume(rng, lo, hi):
    kind = rng.choice(("shells", "ct", "gas"))
    if kind == "gas":
        n = _log_int(rng, lo, hi)
        return {"volume": kind, "x": n, "y": n, "z": n}
    return {"volume": kind, "x": _log_int(rng, lo, hi), "y": _log_int(rng, lo, hi), "z": _log_int(rng, lo, hi)}


def draw(rng):
    form = rng.choice(("plain", "plain", "plain", "batch", "mixed", "static", "serve", "load", "load", "convert",
                       "convert"))
    if form in ("plain", "batch", "static"):
        w, h = _log_int(rng, 96, 1920), _log_int(rng, 96, 1080)
        shaders = rng.sample(SHADERS, rng.choice((1, 1, 2, 5)))
        case = {"form": form, **_draw_volume(rng, 48, 288), "w": w, "h": h,
                "shaders": ",".join(s for s in SHADERS if s in shaders)}
        case["frames"] = 1 if form == "plain" else rng.randint(1, max(1, min(40 // len(shaders), 20000000 // (w * h))))
        return {**case, "save": form == "plain" and rng.random() < 0.5}
    if form == "mixed":
        return {"form": form, **_draw_volume(rng, 48, 256), "views": rng.randint(4, 32)}
    if form == "serve":
        return {"form": form, **_draw_volume(rng, 48, 256), "requests": _log_int(rng, 2, 48)}
    if form == "load":
        tree = rng.choice(("none", "sparse", "rope", "rope", "dag"))
        return {"form": form, **_draw_volume(rng, 24, 320 if tree == "none" else 192), "w": _log_int(rng, 96, 1280),
                "h": _log_int(rng, 96, 720),
                "shaders": "dda" if tree == "none" else "svo-rope" if tree == "rope" else rng.choice(SHADERS[1:4]),
                "tree": tree}
    sd = rng.random() < 0.3
    return {"form": "convert", **_draw_volume(rng, 24, 256 if not sd else 128), "tree": rng.choice(tuple(TREES)),
            "chan_diff": 0 if sd else rng.choice((0, 0, 2, 9, 40)),
            "std_dev": rng.uniform(0.5, 20.0) if sd else -1.0}


# ---- inputs -----------------------------------------------------------------
#
# Another seed is another volume and other cameras.  Image sizes, and the shape
# of a grid to convert (whose node count is the output's size), are the case's:
# there a seed deals the four channels anew, which changes every node's colour
# but not the tree.

CHANNELS = list(itertools.permutations(range(4)))


def _grid(case, seed):
    dims = (case["x"], case["y"], case["z"])
    if case["form"] == "convert":
        fixed = _grid({**case, "form": "load"}, dims[0])
        return np.ascontiguousarray(fixed[..., CHANNELS[seed % len(CHANNELS)]])
    if case["volume"] == "ct":
        return synth.ct_body(dims, seed=seed + 1)
    if case["volume"] == "gas":
        return synth.lognormal(dims[0], seed=seed + 1, base=64)
    m = min(dims)
    return synth.shells(dims, seed=seed + 1, radii=(max(2.0, m / 16), max(3.0, m / 3.2)))


def _path_camera(u, azimuth):
    """Camera at u in [0, 1) of a path like the benchmark's: an orbit at distance 2, a zoom over the pole, and a
    walk along the inside of the volume's faces."""
    if u < 0.4:
        d, elev, az = 2.0, 0.0, azimuth + 2.5 * math.pi * u
    elif u < 0.7:
        v = (u - 0.4) / 0.3
        d, elev, az = 2.0 - 1.5 * v, 1.4 * math.sin(math.pi * v), azimuth + math.pi
    else:
        d, elev, az = 0.5, 0.0, azimuth + 2 * math.pi * (u - 0.7) / 0.3
    eye = 0.5 + d * np.array([math.sin(az) * math.cos(elev), math.sin(elev), -math.cos(az) * math.cos(elev)])
    return workloads.look_at(eye, (0.5, 0.5, 0.5))


class _Pixels:
    """A frame's device memory as an array that torch can wrap."""

    def __init__(self, frame):
        self.frame = frame
        self.__cuda_array_interface__ = {"shape": (frame.height, frame.width, 4), "typestr": "|u1", "version": 2,
                                         "data": (frame.device_ptr(), False)}


def _pixels(frame):
    return torch.as_tensor(_Pixels(frame), device="cuda")


def _dims(grid):
    return [grid.shape[2], grid.shape[1], grid.shape[0]]


def _volumes(ctx, grid, shaders):
    """The grid's volume and its rope octree, {shader: (volume, model dimensions)} for those asked."""
    gvol = ctx.grid_volume(grid)
    vols = {"dda": (gvol, _dims(grid))}
    if any(s != "dda" for s in shaders):
        nodes, st = ctx.build_octree(gvol, tree=abi.TREE_ROPE)
        svol = ctx.svo_volume(nodes, st["side"])
        vols.update({s: (svol, [st["side"]] * 3) for s in SHADERS[1:]})
    return vols


def _path_views(case, seed, ctx, vols):
    """(volume, traversal, camera, uniforms) of every frame and shader of a path case."""
    azimuth = np.random.default_rng(seed).uniform(0, 2 * math.pi)
    views = []
    for k in range(case["frames"]):
        cam = abi.make_camera(*_path_camera((k + 0.5) / case["frames"] if case["frames"] > 1 else 0.1, azimuth))
        for name in case["shaders"].split(","):
            vol, md = vols[name]
            uni = abi.make_uniforms(case["w"], case["h"], md, emission=EMISSION[case["volume"]])
            views.append((vol, abi.TRAVERSALS[name], cam, uni))
    return views


def prepare(case, seed):
    ctx = abi.Context(0)
    s = {"form": case["form"], "ctx": ctx, "case": case}
    grid = _grid(case, seed)
    emission = EMISSION[case["volume"]]
    if case["form"] in ("plain", "batch", "static"):
        views = _path_views(case, seed, ctx, _volumes(ctx, grid, case["shaders"].split(",")))
        if case["save"]:
            s["frame"], s["views"] = ctx.frame(case["w"], case["h"]), views
        else:
            s["views"] = [v + (ctx.frame(case["w"], case["h"]),) for v in views]
            s["pixels"] = [_pixels(v[4]) for v in s["views"]]
        if case["form"] == "batch":
            s["batch"] = ctx.batch()
    elif case["form"] == "mixed":
        # the case's volume and a small one, views as in the many-views batch of the benchmark
        small = synth.shells((64, 64, 64), seed=seed + 2, radii=(4.0, 20.0))
        scenes = {"a": (_volumes(ctx, grid, SHADERS), emission), "b": (_volumes(ctx, small, SHADERS), EMISSION["shells"])}
        s["views"] = []
        rng = np.random.default_rng(seed)
        for name, t, _, w, h in workloads.mixed_views(list(scenes), n=case["views"]):
            vols, e = scenes[name]
            vol, md = vols[abi.TRAVERSAL_NAMES[t]]
            cam = abi.make_camera(*workloads.orbit_camera(rng))
            s["views"].append((vol, t, cam, abi.make_uniforms(w, h, md, emission=e), ctx.frame(w, h)))
        s["pixels"] = [_pixels(v[4]) for v in s["views"]]
        s["batch"] = ctx.batch()
    elif case["form"] == "serve":
        srv = s["server"] = ctx.server()
        gvol = ctx.grid_volume(grid)
        nodes, st = ctx.build_octree(gvol, tree=abi.TREE_ROPE)
        gvol.free()
        ids = {"grid": srv.load_grid(grid), "svo": srv.load_svo(nodes, st["side"])}
        rng = np.random.default_rng(seed)
        reqs, _ = workloads.request_mix({"grid": "grid", "svo": "svo"}, case["requests"], case["requests"])
        s["requests"] = [(ids[name], t, abi.make_camera(*workloads.orbit_camera(rng)), w, h, emission)
                         for name, t, _, w, h in reqs]
    else:
        side = max(_dims(grid))
        if case["form"] == "convert":
            s["grid"] = ctx.grid_volume(grid)
        else:
            s["host"] = grid
            if case["tree"] != "none":
                gvol = ctx.grid_volume(grid)
                nodes, st = ctx.build_octree(gvol, tree=TREES[case["tree"]])
                gvol.free()
                s["host"], side = nodes, st["side"]
            s["side"] = side
            md = _dims(grid) if case["tree"] == "none" else [side] * 3
            azimuth = np.random.default_rng(seed).uniform(0, 2 * math.pi)
            s["cam"] = abi.make_camera(*_path_camera(0.1, azimuth))
            s["uni"] = abi.make_uniforms(case["w"], case["h"], md, emission=emission)
            s["frame"] = ctx.frame(case["w"], case["h"])
    return s


# ---- one pass ---------------------------------------------------------------

def run(s):
    ctx, case = s["ctx"], s["case"]
    if s["form"] == "plain":
        if case["save"]:
            out = []
            for vol, t, cam, uni in s["views"]:
                ctx.render(vol, t, cam, uni, s["frame"])
                out.append(s["frame"].download())
            return out
        for view in s["views"]:
            ctx.render(*view)
        return s["pixels"]
    if s["form"] in ("batch", "mixed"):
        s["batch"].set_views(s["views"])
        s["batch"].render()
        return s["pixels"]
    if s["form"] == "static":
        abi.render_static(ctx, s["views"])
        return s["pixels"]
    if s["form"] == "serve":
        srv = s["server"]
        order = [srv.submit(vid, t, cam, w, h, emission=e)[0] for vid, t, cam, w, h, e in s["requests"]]
        images = {}
        while len(images) < len(order):
            for done in srv.poll():
                if done["status"] != abi.XD_OK:
                    raise RuntimeError("request ended with status %d" % done["status"])
                images[done["id"]] = done["image"]
        return [images[i] for i in order]
    if s["form"] == "load":
        vol = ctx.grid_volume(s["host"]) if case["tree"] == "none" else ctx.svo_volume(s["host"], s["side"])
        ctx.render(vol, abi.TRAVERSALS[case["shaders"]], s["cam"], s["uni"], s["frame"])
        image = s["frame"].download()
        vol.free()
        return image
    sd = case["std_dev"] >= 0
    nodes, stats = ctx.build_octree(s["grid"], chan_diff=case["chan_diff"], tree=TREES[case["tree"]],
                                    heuristic=abi.HEURISTIC_STD_DEV if sd else abi.HEURISTIC_CHAN_DIFF,
                                    std_dev=max(case["std_dev"], 0.0))
    return {"nodes": nodes, "stats": stats}


def work(case):
    """Bytes: the volume's voxels or nodes once and the outputs once.  Operations: about a dozen for each voxel that a
    ray passes, some 0.7 of the box's mean side of them (rays that miss included)."""
    voxels = case["x"] * case["y"] * case["z"]
    nodes = 0.3 * voxels * 40  # octrees of these volumes hold about 0.3 nodes for a voxel
    side = (case["x"] + case["y"] + case["z"]) / 3
    if case["form"] == "convert":
        return {"bytes": 4 * voxels + nodes, "flops": 20 * voxels}
    if case["form"] == "load":
        volume, rays = (4 * voxels if case["tree"] == "none" else nodes), case["w"] * case["h"]
        return {"bytes": 2 * volume + 4 * rays, "flops": 12 * 0.7 * side * rays}
    if case["form"] == "mixed":
        rays = case["views"] * 800 * 560
    elif case["form"] == "serve":
        rays = case["requests"] * 660 * 448
    else:
        rays = case["w"] * case["h"] * case["frames"] * len(case["shaders"].split(","))
    crossed = 0.7 * side * rays
    return {"bytes": 4 * rays + min(4 * voxels, 4 * crossed), "flops": 12 * crossed}
