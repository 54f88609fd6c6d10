"""The work that users of this framework have it do, as measurable cases.

A case is a dict of plain values. `prepare` builds what a viewer, a VR client,
a tile server or a file browser holds before a frame: a device-resident cloud,
cameras, framebuffers and plans. `run` draws one frame (or opens one set of
files and draws its first frame) through the package's entry points and
returns the framebuffer keys and RGBA images, which stay on the GPU.

One context (one stream) serves every state, as in a user's program. torch is
imported before the package, so that both use the one HIP runtime.
"""
import ctypes
import math

import numpy as np
import torch

import compute_rasterizer_amd as pcr
from compute_rasterizer_amd import datasets

EXTENT = 2000.0   # side of the generated terrain and city scenes (m)

# resolutions of the multi-view and serving benchmark
VIEW_SIZES = ((256, 256), (640, 480), (1280, 720), (1920, 1080), (2560, 1440))

_context = None


def _ctx():
    global _context
    if _context is None:
        _context = pcr.Context(0)
    return _context


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # A preview window over a small scan: everything fits the caches, the
        # frame is its launches.
        dict(name="preview_200k", kind="frame", mode="las2", scene="terrain", points=200_000, width=640, height=360,
             camera="fly", height_m=100.0, edl=0.0),
        # An unsorted XYZRGBA point list as it comes from another program, one
        # pass with the colour in the key (1M-point cube, 1280x720).
        dict(name="plain16_cube_1M", kind="points16", mode="plain16", points=1_000_000, width=1280, height=720),
        # The same list with averaged colours (two passes, 1920x1080).
        dict(name="hqs16_cube_1M", kind="points16", mode="hqs16", points=1_000_000, width=1920, height=1080),
        # The reference's default method (compute_loop_las) over an airborne
        # scan: 100M terrain points, flythrough at 100 m.
        dict(name="las_terrain_100M", kind="frame", mode="las", scene="terrain", points=100_000_000, width=1920,
             height=1080, camera="fly", height_m=100.0, edl=0.0),
        # The headline frame: a 1e9-point city at 1920x1080, 100 m above the
        # ground.
        dict(name="city_fly_1e9", kind="frame", mode="las2", scene="city", points=1_000_000_000, width=1920,
             height=1080, camera="fly", height_m=100.0, edl=0.0),
        # The whole city in view, every batch drawn.
        dict(name="city_overview_1e9", kind="frame", mode="las2", scene="city", points=1_000_000_000, width=1920,
             height=1080, camera="overview", height_m=0.0, edl=0.0),
        # High-quality (averaged colour) frame of a 500M-point city on a
        # 2560x1440 screen.
        dict(name="hqs_city_500M", kind="frame", mode="hqs", scene="city", points=500_000_000, width=2560,
             height=1440, camera="fly", height_m=250.0, edl=0.0),
        # VR: both eyes of a headset from one shared-decode launch, new head
        # position each frame.
        dict(name="stereo_hqs_1e9", kind="stereo", mode="hqs", scene="city", points=1_000_000_000, width=1920,
             height=1080),
        # A tile server's batch: 48 views of uneven resolution in one launch.
        dict(name="views48_1e9", kind="views", mode="las2", scene="city", points=1_000_000_000, views=48),
        # LOD viewer: octree cut at one pixel, large screen.
        dict(name="lod_city_100M", kind="lod", mode="nodes", points=100_000_000, width=2560, height=1440,
             height_m=250.0, window=0),
        # LOD with averaged colours and the weighted 3x3 resolve, odd screen.
        dict(name="lod_hqs_10M", kind="lod", mode="nodes_hqs", points=10_000_001, width=1366, height=768,
             height_m=150.0, window=1),
        # Opening four LAS files (formats 2, 3, 7, 8, odd point counts, so that
        # the later files start at unaligned points) and drawing the first
        # frame of the project with eye-dome lighting.
        dict(name="open_las_4M", kind="open_las", points=4_000_010, width=1280, height=720, edl=0.0005),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _screen(rng):
    return dict(width=rng.randint(320, 2560), height=rng.randint(240, 1440))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "points16", "stereo", "views", "lod", "open_las"])
    if kind == "frame":
        mode = rng.choice(["las2", "las2", "las", "hqs"])
        camera = rng.choice(["fly", "fly", "overview"])
        return dict(kind=kind, mode=mode, scene=rng.choice(["terrain", "city"]),
                    points=_log_int(rng, 2e5, 2e8 if mode == "las" else 1e9), camera=camera,
                    height_m=rng.uniform(60.0, 300.0) if camera == "fly" else 0.0,
                    edl=rng.choice([0.0, 0.0005]) if mode != "hqs" else 0.0, **_screen(rng))
    if kind == "points16":
        return dict(kind=kind, mode=rng.choice(["plain16", "hqs16"]), points=_log_int(rng, 1e5, 4e6), **_screen(rng))
    if kind == "stereo":
        return dict(kind=kind, mode="hqs", scene="city", points=_log_int(rng, 1e6, 1e9), **_screen(rng))
    if kind == "views":
        return dict(kind=kind, mode="las2", scene=rng.choice(["terrain", "city"]), points=_log_int(rng, 1e6, 5e8),
                    views=rng.randint(2, 40))
    if kind == "lod":
        mode = rng.choice(["nodes", "nodes_hqs"])
        return dict(kind=kind, mode=mode, points=_log_int(rng, 3e5, 1e8), height_m=rng.uniform(100.0, 400.0),
                    window=rng.randint(0, 2) if mode == "nodes_hqs" else 0, **_screen(rng))
    return dict(kind=kind, points=_log_int(rng, 1e5, 4e6), edl=rng.choice([0.0, 0.0005]), **_screen(rng))


# -------------------------------------------------------------------- prepare
class _DeviceArray:
    """A framebuffer plane as torch reads it in place."""

    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False), "version": 2}


def _plane(fb, ptr, typestr):
    t = torch.as_tensor(_DeviceArray(ptr, (fb.height, fb.width), typestr), device="cuda")
    t.framebuffer = fb   # the memory is the framebuffer's: it lives as long as the tensor
    return t


def _planes(fb, keys=True):
    """The framebuffer's image and keys (if it has any) as tensors over its own memory."""
    lib = pcr.capi.load()
    out = [_plane(fb, lib.pcr_fb_device_rgba(fb.h), "<i4")]
    if keys and fb.kind == pcr.FB_KEY64:
        out.append(_plane(fb, lib.pcr_fb_device_keys(fb.h), "<i8"))
    return out


def _cfg(scene, points, seed):
    return pcr.gen_cfg(pcr.SCENE_CITY if scene == "city" else pcr.SCENE_TERRAIN, points, seed=seed % 100003 + 1,
                       extent=EXTENT, num_buildings=256, terrain_frac=0.2)


def _fly_view(cfg, rng, height_m, width, height):
    """An eye height_m (+-10%) over the ground on a circle round the centre,
    looking ahead and down."""
    c = EXTENT / 2
    a = rng.uniform(0, 2 * math.pi)
    r = 650.0 + rng.uniform(-40, 40)
    ex, ey = c + r * math.cos(a), c + r * math.sin(a)
    ahead = a + math.pi / 2 + rng.uniform(-0.3, 0.3)
    tx, ty = ex + 400 * math.cos(ahead), ey + 400 * math.sin(ahead)
    eye = (ex, ey, pcr.ground_height(cfg, ex, ey) + height_m * rng.uniform(0.9, 1.1))
    tgt = (tx, ty, pcr.ground_height(cfg, tx, ty) + 20.0)
    return pcr.look_at(eye, tgt, up=(0, 0, 1), fovy=60.0, near=1.0, far=5000.0, width=width, height=height)


def _overview(cfg, rng, width, height):
    """Straight down from above the centre, the square (plus 5%) spanning the
    image's shorter side, turned by a random angle."""
    c = EXTENT / 2
    d = 1.05 * c / math.tan(math.radians(30.0)) * max(1.0, height / width)
    a = rng.uniform(0, 2 * math.pi)
    return pcr.look_at((c, c, cfg.amplitude + 80.0 + d), (c, c, 0.0), up=(math.cos(a), math.sin(a), 0), fovy=60.0,
                       near=1.0, far=10000.0, width=width, height=height)


def _server_views(n, rng):
    """Cameras over the scene, the serving resolutions in turn."""
    out = []
    for k in range(n):
        w, h = VIEW_SIZES[3 * k % len(VIEW_SIZES)]
        x, y = rng.uniform(0.15 * EXTENT, 0.85 * EXTENT, 2)
        a = rng.uniform(0, 2 * math.pi)
        out.append(pcr.look_at((x, y, rng.uniform(150.0, 400.0)),
                               (x + 500 * math.cos(a), y + 500 * math.sin(a), rng.uniform(0.0, 80.0)), up=(0, 0, 1),
                               fovy=60.0, near=1.0, far=5000.0, width=w, height=h))
    return out


def _eyes(rng, width, height, ipd=0.065):
    """Two eyes of a head at 250 m, 90 degrees field of view."""
    c = EXTENT / 2
    a = rng.uniform(0, 2 * math.pi)
    head = np.array([c + 650.0 * math.cos(a), c + 650.0 * math.sin(a), 250.0 + rng.uniform(-10, 10)])
    ahead = a + math.pi / 2 + rng.uniform(-0.3, 0.3)
    fwd = np.array([400 * math.cos(ahead), 400 * math.sin(ahead), 60.0 - head[2]])
    right = np.array([fwd[1], -fwd[0], 0.0])
    right *= (ipd / 2) / np.linalg.norm(right)
    return [pcr.look_at(tuple(head + s * right), tuple(head + s * right + fwd), up=(0, 0, 1), fovy=90.0, near=0.1,
                        far=5000.0, width=width, height=height) for s in (-1.0, 1.0)]


# the tiles of one LAS project (m) and its height range
LAS_TILE, LAS_RELIEF = 400.0, 60.0


def _las_file(points, point_format, version, origin, seed):
    """One tile of an airborne project: the points run through the tile cell
    by cell (flight lines), over rolling ground with some vegetation."""
    data = datasets.make_las(points, point_format=point_format, version=version, seed=seed,
                             extent=(LAS_TILE, LAS_TILE, LAS_RELIEF), offset=(origin[0], origin[1], 100.0))[0]
    rl = datasets.RECORD_LENGTH[point_format]
    raw = bytearray(data)
    rec = np.frombuffer(raw, np.uint8, points * rl, len(raw) - points * rl).reshape(points, rl)
    rng = np.random.default_rng(seed + 1)
    g = 64
    cell = np.arange(points, dtype=np.int64) * (g * g) // points
    x = (cell // g + rng.random(points)) * (LAS_TILE / g)
    y = (cell % g + rng.random(points)) * (LAS_TILE / g)
    z = 0.25 * LAS_RELIEF * (2 + np.sin(x / 60.0) * np.cos(y / 45.0)) + rng.exponential(1.0, points)
    xyz = np.stack([x, y, np.clip(z, 0.0, LAS_RELIEF - 0.01)], 1)
    rec[:, 0:12] = (xyz / 0.001).astype(np.int32).view(np.uint8)
    return bytes(raw)


MODES = dict(plain16=pcr.MODE_PLAIN16, las=pcr.MODE_LAS, las2=pcr.MODE_LAS2, hqs=pcr.MODE_HQS, nodes=pcr.MODE_NODES,
             hqs16=pcr.MODE_HQS16, nodes_hqs=pcr.MODE_NODES_HQS)


def prepare(case, seed):
    ctx, kind = _ctx(), case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "open_las":
        formats = ((2, (1, 2)), (3, (1, 3)), (7, (1, 4)), (8, (1, 4)))
        base = case["points"] // 4
        origins = [(500000.0 + LAS_TILE * (k % 2), 4000000.0 + LAS_TILE * (k // 2)) for k in range(4)]
        files = [_las_file(base + k - 1, f, v, origins[k], int(rng.integers(1 << 30)))
                 for k, (f, v) in enumerate(formats)]
        # each file is drawn in its own frame of reference, the project's
        # corner at the origin (the header minimum places the file)
        info = pcr.capi.LasInfo()
        views = []
        eye, tgt = (LAS_TILE, -0.6 * LAS_TILE, 300.0 + rng.uniform(-20, 20)), (LAS_TILE, LAS_TILE, 100.0)
        for d in files:
            pcr.check(pcr.capi.load().pcr_las_parse_header(d, len(d), ctypes.byref(info)))
            origin = (info.min[0] - 500000.0, info.min[1] - 4000000.0, info.min[2])
            views.append(pcr.look_at(eye, tgt, up=(0, 0, 1), near=1.0, far=5000.0, origin=origin,
                                     width=case["width"], height=case["height"]))
        fb = ctx.framebuffer(case["width"], case["height"])
        return dict(kind=kind, files=files, views=views, fb=fb, edl=case["edl"], out=_planes(fb))
    mode = MODES[case["mode"]]
    hqs = mode in (pcr.MODE_HQS, pcr.MODE_HQS16, pcr.MODE_NODES_HQS)
    fb_kind = pcr.FB_HQS if hqs else pcr.FB_KEY64
    if kind == "points16":
        cloud = ctx.generate(pcr.gen_cfg(pcr.SCENE_CUBE, case["points"], seed=seed % 100003 + 1), morton_sort=False,
                             keep_points16=True)
        a = rng.uniform(-0.2, 0.2)
        views = [pcr.look_at((0.5 + 2 * math.sin(a), 0.5, 0.5 + 2 * math.cos(a)), (0.5, 0.5, 0.5), up=(0, 1, 0),
                             fovy=60.0, near=0.1, far=1000.0, width=case["width"], height=case["height"])]
    elif kind == "lod":
        cfg = _cfg("city", case["points"], seed)
        cloud = ctx.octree_generate(cfg, seed=seed % 1009)
        views = [_fly_view(cfg, rng, case["height_m"], case["width"], case["height"])]
    else:
        cfg = _cfg(case["scene"], case["points"], seed)
        cloud = ctx.generate(cfg)
        if kind == "stereo":
            views = _eyes(rng, case["width"], case["height"])
        elif kind == "views":
            views = _server_views(case["views"], rng)
        elif case["camera"] == "overview":
            views = [_overview(cfg, rng, case["width"], case["height"])]
        else:
            views = [_fly_view(cfg, rng, case["height_m"], case["width"], case["height"])]
    prm = pcr.params(mode, edl_strength=case.get("edl", 0.0), resolve_window=case.get("window", 0))
    fbs = [ctx.framebuffer(v.width, v.height, fb_kind) for v in views]
    state = dict(kind=kind, cloud=cloud, views=views, fbs=fbs, prm=prm)
    if kind in ("stereo", "views"):
        # the configuration that autotuning picks for these launches
        state["plan"] = pcr.MultiView(ctx, cloud, views, fbs, prm, tune=pcr.capi.Tune(256, 40, 0, 2048))
    # every view's image; the keys too, but for the many-view launch
    state["out"] = [t for fb in fbs for t in _planes(fb, keys=kind != "views")]
    return state


# ------------------------------------------------------------------------ run
def run(state):
    ctx, kind = _ctx(), state["kind"]
    if kind == "open_las":
        cloud, first = ctx.from_las(state["files"])
        fb = state["fb"]
        prm = None
        for k, view in enumerate(state["views"]):
            prm = pcr.params(pcr.MODE_LAS2, clear_before=int(k == 0), batch_begin=int(first[k]),
                             batch_end=int(first[k + 1]), edl_strength=state["edl"])
            ctx.render(cloud, view, prm, fb)
        ctx.resolve(cloud, prm, fb)
        state["cloud"] = cloud   # the project stays open until the next one
    elif kind == "stereo":
        state["plan"].set_views(state["views"])
        state["plan"].launch()
    elif kind == "views":
        state["plan"].launch()
    else:
        fb = state["fbs"][0]
        ctx.render(state["cloud"], state["views"][0], state["prm"], fb)
        ctx.resolve(state["cloud"], state["prm"], fb)
    return state["out"]


def exact(case, seed):
    """Every output is a whole number: keys hold a point's index (or colour)
    beside the bits of its single-precision depth, images hold bytes. Which
    point owns a pixel is defined by the fixed single-precision order of
    operations; there is no 64-bit value of it."""
    return None


# ----------------------------------------------------------------------- work
def work(case):
    """One pass: the headers and the 10-bit plane of the batches in view, the
    colours that are looked up, and the framebuffer written once (key and
    image). In an averaged-colour frame every point in view gives its colour.
    `share` is the measured part of the scene's points that lie in batches in
    view. A point costs a decode (6 operations), a transform (18), a division
    (3) and the pixel (6)."""
    kind, n = case["kind"], case["points"]
    pixels = case.get("width", 0) * case.get("height", 0)
    hqs = case.get("mode") in ("hqs", "hqs16", "nodes_hqs")
    if kind == "open_las":
        # records (26 to 38 bytes) in, planes and colours (16 bytes) out, then the frame
        return {"bytes": n * (32.5 + 16 + 4) + 12 * pixels, "flops": 33 * n}
    if kind == "points16":
        return {"bytes": 16 * n + (4 if hqs else 12) * pixels, "flops": 27 * n}
    if kind == "lod":
        drawn = min(n, pixels)
        return {"bytes": drawn * (8 if hqs else 4) + (4 if hqs else 12) * pixels, "flops": 33 * drawn}
    if kind == "views":
        per_view = sum(w * h for w, h in VIEW_SIZES) / len(VIEW_SIZES)
        return {"bytes": 4 * n + 12 * per_view * case["views"], "flops": 33 * 0.25 * n * case["views"]}
    eyes = 2 if kind == "stereo" else 1
    share = 1.0 if case.get("camera") == "overview" else 0.3 if hqs else 0.19
    return {"bytes": 64 * n / 10240 + share * n * (8 if hqs else 4) + eyes * (4 if hqs else 12) * pixels,
            "flops": 33 * share * n * eyes}
