"""The framework's measured work: frames rendered from resident scenes.

A program that uses this framework loads a scene once and then asks for
frames of it, one camera after another, one view at a time (a viewer), many
views at once (an offline orbit, training images), through the workspace-free
entry point, or as a stream of requests to the server.  A case is one such
call with its pixels delivered to host memory: the matrices go in, and the
image comes back in a pinned buffer that the program keeps.

The scenes are the kinds that splatter_amd.synth describes, made on the GPU so
that a 32M-splat scene takes seconds: `gaussian` (one blob), `clustered` (64
anisotropic clusters over a ground slab, the spread of a captured scene) and
`tight` (16 dense clusters, most depths tied).  Sizes, views per batch and
options are those of bench.py and of the tests, or lie between them.

Fields of a case:
  form     frame: Renderer.render_frame; views: Renderer.render_views;
           static: Device.render_frame_static; serve: Server
  scene, splats          kind and size of the scene (serve: of the largest of three)
  width, height          the frame (serve: of its largest request)
  views                  views per call (serve: requests)
  sh                     spherical harmonics order
  digits, sort_tile      radix_bits_per_digit and sort_tile_keys
  fov                    vertical field of view in degrees
  ragged                 views of one batch differ in size
  plain_options          True: the reference showcase's options; False: the other
                         branch of each (no depth sorting, axis-aligned squares,
                         contour scales, f32 blend, RGBA)
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import splatter_amd as sa
from splatter_amd._lib import check, lib
from splatter_amd.synth import look_at

_DEFAULTS = {"form": "frame", "scene": "clustered", "views": 1, "sh": 3, "digits": 8, "sort_tile": 4096, "fov": 90,
             "ragged": False, "plain_options": True}


def _case(name, **kw):
    c = dict(_DEFAULTS)
    c.update(kw)
    c["name"] = name
    return c


def listed():
    return [
        # a thumbnail of a small object: launches and latency
        _case("thumb_20k", scene="gaussian", splats=20_000, width=320, height=180, fov=60),
        # the reference's CPU-runnable scene in a window
        _case("window_100k", scene="gaussian", splats=100_000, width=1280, height=720, fov=60),
        # code that may not allocate (stream capture, tight loops)
        _case("static_100k", form="static", scene="gaussian", splats=100_000, width=640, height=480, fov=60),
        # a preview of a captured scene: many splats on few screen tiles
        _case("preview_1500k_vga", splats=1_500_000, width=640, height=480),
        # the showcase's options (SH 2) on a mid-size scene, full HD
        _case("viewer_1m_1080p", splats=1_000_000, width=1920, height=1080, sh=2),
        # the headline scene, one view at a time
        _case("viewer_6m_1080p", splats=6_000_000, width=1920, height=1080),
        # a 4K display
        _case("viewer_3m_4k", splats=3_000_000, width=3840, height=2160),
        # the other branch of every option, at an odd size
        _case("options_400k_odd", splats=400_000, width=1273, height=711, sh=1, plain_options=False),
        # a small batch of unequal odd views (training crops)
        _case("crops_300k_5views", form="views", splats=300_001, width=799, height=601, views=5, ragged=True),
        # the headline batch: 16 orbit views of 6M splats, with the autotuner's sort form
        _case("orbit_6m_16views", form="views", splats=6_000_000, width=1920, height=1080, views=16, digits=10,
              sort_tile=16384),
        # the sort's stress scene: 32M splats, nearly all visible, most depths tied, 8 views at 4K
        _case("stress_32m_8views", form="views", scene="tight", splats=32_000_000, width=3840, height=2160, views=8),
        # a burst of requests for three scenes at the server's four usual sizes
        _case("serve_12_requests", form="serve", splats=3_000_000, width=3840, height=2160, views=12),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    form = rng.choice(["frame", "frame", "frame", "views", "views", "static", "serve"])
    kw = {"form": form, "fov": rng.choice([45, 60, 75, 90]), "sh": rng.choice([0, 1, 2, 3, 3]),
          "digits": rng.choice([8, 8, 10]), "sort_tile": rng.choice([4096, 8192, 16384]),
          "scene": rng.choice(["gaussian", "clustered", "clustered", "tight"])}
    width = _log_uniform(rng, 160, 3840)
    height = max(90, min(2160, int(width * rng.uniform(0.45, 0.85))))
    kw.update(width=width, height=height)
    if form == "frame":
        kw.update(splats=_log_uniform(rng, 5_000, 8_000_000), plain_options=rng.random() < 0.8)
    elif form == "views":
        kw.update(splats=_log_uniform(rng, 20_000, 6_000_000), views=rng.randint(2, 16), ragged=rng.random() < 0.5)
    elif form == "static":
        kw.update(splats=_log_uniform(rng, 2_000, 131_072), scene="gaussian", fov=60)
        kw["width"] = min(width, 1920)
        kw["height"] = min(height, 1080)
    else:
        kw.update(splats=_log_uniform(rng, 100_000, 3_000_000), views=rng.randint(3, 16), scene="clustered")
    c = _case(None, **kw)
    del c["name"]
    return c


# ---- inputs ---------------------------------------------------------------


def _rotations(gen, k):
    q = torch.randn(k, 4, generator=gen, dtype=torch.float64)
    w, x, y, z = (q / q.norm(dim=1, keepdim=True)).unbind(1)
    return torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                        2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                        2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], 1).view(k, 3, 3)


def _load(scene, kind, count, seed):
    """Fills a scene with `count` records of the distributions in
    splatter_amd.synth, 4M at a time through Scene.load_records."""
    host = torch.Generator().manual_seed(seed)
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    k = 64 if kind == "clustered" else 16
    spread = 10.0 if kind == "clustered" else 5.0
    centres = ((torch.rand(k, 3, generator=host) * 2 - 1) * spread).to(dev)
    sigmas = torch.exp(torch.rand(k, 3, generator=host) * math.log(10.0) + math.log(0.1)).to(dev)
    turns = _rotations(host, k).float().to(dev)
    for first in range(0, count, 1 << 22):
        n = min(1 << 22, count - first)

        def normal(*shape, mean=0.0, std=1.0):
            return torch.randn(*shape, generator=gen, device=dev) * std + mean

        rec = torch.zeros(n, 62, device=dev)
        if kind == "gaussian":
            rec[:, 0:3] = normal(n, 3, std=2.0)
        else:
            cid = torch.randint(k, (n,), generator=gen, device=dev)
            if kind == "tight":
                rec[:, 0:3] = centres[cid] + normal(n, 3, std=0.05)
            else:
                local = normal(n, 3) * sigmas[cid]
                pos = centres[cid] + (turns[cid] * local[:, None, :]).sum(2)
                slab = (torch.rand(n, 3, generator=gen, device=dev) * 2 - 1) * torch.tensor([30.0, 30.0, 0.2], device=dev)
                ground = torch.rand(n, 1, generator=gen, device=dev) >= 0.8
                rec[:, 0:3] = torch.where(ground, slab, pos)
        rec[:, 6:54] = normal(n, 48, std=0.05)
        rec[:, 6:9] = normal(n, 3, std=0.5)
        rec[:, 54] = normal(n, std=1.5)
        rec[:, 55:58] = normal(n, 3, mean=-4.0, std=0.5)
        rec[:, 58:62] = normal(n, 4)
        scene.load_records(first, rec.cpu().numpy().view(sa.SERIALIZED_SPLAT_DTYPE).reshape(n))


def _pose(case, rng, turn):
    """A camera on an orbit around the scene, `turn` of a full circle on."""
    radius = {"gaussian": 5.0, "clustered": 6.0, "tight": 9.0}[case["scene"]]
    az = 2.0 * math.pi * (rng.uniform() + turn)
    el = math.radians(20.0 + 10.0 * rng.uniform(-1.0, 1.0))
    eye = (radius * math.cos(el) * math.cos(az), radius * math.cos(el) * math.sin(az), radius * math.sin(el))
    return look_at(eye, (0.0, 0.0, 0.0), (0.0, 0.0, 1.0))


def _configuration(case, splats, views):
    cfg = sa.Configuration(spherical_harmonics_order=case["sh"], max_splat_count=splats, max_views=views,
                           radix_bits_per_digit=case["digits"], sort_tile_keys=case["sort_tile"],
                           field_of_view_y=math.radians(case["fov"]), tile_pairs_per_splat=8)
    if not case["plain_options"]:
        cfg.depth_sorting = sa.DepthSorting.NONE
        cfg.use_covariance_for_scale = False
        cfg.use_unaligned_rectangles = False
        cfg.blend_mode = sa.BlendMode.F32
        cfg.frame_format = sa.FrameFormat.RGBA8_UNORM
    return cfg


_SERVED_SIZES = ((1, 1), (2, 2), (3, 3), (6, 4.5))  # largest request over this one: 4K, 1080p, 720p, VGA


def _sizes(case):
    w, h = case["width"], case["height"]
    if case["form"] == "serve":
        return [(max(16, int(w / a)), max(16, int(h / b))) for a, b in
                (_SERVED_SIZES[i % 4] for i in range(case["views"]))]
    if case["ragged"]:
        return [(max(33, w - 61 * i), max(17, h - 43 * i)) for i in range(case["views"])]
    return [(w, h)] * case["views"]


_device = None


def _open():
    global _device
    if _device is None:
        torch.zeros(1, device="cuda")
        _device = sa.Device(0)
    return _device


class _State:
    pass


def prepare(case, seed):
    """A program with its scene resident: renderer (or server), scene, frames,
    the cameras of this call and the host buffers the images go to."""
    dev = _open()
    rng = np.random.default_rng([seed, 0xCA])
    s = _State()
    s.form, s.device = case["form"], dev
    s.sizes = _sizes(case)
    s.poses = [_pose(case, rng, i / case["views"]) for i in range(case["views"])]
    s.cams, s.views = [p[0] for p in s.poses], [p[1] for p in s.poses]
    s.host = [torch.empty(h, w, 4, dtype=torch.uint8, pin_memory=True) for w, h in s.sizes]
    n = case["splats"]
    if s.form == "serve":
        s.config = _configuration(case, n, 8)
        s.server = sa.Server(dev, s.config, max_width=case["width"], max_height=case["height"])
        s.scenes = []
        for i, m in enumerate((max(1, n // 10), max(1, n // 3), n)):
            s.scenes.append(s.server.create_scene(m))
            _load(s.scenes[-1], case["scene"], m, 3 * seed + i)
        return s
    s.config = _configuration(case, n, case["views"])
    s.renderer = sa.Renderer(dev, s.config)
    s.scene = sa.Scene(s.renderer, n)
    _load(s.scene, case["scene"], n, seed)
    s.frames = [sa.Frame(dev, w, h) for w, h in s.sizes]
    return s


def run(s):
    """One call: render, then each image into its pinned buffer."""
    if s.form == "serve":
        tickets = [s.server.submit(s.scenes[i % 3], w, h, s.cams[i], s.views[i]) for i, (w, h) in enumerate(s.sizes)]
        for t, out in zip(tickets, s.host):
            check(lib().spl_server_read(s.server.handle, t, C.c_void_p(out.data_ptr()), out.numel()))
            s.server.release(t)
        s.server.poll()
        return s.host
    if s.form == "frame":
        s.renderer.render_frame(s.frames[0], s.cams[0], s.views[0], s.scene)
    elif s.form == "static":
        s.device.render_frame_static(s.config, s.frames[0], s.cams[0], s.views[0], s.scene)
    else:
        s.renderer.render_views(s.frames, s.cams, s.views, s.scene)
    for f, out in zip(s.frames, s.host):
        check(lib().spl_frame_read(f.handle, C.c_void_p(out.data_ptr()), out.numel()))
    return s.host


# ---- what a pass cannot do without -----------------------------------------

# Share of the splats that a view sees, and fragments blended per pixel
# before it is opaque: the means of these scenes from such orbits.
_VISIBLE = {"gaussian": 0.8, "clustered": 0.5, "tight": 1.0}
_FRAGMENTS = 16
_PROJECT_FLOPS, _FRAGMENT_FLOPS = 450, 35


def work(case):
    """Every centre read once, the other attributes of the splats that some
    view sees read once, every pixel written once; the projection of each
    visible splat in each view and the blends of each pixel."""
    sh = 12 * (case["sh"] + 1) ** 2
    n, views = case["splats"], case["views"]
    pixels = sum(w * h for w, h in _sizes(case))
    seen = _VISIBLE[case["scene"]]
    if case["form"] == "serve":
        n, views = int(n * (1 + 1 / 3 + 0.1)), views / 3
    return {"bytes": n * (12 + seen * (32 + sh)) + 4 * pixels,
            "flops": views * n * seen * _PROJECT_FLOPS + pixels * _FRAGMENTS * _FRAGMENT_FLOPS}


def tolerance(case):
    """Pixels are bytes: the order of the blends is the depth order with ties
    by splat index, each blend rounds as the 8-bit target does, and the same
    scene and camera give the same image on every path.  (The images are
    compared with a 64-bit oracle by the tests.)"""
    return "exact"
