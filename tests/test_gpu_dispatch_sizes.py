"""The sizes at which a launch changes form, against the oracle: how the
raster deals screen tiles to the XCDs, how many blocks project a cull tile,
which radix-sort tile one view takes."""
import numpy as np
import pytest

import oracle_bind as ob
import splatter_amd as sa
from gpu_common import Case, config, device, image_diff, normwise_rel, say
from splatter_amd.synth import Workload, look_at, sphere_pose

pytestmark = pytest.mark.gpu

IMAGE_TOL = 2      # of 255, the image bar of test_gpu_parity
RECORD_TOL = 1e-5  # the record bar of test_gpu_parity


# 1, 31, 32, 33 and 64 + 1 tiles: one tile, the edges of eight runs of four
# tiles (one turn of the XCDs), and a second turn that has just begun
@pytest.mark.parametrize("width,height", [(16, 16), (31 * 16, 9), (32 * 16, 16), (33 * 16 - 3, 16), (13 * 16, 5 * 16)])
def test_every_tile_is_drawn_once(width, height):
    say(f"frame {width}x{height}")
    case = Case(Workload("gaussian", 3000, seed=31), config(max_views=2), width, height, sphere_pose(31, radius=4))
    img = case.render()
    _, _, _, oimg = case.oracle()
    assert image_diff(img, oimg) <= IMAGE_TOL
    other = sa.Frame(device(), 40, 40)  # the same view beside a smaller one, whose tiles end inside a turn
    case.renderer.render_views([other, case.frame], [case.cam] * 2, [case.view] * 2, case.scene)
    assert np.array_equal(case.frame.read()[..., [2, 1, 0, 3]], img)


# 48, 96, 192 and 384 cull tiles of 4096 splats are the most that 16, 8, 4 and
# 2 blocks share on 256 CUs; one splat more starts the next form, with a last
# tile of one splat
@pytest.mark.parametrize("count", [1, 255, 4097, 48 * 4096, 48 * 4096 + 1, 96 * 4096 + 1, 192 * 4096 + 1,
                                   384 * 4096 + 1])
@pytest.mark.parametrize("views", [1, 3])
def test_blocks_that_share_a_cull_tile(count, views):
    say(f"{count} splats, {views} views")
    w = Workload("gaussian", count, seed=33)
    cfg = config(max_splat_count=count, max_views=views, tile_pairs_per_splat=8)
    r = sa.Renderer(device(), cfg)
    scene = sa.Scene(r, count)
    records = w.all()
    scene.load_records(0, records)
    splats = ob.decode(records)
    poses = [sphere_pose(40 + v, radius=4) for v in range(views)]
    frames = [sa.Frame(device(), 96, 64) for _ in range(views)]
    r.render_views(frames, [p[0] for p in poses], [p[1] for p in poses], scene)
    for v, (cam, view) in enumerate(poses):
        r.select_view(v)
        _, idx = r.read_entries()
        u = ob.uniforms(cam, view, 96, 64)
        _, oidx = ob.cpu_depth_sort(splats["center"], ob.vp_of(u), 1.1)
        assert np.array_equal(idx, oidx)
        if not len(idx):
            continue
        sub = np.unique(np.linspace(0, len(idx) - 1, min(len(idx), 3000)).astype(np.int64))
        rec = r.read_records()[sub]
        orec, _ = ob.project(splats[idx[sub]], u, cfg.spherical_harmonics_order, cfg.use_covariance_for_scale)
        assert np.array_equal(rec[:, :4], orec[:, :4])
        assert normwise_rel(rec[:, 4:], orec[:, 4:]).max() <= RECORD_TOL


# the sizes at which one view's depth sort (test_sort_tiles.py has its lines) and
# pair sort (2^15, 2^19, 2^21 splats) change their tiles, and where a batch's do
# (2^22)
@pytest.mark.parametrize("count", [1000, 1 << 15, (1 << 15) + 1, 7 << 14, (7 << 14) + 1, 1 << 17, (1 << 17) + 1,
                                   1 << 19, (1 << 19) + 1, 1 << 20, (1 << 20) + 1, 1 << 21, (1 << 21) + 1,
                                   (1 << 22) + 1])
@pytest.mark.parametrize("bits", [8, 10])
def test_sort_tile_of_one_view(count, bits):
    say(f"{count} splats, {bits}-bit digits")
    r = sa.Renderer(device(), config(max_splat_count=count, radix_bits_per_digit=bits, tile_pairs_per_splat=8,
                                     max_views=2))
    w = Workload("gaussian", count, seed=35)
    scene = sa.Scene(r, count)
    centers = np.empty((count, 3), np.float32)
    for first, rec in w.chunks():
        scene.load_records(first, rec)
        centers[first:first + len(rec)] = rec["center"]
    cam, view = sphere_pose(35, radius=5)
    frames = [sa.Frame(device(), 640, 360) for _ in range(2)]
    r.render_frame(frames[0], cam, view, scene)
    keys, idx = r.read_entries()
    okeys, oidx = ob.cpu_depth_sort(centers, ob.vp_of(ob.uniforms(cam, view, 640, 360)), 1.1)
    assert np.array_equal(idx, oidx) and np.array_equal(keys, okeys)
    # a batch of the view twice, in the batches' tiles: the same lists, the same image
    r.render_views(frames[::-1], [cam] * 2, [view] * 2, scene)
    assert np.array_equal(frames[0].read(), frames[1].read())
    batch = frames[0].read()
    r.render_frame(frames[0], cam, view, scene)
    assert np.array_equal(frames[0].read(), batch)


# One view of 2^21 splats sorts its pairs in 8192-key tiles while one a CU holds
# them (2^21 on 256 CUs) and in 16384-key ones beyond: one pair short, that many
# and a few more, each splat but the first in the middle of a screen tile.
@pytest.mark.parametrize("first", ["behind", "small", "large"])
def test_pair_tile_by_count(first):
    n, width, height = 1 << 21, 1280, 720
    rng = np.random.default_rng(73)
    z = rng.uniform(3.0, 6.0, n)
    x = (2.0 * (16 * rng.integers(0, width // 16, n) + 8) / width - 1.0) * z * width / height
    y = (2.0 * (16 * rng.integers(0, height // 16, n) + 8) / height - 1.0) * z
    base = Workload("gaussian", 1 << 16, seed=73).all()
    rec = np.tile(base, n // len(base))
    rec["center"] = np.stack([x, y, z - 5.0], axis=1)
    rec["scale"] = -4.5  # a pixel or two
    if first == "behind":
        rec["center"][0] = (0.0, 0.0, -20.0)
    if first == "large":
        rec["scale"][0] = -1.5
    r = sa.Renderer(device(), config(max_splat_count=n, max_views=2, tile_pairs_per_splat=2))
    assert sa.sort_tiles(r.config, n, 1)[1] == 0
    scene = sa.Scene(r, n)
    scene.load_records(0, rec)
    cam, view = look_at((0, 0, -5), (0, 0, 0))
    frames = [sa.Frame(device(), width, height) for _ in range(2)]
    for _ in range(2):  # the second frame finds what the first one cleared
        r.render_frame(frames[0], cam, view, scene)
    img, pairs = frames[0].read(), r.pair_count()
    say(f"first splat {first}: {pairs} pairs")
    assert pairs == n - 1 if first == "behind" else pairs == n if first == "small" else n < pairs < n + 100
    # a batch of the view twice sorts them in 4096-key tiles: the same image
    r.render_views(frames[::-1], [cam] * 2, [view] * 2, scene)
    assert r.pair_count() == pairs
    assert np.array_equal(frames[0].read(), img) and np.array_equal(frames[1].read(), img)
    assert img[..., :3].any()


# Batches sort in the configured tile, of sixteen keys a lane above 2^21 splats
# in all and of eight below; above 2^22 splats in 16384-key tiles (depths).
@pytest.mark.parametrize("count", [1 << 20, (1 << 20) + 1, (1 << 22) + 1])
@pytest.mark.parametrize("tile", [4096, 8192, 16384])
@pytest.mark.parametrize("bits", [8, 10])
def test_sort_tile_of_batches(count, tile, bits):
    say(f"{count} splats, {tile}-key tiles, {bits}-bit digits")
    cfg = config(max_splat_count=count, radix_bits_per_digit=bits, sort_tile_keys=tile, tile_pairs_per_splat=8,
                 max_views=2)
    assert sa.sort_tiles(cfg, count, 2) == ((tile, tile) if count <= 1 << 22 else (16384, max(tile, 8192)))
    r = sa.Renderer(device(), cfg)
    w = Workload("gaussian", count, seed=35)
    scene = sa.Scene(r, count)
    centers = np.empty((count, 3), np.float32)
    for first, rec in w.chunks():
        scene.load_records(first, rec)
        centers[first:first + len(rec)] = rec["center"]
    poses = [sphere_pose(35, radius=5), sphere_pose(36, radius=5)]
    frames = [sa.Frame(device(), 320, 180) for _ in range(2)]
    r.render_views(frames, [p[0] for p in poses], [p[1] for p in poses], scene)
    batch = [f.read() for f in frames]
    for v, (cam, view) in enumerate(poses):
        r.select_view(v)
        keys, idx = r.read_entries()
        okeys, oidx = ob.cpu_depth_sort(centers, ob.vp_of(ob.uniforms(cam, view, 320, 180)), 1.1)
        assert np.array_equal(idx, oidx) and np.array_equal(keys, okeys)
    r.select_view(0)
    for f, img, (cam, view) in zip(frames, batch, poses):
        r.render_frame(f, cam, view, scene)  # its pairs in the single view's tiles
        assert np.array_equal(f.read(), img)


# Every instance of the raster: batches with 128 and with 256 entries a round, one
# list with blocks of its own (all splats at the first tile) and ordinary ones
# of several rounds.
@pytest.mark.parametrize("entries", [128, 256])
@pytest.mark.parametrize("mode", [0, 1, 2, 3])
@pytest.mark.parametrize("unaligned,blend", [(True, sa.BlendMode.UNORM8), (False, sa.BlendMode.F32),
                                             (True, sa.BlendMode.F32), (False, sa.BlendMode.UNORM8)])
def test_raster_forms_of_batches(entries, mode, unaligned, blend):
    say(f"{entries} entries a round, mode {mode}, unaligned {unaligned}, blend {blend}")
    count, width, height = 8000, 100, 75
    case = Case(Workload("gaussian", count, seed=81),
                config(max_splat_count=count, max_views=2, raster_mode=mode, raster_batch=entries,
                       use_unaligned_rectangles=unaligned, blend_mode=blend, tile_pairs_per_splat=16), width, height,
                sphere_pose(81, radius=6))
    other = sa.Frame(device(), 16, 16)
    case.renderer.enable_tile_stats(True)
    case.renderer.render_views([case.frame, other], [case.cam] * 2, [case.view] * 2, case.scene)
    lens = case.renderer.tile_stats()[:, 0]
    say(f"  lists {lens.min()} to {lens.max()}")
    assert lens.max() >= 512 and np.count_nonzero((lens > 256) & (lens < 512)) >= 2
    img = case.frame.read()
    if case.cfg.frame_format == sa.FrameFormat.BGRA8_UNORM:
        img = img[..., [2, 1, 0, 3]]
    _, _, _, oimg = case.oracle()
    assert image_diff(img, oimg) <= IMAGE_TOL
    small = other.read()
    assert np.array_equal(case.render(), img)
    case.renderer.render_frame(other, case.cam, case.view, case.scene)
    assert np.array_equal(other.read(), small)


# A list of 512 pairs and 1/1000 of the frame's makes a tile heavy.  Lists from
# one below that to a few batches of 128 and chunks of 64 entries more, in
# whole and cut sub-blocks, that stay transparent or turn opaque on the way.
@pytest.mark.parametrize("count,logit", [(511, -4.0), (512, -4.0), (513, -4.0), (640, -4.0), (641, -6.0), (1000, -4.0),
                                         (5000, -6.0), (5000, 0.0), (5000, 6.0)])
@pytest.mark.parametrize("width,height", [(16, 16), (13, 5), (21, 18)])
@pytest.mark.parametrize("unaligned,blend", [(True, sa.BlendMode.UNORM8), (False, sa.BlendMode.F32),
                                             (True, sa.BlendMode.F32), (False, sa.BlendMode.UNORM8)])
def test_heavy_tiles(count, logit, width, height, unaligned, blend):
    say(f"{count} splats, opacity logit {logit}, {width}x{height}, unaligned {unaligned}, blend {blend}")
    case = Case(Workload("gaussian", 0, seed=0),
                config(max_splat_count=count, max_views=2, use_unaligned_rectangles=unaligned, blend_mode=blend,
                       tile_pairs_per_splat=8), width, height, sphere_pose(51, radius=5))
    rec = Workload("gaussian", count, seed=51).all()
    rec["center"] *= 0.1  # in front of the camera, all in the first tile of a 16x16 frame
    rec["scale"] += 2.0   # a few pixels each
    rec["alpha"] = logit
    case.records, case.splats = rec, ob.decode(rec)
    case.scene = sa.Scene(case.renderer, count)
    case.scene.load_records(0, rec)
    case.renderer.enable_tile_stats(True)
    img = case.render()
    lens = case.renderer.tile_stats()
    say(f"  lists {lens[:, 0].tolist()}, consumed {lens[:, 1].tolist()}")
    if (width, height) == (16, 16):
        assert lens[0, 0] == count  # the list the case is about
    assert (lens[:, 1] <= lens[:, 0]).all()
    if logit < 0.0:  # nothing turns opaque: every tile's list is read to its end
        assert (lens[:, 1] == lens[:, 0]).all()
    _, _, _, oimg = case.oracle()
    assert image_diff(img, oimg) <= IMAGE_TOL
    # the same view in a batch, whose other view has lists of its own
    other = sa.Frame(device(), 40, 24)
    case.renderer.render_views([case.frame, other], [case.cam] * 2, [case.view] * 2, case.scene)
    got = case.frame.read()
    assert np.array_equal(got[..., [2, 1, 0, 3]] if case.cfg.frame_format == sa.FrameFormat.BGRA8_UNORM else got, img)


# Bin tiles of 256 entries up to 2^17 splats in the batch and of 1024 beyond,
# whose pairs expand 4096 slots at a time: one splat that covers thousands of
# screen tiles, a tile's pairs just below and above 4096, boxes as wide as the
# frame
@pytest.mark.parametrize("count,big,width,height", [(1, 1, 2048, 1024), (256, 1, 1024, 1008), (257, 256, 64, 64),
                                                    (1024, 1024, 32, 32), (1025, 1024, 48, 32), (5000, 300, 320, 240),
                                                    ((1 << 17) + 1, 64, 640, 480)])
@pytest.mark.parametrize("views", [1, 2])
def test_bin_slots(count, big, width, height, views):
    say(f"{count} splats, {big} of them large, {width}x{height}, {views} views")
    rec = Workload("gaussian", count, seed=61).all()
    rec["center"][:big] *= 0.2
    rec["scale"][:big] = 1.0     # e, as large as the view
    rec["alpha"][:big] = -5.0
    cfg = config(max_splat_count=count, max_views=views, tile_pairs_per_splat=16384 if count < 2000 else 64)
    case = Case(Workload("gaussian", 0, seed=0), cfg, width, height, sphere_pose(61, radius=5))
    case.records, case.splats = rec, ob.decode(rec)
    case.scene = sa.Scene(case.renderer, count)
    case.scene.load_records(0, rec)
    others = [sa.Frame(device(), 33, 17) for _ in range(views - 1)]
    case.renderer.render_views([case.frame] + others, [case.cam] * views, [case.view] * views, case.scene)
    say(f"  pairs {case.renderer.pair_count()}")
    _, _, _, oimg = case.oracle()
    assert image_diff(case.frame.read()[..., [2, 1, 0, 3]], oimg) <= IMAGE_TOL


# ordinary tiles with at least 128 pairs (a quarter of the heavy threshold) and
# twice the view's mean start first, one block each, in single views and batches
@pytest.mark.parametrize("count,views", [(6000, 1), (6000, 3), (60_000, 2)])
def test_long_tiles(count, views):
    say(f"{count} splats, {views} views")
    case = Case(Workload("gaussian", count, seed=71), config(max_views=views, tile_pairs_per_splat=16), 500, 300,
                sphere_pose(71, radius=9))
    case.renderer.enable_tile_stats(True)
    others = [sa.Frame(device(), 300 - 40 * i, 200) for i in range(views - 1)]
    case.renderer.render_views([case.frame] + others, [case.cam] * views, [case.view] * views, case.scene)
    lens = case.renderer.tile_stats()[:, 0].astype(np.int64)
    few = max(512, lens.sum() // 1000)
    longs = np.count_nonzero((lens >= max(few // 4, 2 * (lens.sum() // len(lens)))) & (lens < few))
    say(f"  mean list {lens.mean():.0f}, max {lens.max()}, long tiles {longs}")
    assert longs > 0
    _, _, _, oimg = case.oracle()
    assert image_diff(case.frame.read()[..., [2, 1, 0, 3]], oimg) <= IMAGE_TOL
    for f in others:  # each view of the batch equals its own frame
        got = f.read()
        case.renderer.render_frame(f, case.cam, case.view, case.scene)
        assert np.array_equal(f.read(), got)
