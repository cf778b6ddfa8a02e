"""The staged autotuner's selection rule (host logic, no device): each stage
tries its candidates in order of preference and a later candidate replaces
the pick only when it is more than the tie margin faster."""
from types import SimpleNamespace

import pytest

import splatter_amd as sa
from splatter_amd import autotune as at


def _run(monkeypatch, fps_of):
    order = []

    def fake_measure(sa, device, base, scene_loader, poses, width, height, cand, steps, in_flight):
        order.append(cand.key())
        return fps_of(cand)

    monkeypatch.setattr(at, "measure", fake_measure)
    base = SimpleNamespace(raster_batch=128)
    res = at.autotune_staged(None, None, base, None, None, 64, 48, 16, steps=1, in_flight=2)
    return res, order


def test_preference_order_and_tie(monkeypatch):
    # 8192-key tiles 2% ahead of 16384: inside the 3% margin, so 16384 stays
    def fps_of(c):
        f = {16384: 1500.0, 8192: 1530.0, 4096: 1400.0}[c.sort_tile_keys]
        f += 1.0 if c.radix_bits_per_digit == 10 else 0.0
        f -= 100.0 * (c.raster_batch == 256)
        return f
    res, order = _run(monkeypatch, fps_of)
    assert order[0] == "r10-t16384-b128-m3-o0-v16" and order[1] == "r8-t16384-b128-m3-o0-v16"
    assert res.best.sort_tile_keys == 16384 and res.best.radix_bits_per_digit == 10
    assert res.best.raster_batch == 128 and res.best.raster_longest_first == 0
    assert res.best.raster_mode == 3  # the preferred walk, no slower than entry-major here
    assert len(res.table) == 6 + 4


def test_clear_win_replaces_the_pick(monkeypatch):
    # 4096-key tiles 10% ahead: a clear win; 256-entry batches 5% ahead: taken too
    def fps_of(c):
        f = {16384: 1000.0, 8192: 1010.0, 4096: 1100.0}[c.sort_tile_keys]
        return f * (1.05 if c.raster_batch == 256 else 1.0)
    res, _ = _run(monkeypatch, fps_of)
    assert res.best.sort_tile_keys == 4096 and res.best.raster_batch == 256


@pytest.mark.parametrize("splats,views,sorts,rasters", [
    (1 << 22, 16, 6, 4),        # every candidate is a form of its own
    ((1 << 22) + 1, 16, 4, 4),  # depths in 16384-key tiles, pairs in 8192 or 16384: 4096 repeats 8192
    (1 << 22, 1, 2, 2),         # one view: the digit width and the walk are what is left
])
def test_candidates_that_run_the_same_launches_are_timed_once(monkeypatch, splats, views, sorts, rasters):
    order = []
    monkeypatch.setattr(at, "measure", lambda sa_, d, b, s, p, w, h, cand, *rest: order.append(cand) or 1.0)
    base = sa.Configuration(max_splat_count=splats, max_views=views)
    at.autotune_staged(sa, None, base, None, None, 64, 48, views, steps=1, splats=splats)
    assert len(order) == sorts + rasters

    def launches(c):
        tiles = sa.sort_tiles(at.configured(base, c), splats, c.max_views)
        return c.radix_bits_per_digit, tiles, c.raster_mode, c.raster_batch if views > 1 else 0
    assert len({launches(c) for c in order[:sorts]}) == sorts
    assert len({launches(c) for c in order[sorts:]}) == rasters


def test_sort_tiles_tells_what_a_batch_runs():
    def tiles(splats, views, **kw):
        return sa.sort_tiles(sa.Configuration(max_splat_count=1 << 25, max_views=16, **kw), splats, views)
    for t in (4096, 8192, 16384):
        assert tiles(1 << 22, 16, sort_tile_keys=t) == (t, t)
        assert tiles((1 << 22) + 1, 2, sort_tile_keys=t) == (16384, max(t, 8192))
        assert tiles(6_000_000, 1, sort_tile_keys=t) == tiles(6_000_000, 1)
    for splats, views in ((1 << 26, 1), (100, 0), (100, 17)):
        with pytest.raises(sa.SplatterError):
            tiles(splats, views)
