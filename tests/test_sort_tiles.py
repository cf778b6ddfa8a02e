"""The radix-sort tiles that one view takes (host logic, no device): the lines
at which one tile's sort is as fast as the next one's, as measured on MI355X."""
import pytest

import splatter_amd as sa


def tiles(splats, views=1, **kw):
    kw.setdefault("max_splat_count", 1 << 23)
    return sa.sort_tiles(sa.Configuration(**kw), splats, views)


# up to this many splats, depths sort in tiles of so many keys; a 1024-key tile
# of 10-bit digits has as many digits as keys, and no size is faster so (0: by
# how many are visible)
@pytest.mark.parametrize("bits,lines", [(8, [(7 << 14, 1024), (1 << 20, 4096), (1 << 21, 8192), (1 << 23, 0)]),
                                        (10, [(1 << 17, 4096), (1 << 21, 8192), (1 << 23, 0)])])
@pytest.mark.parametrize("sort_tile_keys", [4096, 16384])
def test_depth_tile_of_one_view(bits, lines, sort_tile_keys):
    first = 0
    for last, keys in lines:
        for n in (first, last):
            assert tiles(n, radix_bits_per_digit=bits, sort_tile_keys=sort_tile_keys)[0] == keys
        first = last + 1


# the splats' share of the pair capacity bounds how many pairs they can have:
# with room for eight a splat, 1024-key tiles up to 2^15 splats, 4096-key ones
# up to 2^19, then by the number of pairs (0), then 16384
@pytest.mark.parametrize("capacity", [1 << 15, 1 << 17, 1 << 23])
def test_pair_tile_of_one_view(capacity):
    lines = [(1 << 15, 1024 if capacity <= 1 << 17 else 4096), (1 << 19, 4096), (1 << 21, 0), (1 << 23, 16384)]
    first = 0
    for last, keys in lines:
        for n in (first, last):
            if n <= capacity:
                assert tiles(n, max_splat_count=capacity, tile_pairs_per_splat=8)[1] == keys
        first = last + 1


@pytest.mark.parametrize("splats,per_splat,keys", [
    (1 << 15, 8, 1024), (1 << 15, 9, 4096),           # room for 2^18 pairs and for more
    (1 << 15, 128, 4096), (1 << 15, 129, 0),          # 2^22 and more
    (100_000, 200, 0), (1 << 19, 8, 4096), (1 << 19, 9, 0),
    (1_500_000, 40, 0), ((1 << 21) + 1, 40, 16384),
])
def test_pair_tile_goes_by_what_the_capacity_holds(splats, per_splat, keys):
    assert tiles(splats, max_splat_count=splats, tile_pairs_per_splat=per_splat)[1] == keys
