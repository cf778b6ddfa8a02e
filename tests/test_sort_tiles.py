"""The radix-sort tiles that one view takes (host logic, no device): the lines
at which one tile's sort is as fast as the next one's, as measured on MI355X."""
import pytest

import splatter_amd as sa


def tiles(splats, views=1, **kw):
    kw.setdefault("max_splat_count", 1 << 23)
    return sa.sort_tiles(sa.Configuration(**kw), splats, views)


# up to this many splats, depths sort in tiles of so many keys; a 1024-key tile
# of 10-bit digits has as many digits as keys, and no size is faster so
@pytest.mark.parametrize("bits,lines", [(8, [(7 << 14, 1024), (1 << 20, 4096), (1 << 21, 8192), (1 << 23, 16384)]),
                                        (10, [(1 << 17, 4096), (1 << 21, 8192), (1 << 23, 16384)])])
@pytest.mark.parametrize("sort_tile_keys", [4096, 16384])
def test_depth_tile_of_one_view(bits, lines, sort_tile_keys):
    first = 0
    for last, keys in lines:
        for n in (first, last):
            assert tiles(n, radix_bits_per_digit=bits, sort_tile_keys=sort_tile_keys)[0] == keys
        first = last + 1
