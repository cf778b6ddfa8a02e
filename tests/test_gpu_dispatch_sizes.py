"""The sizes at which a launch changes form, against the oracle: how the
raster deals screen tiles to the XCDs, how many blocks project a cull tile,
which radix-sort tile one view takes."""
import numpy as np
import pytest

import oracle_bind as ob
import splatter_amd as sa
from gpu_common import Case, config, device, image_diff, normwise_rel, say
from splatter_amd.synth import Workload, sphere_pose

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
