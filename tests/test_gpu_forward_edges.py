"""GPU parity of the forward kernel where the grid ends around half a segment: the second
wavefront of a pair then has no column to finish, or one."""
import pytest

from wavetool_amd import scenes
from helpers import NRM_TOL, POS_TOL
from test_gpu_forward import check_parity, scene_setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(2, 8, 64), (2, 8, 32), (2, 4, 16), (2, 16, 8)])
@pytest.mark.parametrize("halves,over", [(1, -1), (1, 0), (1, 1), (3, 0), (3, 1)])
def test_grid_ends_at_half_a_segment(torch_cuda, wtctx, shape, halves, over):
    """Every vertex is written (the buffers start as NaN) and as close to the oracle as on whole segments."""
    split, steps, lanes = shape
    cfg, corners, waves, cam_pos, t, texels = scene_setup(scenes.scene_1024_w64_heightmap())
    cfg = dict(cfg, N=halves * steps * lanes // 2 + over)
    print("[case] %s, side %d" % (shape, cfg["N"]), flush=True)
    wtctx.set_launch_config(*shape)
    try:
        res = check_parity(torch_cuda, wtctx, cfg, corners, waves[:13], cam_pos, t, texels, with_tb=True)
    finally:
        wtctx.set_launch_config()
    assert res["pos_max"] <= POS_TOL and res["nrm_max"] <= NRM_TOL, res
