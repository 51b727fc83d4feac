"""GPU test of a batch that mixes every segment shape in its one launch."""
import numpy as np
import pytest

import wavetool_amd as wt
from wavetool_amd import scenes

pytestmark = pytest.mark.gpu

# one vertex either side of each shape's segment (128, 256 and 512 columns) and the smallest side
SIDES = (2, 127, 128, 129, 255, 256, 257, 511, 513)
WAVES = (0, 1, 64, 65, 3)  # both sides of a 64-wave chunk, so that the cost order interleaves the shapes


@pytest.mark.parametrize("texture", ["none", "r32_repeat", "r8_mirror"])
def test_mixed_shapes_equal_plain(torch_cuda, wtctx, texture):
    """Bit for bit what each patch gives alone in the launch shape the batch chose for it."""
    torch = torch_cuda
    print("[case] mixed shapes, %s" % texture, flush=True)
    specs = scenes.batched_patches(seed=21, count=len(SIDES))
    for i, s in enumerate(specs):
        s["N"], s["W"] = SIDES[i], WAVES[i % len(WAVES)]
    patches, waves, V = wt.batch_inputs(specs)
    w = torch.from_numpy(waves).cuda()
    tex = scenes.value_noise(3, 64)
    kw = {}
    if texture == "r32_repeat":
        kw = dict(heightmap=torch.from_numpy(tex).cuda())
    elif texture == "r8_mirror":
        kw = dict(heightmap=torch.from_numpy((tex * 255).astype(np.uint8)).cuda(), hm_format=wt.WT_TEXEL_R8_UNORM,
                  hm_wrap=wt.WT_WRAP_MIRRORED_REPEAT)
    pos = torch.full((V * 3,), float("nan"), device="cuda")
    nrm = torch.full_like(pos, float("nan"))
    batch = wt.Batch(wtctx, patches)
    batch.displace(w, pos, nrm, time_offset=0.25, **kw)
    shapes = set()
    try:
        for i, (s, p) in enumerate(zip(specs, patches)):
            shape = batch.patch_launch_config(i)
            shapes.add(shape)
            wtctx.set_launch_config(*shape)
            n = 3 * s["N"] ** 2
            params = wt.water_params(np.ctypeslib.as_array(p.corners).copy(), s["camera"][4:7], s["N"], s["time"] + 0.25,
                                     0.02, 0.05, 0.0, (0.3, 0.0))
            P, Q = torch.empty(n, device="cuda"), torch.empty(n, device="cuda")
            wtctx.displace(params, w[p.wave_offset:p.wave_offset + p.wave_count], P, Q, wave_count=p.wave_count, **kw)
            o = 3 * p.vertex_offset
            assert torch.equal(P, pos[o:o + n]) and torch.equal(Q, nrm[o:o + n]), (s["N"], s["W"])
    finally:
        wtctx.set_launch_config()
        batch.close()
    assert len(shapes) == 3


@pytest.mark.parametrize("side,waves", [(64, 33), (65, 1), (128, 2), (129, 130), (640, 65), (641, 7), (1100, 3)])
def test_half_segments_equal_whole(torch_cuda, wtctx, side, waves):
    """The plain kernel takes every segment in halves up to 640 workgroups (side 640 here), past that, as the batch at any
    size, only those at the rows' ends whose upper halves are empty: the same bits, tangents included, with a heightmap
    and without."""
    torch = torch_cuda
    print("[case] halves, side %d" % side, flush=True)
    spec = dict(scenes.batched_patches(seed=23, count=1)[0], N=side, W=waves)
    patches, w, V = wt.batch_inputs([spec])
    p = patches[0]
    w = torch.from_numpy(w).cuda()
    params = wt.water_params(np.ctypeslib.as_array(p.corners).copy(), spec["camera"][4:7], side, spec["time"], 0.02, 0.05,
                             0.0, (0.3, 0.0))
    batch = wt.Batch(wtctx, patches)
    try:
        wtctx.set_launch_config(*batch.patch_launch_config(0))
        for kw in ({}, dict(heightmap=torch.from_numpy(scenes.value_noise(3, 64)).cuda())):
            a, b = (torch.full((4, V * 3), float("nan"), device="cuda") for _ in range(2))
            batch.displace(w, *a, **kw)
            wtctx.displace(params, w, *b, **kw)
            assert torch.equal(a, b) and torch.isfinite(a).all()
    finally:
        wtctx.set_launch_config()
        batch.close()
