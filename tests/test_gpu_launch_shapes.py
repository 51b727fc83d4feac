"""Which forward kernel a launch shape runs, read from the captured node: a shape that was asked for (or tuned) runs as it
is, and only the library's own choice takes segments in halves; both give the same bits."""
import ctypes

import numpy as np
import pytest

import wavetool_amd as wt
from wavetool_amd import scenes

pytestmark = pytest.mark.gpu

MAPS = {"none": None, "r32_repeat": (wt.WT_TEXEL_R32F, wt.WT_WRAP_REPEAT), "r32_mirror": (wt.WT_TEXEL_R32F, wt.WT_WRAP_MIRRORED_REPEAT),
        "r8_repeat": (wt.WT_TEXEL_R8_UNORM, wt.WT_WRAP_REPEAT), "r8_mirror": (wt.WT_TEXEL_R8_UNORM, wt.WT_WRAP_MIRRORED_REPEAT)}


class Dim3(ctypes.Structure):
    _fields_ = [("x", ctypes.c_uint32), ("y", ctypes.c_uint32), ("z", ctypes.c_uint32)]


class KernelNode(ctypes.Structure):  # hipKernelNodeParams
    _fields_ = [("block", Dim3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", Dim3),
                ("args", ctypes.c_void_p), ("lds", ctypes.c_uint32)]


def launched(torch, call):
    """(kernel name, workgroups) of the one kernel that `call` puts on a stream, which is captured and not run."""
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    hip = ctypes.CDLL(path)
    hip.hipKernelNameRefByPtr.restype = ctypes.c_char_p
    hip.hipKernelNameRefByPtr.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    stream = torch.cuda.Stream()
    handle, graph = ctypes.c_void_p(stream.cuda_stream), ctypes.c_void_p()
    assert hip.hipStreamBeginCapture(handle, 1) == 0
    try:
        call(stream)
    finally:
        assert hip.hipStreamEndCapture(handle, ctypes.byref(graph)) == 0
    count = ctypes.c_size_t()
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(count)) == 0 and count.value == 1
    node = ctypes.c_void_p()
    assert hip.hipGraphGetNodes(graph, ctypes.byref(node), ctypes.byref(count)) == 0
    at = KernelNode()
    assert hip.hipGraphKernelNodeGetParams(node, ctypes.byref(at)) == 0
    name = hip.hipKernelNameRefByPtr(at.func, handle).decode()
    hip.hipGraphDestroy(graph)
    return name, at.grid.x


def scene(torch, side, waves, mode="none"):
    spec = dict(scenes.batched_patches(seed=29, count=1)[0], N=side, W=waves)
    patches, w, _ = wt.batch_inputs([spec])
    params = wt.water_params(np.ctypeslib.as_array(patches[0].corners).copy(), spec["camera"][4:7], side, spec["time"], 0.02,
                             0.05, 0.0, (0.3, 0.0))
    kw = {}
    if MAPS[mode]:
        tex = scenes.value_noise(3, 64)
        tex = (tex * 255).astype(np.uint8) if mode.startswith("r8") else tex
        kw = dict(heightmap=torch.from_numpy(tex).cuda(), hm_format=MAPS[mode][0], hm_wrap=MAPS[mode][1])
    return params, torch.from_numpy(w).cuda(), kw


def groups(side, lanes, steps):
    """Workgroups of whole segments, two a workgroup."""
    segments = -(-side // (lanes * steps)) * -(-side // (64 // lanes))
    return -(-segments // 2)


# side, lanes per row: under 640 workgroups, and past it with rows that end in the lower half of a segment
@pytest.mark.parametrize("side,lanes", [(100, 16), (200, 32), (300, 64), (620, 64), (700, 64), (1025, 64), (890, 32), (1040, 16)])
def test_a_requested_shape_runs(torch_cuda, wtctx, side, lanes):
    torch = torch_cuda
    params, w, kw = scene(torch, side, 5)
    out = [torch.empty(3 * side * side, device="cuda") for _ in range(2)]
    wtctx.displace(params, w, *out)  # loads the code before the capture
    torch.cuda.synchronize()
    wtctx.set_launch_config(2, 8, lanes)
    try:
        name, count = launched(torch, lambda s: wtctx.displace(params, w, *out, stream=s))
    finally:
        wtctx.set_launch_config()
    print("[case] side %d, lanes %d: %s, %d workgroups" % (side, lanes, name, count), flush=True)
    assert "water_forward_kernelILi8ELi%dELi2E" % lanes in name and name.split("_kernel")[1].startswith("ILi8E")
    assert "Lb1E" not in name and count == groups(side, lanes, 8)


# the last side of each rule and the next: 640 workgroups of whole segments, rows of 512 columns and half a segment
@pytest.mark.parametrize("mode", list(MAPS))
@pytest.mark.parametrize("side,waves,kernel", [(100, 3, "Lb1E"), (256, 65, "Lb1E"), (257, 1, "Lb1E"), (640, 9, "Lb1E"),
                                               (641, 32, "tail"), (700, 66, "tail"), (768, 33, "tail"), (769, 2, "whole"),
                                               (1024, 3, "whole"), (1025, 32, "tail"), (1281, 2, "whole")])
def test_own_choice_equals_whole_segments(torch_cuda, wtctx, side, waves, kernel, mode):
    """Tangents and bitangents included."""
    torch = torch_cuda
    params, w, kw = scene(torch, side, waves, mode)
    a, b = (torch.full((4, 3 * side * side), float("nan"), device="cuda") for _ in range(2))
    wtctx.displace(params, w, *a, **kw)
    torch.cuda.synchronize()
    shape = wtctx.get_launch_config(side, waves)
    name, _ = launched(torch, lambda s: wtctx.displace(params, w, *a, stream=s, **kw))
    print("[case] side %d, %s: %s" % (side, mode, name), flush=True)
    assert ("tail_kernel" in name) == (kernel == "tail") and ("Lb1E" in name) == (kernel == "Lb1E")
    wtctx.set_launch_config(**shape)
    try:
        wtctx.displace(params, w, *b, **kw)
    finally:
        wtctx.set_launch_config()
    assert torch.isfinite(a).all() and torch.equal(a, b)


@pytest.mark.parametrize("side,waves,mode,tail", [(641, 31, "r32_repeat", False), (768, 4, "r8_mirror", False),
                                                  (768, 32, "r32_repeat", True), (1025, 1, "r32_repeat", True),
                                                  (641, 1, "none", True), (768, 31, "none", True)])
def test_few_waves_end_rows_in_whole_segments(torch_cuda, wtctx, side, waves, mode, tail):
    """Where every workgroup of whole segments runs at once, half segments at the rows' ends pay from 32 waves on, or
    without a map."""
    torch = torch_cuda
    params, w, kw = scene(torch, side, waves, mode)
    out = [torch.empty(3 * side * side, device="cuda") for _ in range(2)]
    wtctx.displace(params, w, *out, **kw)
    torch.cuda.synchronize()
    name, _ = launched(torch, lambda s: wtctx.displace(params, w, *out, stream=s, **kw))
    assert ("tail_kernel" in name) == tail, name


@pytest.mark.parametrize("side,waves,mode,outputs,tail", [
    (1025, 1, "none", 2, True), (1537, 7, "none", 2, False), (1537, 8, "none", 2, True), (1600, 1, "none", 2, True),
    (1025, 15, "none", 3, False), (1025, 16, "none", 3, True), (1280, 11, "none", 3, False), (1280, 12, "none", 3, True),
    (1025, 31, "none", 4, False), (1280, 23, "none", 4, False), (1280, 24, "none", 4, True),
    (1025, 2, "r32_repeat", 4, True), (2049, 23, "r8_mirror", 4, False), (2049, 24, "r8_mirror", 4, True),
    (2049, 2, "r32_mirror", 3, True), (2304, 2, "r8_repeat", 4, True)])
def test_rows_bound_by_their_stores_end_in_whole_segments(torch_cuda, wtctx, side, waves, mode, outputs, tail):
    torch = torch_cuda
    params, w, kw = scene(torch, side, waves, mode)
    out = [torch.empty(3 * side * side, device="cuda") for _ in range(outputs)]
    wtctx.displace(params, w, *out, **kw)
    torch.cuda.synchronize()
    name, _ = launched(torch, lambda s: wtctx.displace(params, w, *out, stream=s, **kw))
    assert ("tail_kernel" in name) == tail, name


def test_tuned_shapes_run_as_they_were_timed(torch_cuda, tmp_path):
    """A table says whether a size keeps the library's choice; tables of six columns do where they hold its shape."""
    torch = torch_cuda
    params, w, _ = scene(torch, 300, 5)
    out = [torch.empty(3 * 300 * 300, device="cuda") for _ in range(2)]
    ctx = wt.Context()
    ctx.displace(params, w, *out)
    torch.cuda.synchronize()
    for line, halves in (("9 3 2 8 64 64 1", True), ("9 3 2 8 64 64 0", False), ("9 3 2 8 64 64", True), ("9 3 2 8 32 64 1", False)):
        path = tmp_path / "tune.txt"
        path.write_text(line + "\n")
        ctx.autotune_load(path)
        name, _ = launched(torch, lambda s: ctx.displace(params, w, *out, stream=s))
        assert ("Lb1E" in name) == halves, (line, name)
        ctx.autotune_save(path)
        again = wt.Context()
        again.autotune_load(path)
        assert again.get_launch_config(300, 5) == ctx.get_launch_config(300, 5)
        name, _ = launched(torch, lambda s: again.displace(params, w, *out, stream=s))
        assert ("Lb1E" in name) == halves, (line, name)
        again.close()
    ctx.close()
