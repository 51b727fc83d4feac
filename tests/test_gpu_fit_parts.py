"""How small fits are cut: parts of 1, 2, 4 or 8 tiles of 16 (row, snapshot) pairs over 64 columns, each a workgroup, at the
last count of tiles of each rule and past it. Gradients against the oracle, tolerance as in test_gpu_fit_tiles."""
import ctypes

import numpy as np
import pytest

import wavetool_amd as wt
from test_gpu_fit_tiles import GRAD_TOL, LOSS_TOL, evaluate, problem
from test_gpu_launch_shapes import KernelNode

pytestmark = pytest.mark.gpu


def workgroups(torch, call):
    """Workgroups of the first kernel that `call` puts on a stream, which is captured and not run."""
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    hip = ctypes.CDLL(path)
    stream = torch.cuda.Stream()
    handle, graph, count = ctypes.c_void_p(stream.cuda_stream), ctypes.c_void_p(), ctypes.c_size_t(1)
    assert hip.hipStreamBeginCapture(handle, 1) == 0
    try:
        call(stream)
    finally:
        assert hip.hipStreamEndCapture(handle, ctypes.byref(graph)) == 0
    node, at = ctypes.c_void_p(), KernelNode()
    assert hip.hipGraphGetRootNodes(graph, ctypes.byref(node), ctypes.byref(count)) == 0 and count.value == 1
    assert hip.hipGraphKernelNodeGetParams(node, ctypes.byref(at)) == 0
    hip.hipGraphDestroy(graph)
    return at.grid.x


# tiles: strips of 64 columns times sixteenths of n S pairs
@pytest.mark.parametrize("n,S,W,tiles,per", [(128, 16, 9, 256, 1), (128, 17, 16, 272, 2), (128, 32, 33, 512, 2),
                                             (192, 15, 64, 540, 4), (256, 16, 7, 1024, 4), (256, 17, 65, 1088, 8)])
def test_tiles_of_a_part(torch_cuda, wtctx, n, S, W, tiles, per):
    torch = torch_cuda
    print("[case] fit parts n=%d S=%d W=%d" % (n, S, W), flush=True)
    strips = -(-n // 64)
    assert strips * -(-n * S // 16) == tiles
    params, target = problem(7400 + n + S, n, S, W)
    loss, g, ref_loss, ref = evaluate(torch, wtctx, n, S, W, params, target)
    assert abs(loss - ref_loss) <= LOSS_TOL * ref_loss
    assert np.abs(g - ref).max() <= GRAD_TOL * np.abs(ref).max()
    tt = torch.from_numpy(np.ascontiguousarray(target, dtype=np.float32)).cuda()
    tp = torch.from_numpy(np.ascontiguousarray(params, dtype=np.float32)).cuda()
    fit = wt.Fit(wtctx, [wt.fit_problem(n, S, W, 0.5, 0.0, 0.0, 0.0, 0.25, tt, tp)])
    grad = torch.zeros(5 * W, device="cuda")
    fit.loss_grad(grad)
    torch.cuda.synchronize()
    count = workgroups(torch, lambda s: fit.loss_grad(grad, stream=s))
    fit.close()
    parts = strips * -(-(tiles // strips) // per)
    assert count == (parts if parts < 512 else parts // 2)  # from 512 on two that fit side by side share one
