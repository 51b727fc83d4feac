"""Fits of few waves, which a kernel of their own takes: up to 4 waves, and up to 6 in small problems (512 tiles of 16
(row, snapshot) pairs). Gradients against the oracle's FP64 adjoint, and the same bits beside problems of more waves, whose
kernel then holds them.

Tolerance: that of test_gpu_fit_tiles. A term is a residual times a cosine or sine formed from two factors within 1e-7 of
their value, each operation rounded in FP32 (6e-8): within 7e-7 as the matrix products there."""
import ctypes

import numpy as np
import pytest

import wavetool_amd as wt
from test_gpu_fit_tiles import GRAD_TOL, LOSS_TOL, evaluate, problem
from test_gpu_launch_shapes import KernelNode

pytestmark = pytest.mark.gpu


def kernels(torch, call):
    """Names of the kernels that `call` puts on a stream, which is captured and not run."""
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    hip = ctypes.CDLL(path)
    hip.hipKernelNameRefByPtr.restype = ctypes.c_char_p
    hip.hipKernelNameRefByPtr.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    stream = torch.cuda.Stream()
    handle, graph, count = ctypes.c_void_p(stream.cuda_stream), ctypes.c_void_p(), ctypes.c_size_t()
    assert hip.hipStreamBeginCapture(handle, 1) == 0
    try:
        call(stream)
    finally:
        assert hip.hipStreamEndCapture(handle, ctypes.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(count)) == 0
    nodes = (ctypes.c_void_p * count.value)()
    assert hip.hipGraphGetNodes(graph, nodes, ctypes.byref(count)) == 0
    names = []
    for node in nodes:
        at, kind = KernelNode(), ctypes.c_int()
        assert hip.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)) == 0
        if kind.value == 0:  # a kernel
            assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(at)) == 0
            names.append(hip.hipKernelNameRefByPtr(at.func, handle).decode())
    hip.hipGraphDestroy(graph)
    return names


def make(torch, sizes):
    """Problems of (n, S, W) with their tensors, and their gradient's places."""
    dev, out = torch.device("cuda"), []
    for i, (n, S, W) in enumerate(sizes):
        params, target = problem(7300 + i, n, S, W)
        tt = torch.from_numpy(np.ascontiguousarray(target, dtype=np.float32)).to(dev)
        tp = torch.from_numpy(np.ascontiguousarray(params, dtype=np.float32)).to(dev)
        x0 = -0.25 * (n - 1)
        out.append((wt.fit_problem(n, S, W, 0.5, x0, x0, 0.0, 0.25, tt, tp), tp, tt))
    return out


# every wave count, columns past the grid and past a strip, pairs past the last tile of 4 and of 8, one snapshot and 32, the
# last size of the small problems and the next (512 and 514 tiles), several rounds of tiles in a part
SIZES = [(1, 1, 1), (2, 3, 2), (5, 5, 3), (16, 4, 4), (63, 1, 5), (64, 32, 6), (65, 7, 1), (127, 2, 2), (200, 13, 3),
         (256, 8, 4), (256, 8, 6), (257, 6, 4), (257, 7, 2), (320, 31, 4), (513, 32, 1), (700, 32, 3)]


@pytest.mark.parametrize("n,S,W", SIZES)
def test_few_waves(torch_cuda, wtctx, n, S, W):
    print("[case] few waves n=%d S=%d W=%d" % (n, S, W), flush=True)
    params, target = problem(7200 + n + S, n, S, W)
    loss, g, ref_loss, ref = evaluate(torch_cuda, wtctx, n, S, W, params, target, t0=3.0)
    assert abs(loss - ref_loss) <= LOSS_TOL * ref_loss
    assert np.abs(g - ref).max() <= GRAD_TOL * np.abs(ref).max()


@pytest.mark.parametrize("sizes,kernel", [([(64, 4, 1)], "few"), ([(64, 4, 6)], "few"), ([(64, 4, 7)], "ILi4ELi8ELb1ELb0E"),
                                          ([(512, 8, 4)], "few"), ([(512, 8, 5)], "ILi4ELi8ELb1ELb0E"),
                                          ([(64, 4, 1), (64, 4, 7)], "ILi4ELi8ELb1ELb1E")])
def test_kernel_by_waves_and_size(torch_cuda, wtctx, sizes, kernel):
    """The matrix contraction takes 1.1 to 1.9 times as long for few waves, and a second launch beside another class of
    problems up to 1.5 times as long as one for both."""
    torch = torch_cuda
    made = make(torch, sizes)
    fit = wt.Fit(wtctx, [m[0] for m in made])
    grad, losses = torch.zeros(sum(5 * s[2] for s in sizes), device="cuda"), torch.zeros(len(sizes), device="cuda")
    fit.loss_grad(grad, losses)
    torch.cuda.synchronize()
    names = kernels(torch, lambda s: fit.loss_grad(grad, losses, stream=s))
    fit.close()
    assert len(names) == 2 and kernel in names[0] and "adjoint" in names[0], names


@pytest.mark.parametrize("others", [[(100, 9, 3)] * 3, [(70, 4, 20)], [(70, 4, 20), (60, 6, 90)], [(40, 3, 100)]])
def test_batch_repeats_the_bits(torch_cuda, wtctx, others):
    """Problems of few waves alone, with one another, and beside problems of the other classes; gradients and Adam steps."""
    torch = torch_cuda
    sizes = [(64, 4, 1), (256, 8, 6), (257, 7, 2), (300, 16, 4), (33, 5, 5), (512, 16, 3)]

    def run(which):
        made = make(torch, which)
        fit = wt.Fit(wtctx, [m[0] for m in made])
        grad, losses = torch.zeros(sum(5 * s[2] for s in which), device="cuda"), torch.zeros(len(which), device="cuda")
        fit.loss_grad(grad, losses)
        first = losses.clone()
        fit.iterate(3, losses=losses)
        torch.cuda.synchronize()
        fit.close()
        return grad, first, losses, torch.cat([m[1].reshape(-1) for m in made])

    together = run(sizes + others)
    at = 0
    for i, size in enumerate(sizes):
        made = make(torch, sizes[:i + 1])[i]  # the same inputs as in the batch
        fit = wt.Fit(wtctx, [made[0]])
        grad, loss = torch.zeros(5 * size[2], device="cuda"), torch.zeros(1, device="cuda")
        fit.loss_grad(grad, loss)
        assert torch.equal(grad, together[0][at:at + 5 * size[2]]) and loss.item() == together[1][i].item(), size
        fit.iterate(3, losses=loss)
        torch.cuda.synchronize()
        fit.close()
        assert torch.equal(made[1].reshape(-1), together[3][at:at + 5 * size[2]]) and loss.item() == together[2][i].item(), size
        at += 5 * size[2]


def test_non_finite_target_of_few_waves(torch_cuda, wtctx):
    params, target = problem(32, 70, 6, 2)
    target = target.copy().reshape(6, -1, 3)
    target[3, 70 * 41 + 67, 1] = np.nan
    loss, g, _, _ = evaluate(torch_cuda, wtctx, 70, 6, 2, params, target)
    assert not np.isfinite(loss) and not np.isfinite(g[:, [0, 1, 2, 4]]).any()
