"""The adjoint kernel at the edges of its tiling: strips of 64 columns, tiles of 16 (row,
snapshot) pairs, chunks of 16 waves (32 per matrix operand), the row-and-time table from
five snapshots on and the class above 64 waves; and over the magnitudes its split operands
have to be scaled to. Gradients against the oracle's FP64 adjoint.

Tolerance: every operand of the contractions is within about 2^-22 of its value, and so is
every product (three operands: 7e-7 of a term). A gradient component is a sum of signed
terms whose absolute sum stays within about 40 times the largest component, so 3e-5 of the
largest component bounds it; the loss is a sum of squares of residuals of the size of the
displacement, within 5e-6."""
import os

import numpy as np
import pytest

import oracle as orc
import wavetool_amd as wt
from wavetool_amd import scenes

pytestmark = pytest.mark.gpu
NTHREADS = min(16, os.cpu_count() or 1)
GRAD_TOL, LOSS_TOL = 3e-5, 5e-6


def evaluate(torch, ctx, n, S, W, params, target, t0=0.0):
    dev = torch.device("cuda")
    x0 = -0.25 * (n - 1)
    tt = torch.from_numpy(np.ascontiguousarray(target, dtype=np.float32)).to(dev)
    tp = torch.from_numpy(np.ascontiguousarray(params, dtype=np.float32)).to(dev)
    fit = wt.Fit(ctx, [wt.fit_problem(n, S, W, 0.5, x0, x0, t0, 0.25, tt, tp)])
    grad = torch.zeros(W * 5, device=dev)
    loss = torch.zeros(1, device=dev)
    fit.loss_grad(grad, loss)
    torch.cuda.synchronize()
    fit.close()
    used = tp.cpu().numpy().astype(np.float64)
    fd = orc.FitData(n, S, 0.5, x0, x0, t0, 0.25, target)
    ref_loss, ref = orc.fit_loss_grad(fd, used, nthreads=NTHREADS)
    return loss.item(), grad.cpu().numpy().astype(np.float64).reshape(W, 5), ref_loss, ref


def problem(seed, n, S, W):
    prob = scenes.fit_problem(seed, n=n, S=S, W_hidden=W, W_fit=W)
    return prob["init"], scenes.fit_target(prob)


SIZES = [(1, 1, 1), (2, 3, 2), (5, 5, 15), (16, 4, 16), (31, 16, 17), (33, 17, 31), (63, 8, 32), (64, 5, 33),
         (65, 7, 48), (65, 4, 49), (127, 2, 64), (128, 32, 5), (129, 1, 16), (64, 6, 65), (66, 9, 96), (40, 12, 128),
         (200, 31, 20)]


@pytest.mark.parametrize("n,S,W", SIZES)
def test_tile_edges(torch_cuda, wtctx, n, S, W):
    print("[case] fit tiles n=%d S=%d W=%d" % (n, S, W), flush=True)
    params, target = problem(7000 + n + S, n, S, W)
    loss, g, ref_loss, ref = evaluate(torch_cuda, wtctx, n, S, W, params, target)
    assert abs(loss - ref_loss) <= LOSS_TOL * ref_loss
    assert np.abs(g - ref).max() <= GRAD_TOL * np.abs(ref).max()


@pytest.mark.parametrize("amplitude,targets,t0", [(1e-7, 1e-7, 0.0), (1e6, 1e6, 0.0), (1e-6, 1.0, 0.0),
                                                  (1.0, 1e4, 0.0), (0.0, 1.0, 0.0), (1.0, 1.0, 5e3)])
def test_magnitudes(torch_cuda, wtctx, amplitude, targets, t0):
    print("[case] fit magnitudes A x %g, target x %g, t0 %g" % (amplitude, targets, t0), flush=True)
    params, target = problem(31, 70, 6, 12)
    params = params.copy()
    params[:, 0] *= amplitude
    loss, g, ref_loss, ref = evaluate(torch_cuda, wtctx, 70, 6, 12, params, target * np.float32(targets), t0)
    assert abs(loss - ref_loss) <= LOSS_TOL * ref_loss
    for k in range(5):  # the parameters' derivatives differ by the amplitude: each against its own largest
        assert np.abs(g[:, k] - ref[:, k]).max() <= GRAD_TOL * np.abs(ref[:, k]).max(), k


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_non_finite_target_reaches_loss_and_gradient(torch_cuda, wtctx, bad):
    params, target = problem(32, 70, 6, 12)
    target = target.copy().reshape(6, -1, 3)
    target[3, 70 * 41 + 67, 1] = bad
    loss, g, _, _ = evaluate(torch_cuda, wtctx, 70, 6, 12, params, target)
    assert not np.isfinite(loss)
    # dQ sums the x and z residuals alone; every other derivative takes the y residual
    assert not np.isfinite(g[:, [0, 1, 2, 4]]).any()


# (n, S) whose 16-pair tiles are cut into parts of 1, 2, 4 and 8 tiles, at the last size of each rule and the next
PARTS = [(64, 64, 16), (128, 32, 16), (129, 32, 20), (181, 20, 33), (182, 20, 100), (256, 16, 64), (257, 17, 8),
         (360, 16, 12), (420, 24, 5)]


@pytest.mark.parametrize("n,S,W", [(n, min(S, 32), W) for n, S, W in PARTS])
def test_parts_of_a_small_problem(torch_cuda, wtctx, n, S, W):
    """Against the oracle, and bit for bit the same when the problem's parts share workgroups side by side in a batch."""
    torch = torch_cuda
    print("[case] fit parts n=%d S=%d W=%d" % (n, S, W), flush=True)
    params, target = problem(7100 + n + S, n, S, W)
    loss, g, ref_loss, ref = evaluate(torch, wtctx, n, S, W, params, target)
    assert abs(loss - ref_loss) <= LOSS_TOL * ref_loss
    assert np.abs(g - ref).max() <= GRAD_TOL * np.abs(ref).max()
    dev = torch.device("cuda")
    x0 = -0.25 * (n - 1)
    tt = torch.from_numpy(np.ascontiguousarray(target, dtype=np.float32)).to(dev)
    tp = torch.from_numpy(np.ascontiguousarray(params, dtype=np.float32)).to(dev)
    for count in (3, 40):
        fit = wt.Fit(wtctx, [wt.fit_problem(n, S, W, 0.5, x0, x0, 0.0, 0.25, tt, tp)] * count)
        grad, losses = torch.zeros(count * W * 5, device=dev), torch.zeros(count, device=dev)
        fit.loss_grad(grad, losses)
        torch.cuda.synchronize()
        fit.close()
        assert torch.equal(grad.cpu(), torch.from_numpy(g.astype(np.float32)).reshape(-1).repeat(count)), count
        assert (losses == loss).all(), count
