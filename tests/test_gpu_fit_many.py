"""Batches whose launches would pass the 2^32 threads of one launch."""
import numpy as np
import pytest

import wavetool_amd as wt

pytestmark = pytest.mark.gpu


def test_more_reduction_blocks_than_one_launch_holds(torch_cuda, wtctx):
    """2^22 blocks of 1024 threads and some: a block for each problem of up to 3 waves."""
    torch = torch_cuda
    count = (1 << 22) + 9
    target = torch.tensor([0.3, -0.2, 0.1], device="cuda")
    params = torch.tensor([[0.5, 7.0, 0.4, 0.6, 0.2]], device="cuda")
    p = wt.fit_problem(1, 1, 1, 0.5, 0.0, 0.0, 0.0, 0.25, target, params)
    grad, losses = torch.zeros(5 * count, device="cuda"), torch.zeros(count, device="cuda")
    print("[case] %d problems" % count, flush=True)
    many = wt.Fit(wtctx, [p] * count)
    many.loss_grad(grad, losses)
    torch.cuda.synchronize()
    many.close()
    one = wt.Fit(wtctx, [p])
    want, loss = torch.zeros(5, device="cuda"), torch.zeros(1, device="cuda")
    one.loss_grad(want, loss)
    torch.cuda.synchronize()
    one.close()
    assert torch.isfinite(want).all() and loss.item() > 0
    assert (losses == loss).all() and (grad.view(-1, 5) == want).all()
