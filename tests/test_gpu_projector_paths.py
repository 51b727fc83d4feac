"""GPU test of the device projector's two kernels: a wavefront per camera for small
counts, a thread per camera for large ones. Both form every value by the same
operations, so they agree bit for bit."""
import numpy as np
import pytest

import wavetool_amd as wt
from wavetool_amd import scenes
from test_gpu_projector import camera_set

pytestmark = pytest.mark.gpu

MANY = 1 << 14  # past the bound of the wavefront kernel


def edge_cameras():
    """The camera set of the host comparison, with every pitch and height that picks a branch: straight up and down,
    the horizon from both sides, on y = 0 (no aim point), on and at the slab's planes, and a slab of no height."""
    cams, amps = camera_set()
    for h in (-5.0, -2.0, 0.0, 1e-3, 2.0, 3.0, 40.0):
        for pitch in (-90.0, -89.0, -30.0, -0.05, 0.0, 0.05, 30.0, 89.0):
            cams.append(scenes.camera_tuple(height=h, pitch_deg=pitch, yaw_deg=17.0 * pitch))
            amps.append(2.0 if h else 0.0)
    return cams, amps


@pytest.mark.parametrize("count", [1, 2, 63, 257])
def test_small_counts_equal_large(torch_cuda, wtctx, count):
    torch = torch_cuda
    cams, amps = edge_cameras()
    n = len(cams)
    rows, a = wt.camera_rows(cams), np.asarray(amps, np.float32)
    many = np.arange(MANY) % n
    print("[case] projector kernels, %d cameras in calls of %d" % (n, count), flush=True)

    def run(idx):
        c = torch.from_numpy(np.ascontiguousarray(rows[idx])).cuda()
        out = torch.zeros((len(idx), 4, 4), dtype=torch.float64, device="cuda")
        st = torch.full((len(idx),), -1, dtype=torch.int32, device="cuda")
        wt.projector_corners_batched(wtctx, c, torch.from_numpy(a[idx].copy()).cuda(), out, st)
        return out.cpu().numpy(), st.cpu().numpy()

    want, want_st = run(many)
    assert set(want_st) >= {wt.WT_OK, wt.WT_ERR_NO_INTERSECTION, wt.WT_ERR_INVALID_ARG}
    for lo in range(0, n, count) if count > 2 else range(n - 70, n, count):
        idx = np.arange(lo, min(lo + count, n))
        got, st = run(idx)
        assert np.array_equal(st, want_st[idx]), lo
        ok = st == wt.WT_OK
        assert np.array_equal(got[ok].view(np.int64), want[idx][ok].view(np.int64)), lo
        assert np.isnan(got[~ok]).all()
