"""What the Python wrappers hand to the C ABI: the current stream of the calling thread,
and matrices as column-major floats."""
import threading

import numpy as np
import pytest

import wavetool_amd as wt


@pytest.mark.gpu
def test_current_stream_is_followed(torch_cuda):
    """None stands for the calling thread's current stream, inside and outside a stream context and after a change;
    a thread's stream context does not reach another thread."""
    torch = torch_cuda
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    assert wt._stream(None) == torch.cuda.current_stream().cuda_stream == torch.cuda.default_stream().cuda_stream
    seen = []
    with torch.cuda.stream(a):
        assert wt._stream(None) == a.cuda_stream
        assert wt._stream(b) == b.cuda_stream
        t = threading.Thread(target=lambda: seen.append(wt._stream(None)))
        t.start()
        t.join()
        with torch.cuda.stream(b):
            assert wt._stream(None) == b.cuda_stream
        assert wt._stream(None) == a.cuda_stream
    assert seen == [torch.cuda.default_stream().cuda_stream]
    assert wt._stream(None) == torch.cuda.default_stream().cuda_stream


@pytest.mark.parametrize("make", [np.asarray, np.asfortranarray, lambda m: m.astype(np.float32), lambda m: m.tolist(),
                                  lambda m: m.T.copy().reshape(-1), lambda m: np.stack([m, m])[1][:, ::-1][:, ::-1]])
def test_matrices_are_column_major(make):
    m = np.random.default_rng(3).normal(size=(4, 4)) * np.logspace(-30, 30, 16).reshape(4, 4)
    want = [np.float32(v) for v in np.asarray(make(m), dtype=np.float64).reshape(-1)]
    if np.ndim(make(m)) == 2:
        want = [np.float32(m[k % 4][k // 4]) for k in range(16)]
    assert [np.float32(v) for v in wt._column_major(make(m))] == want


def test_too_many_matrix_elements_are_refused():
    with pytest.raises(IndexError):
        wt._column_major(np.zeros((5, 5)))
