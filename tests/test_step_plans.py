"""What a step's plans are made of on the host and how it gets to the device."""
import numpy as np
import pytest
import torch

from scalellm_amd import kernels
from scalellm_amd import latent_kernels as lk
from scalellm_amd.kernels import SlmError

ARRAYS = [np.arange(5, dtype=np.int32), np.arange(42, dtype=np.int32).reshape(6, 7), np.zeros((0, 3), dtype=np.int32), np.array([-7], dtype=np.int32)]


def test_arrays_on_the_host():
    got = lk.arrays_to_device(ARRAYS, "cpu")
    assert all(np.array_equal(t.numpy(), a) and t.shape == a.shape for t, a in zip(got, ARRAYS))


@pytest.mark.gpu
def test_arrays_on_the_device():
    """Many plans one after the other, behind work that keeps the stream busy: a host buffer is not used again before its copy is done."""
    x = torch.randn(4096, 4096, device="cuda")
    kept = []
    for i in range(40):
        x = torch.tanh(x @ x)
        kept.append(lk.arrays_to_device([a + i for a in ARRAYS], x.device))
    for i, got in enumerate(kept):
        for t, a in zip(got, ARRAYS):
            assert t.is_cuda and t.is_contiguous() and t.dtype == torch.int32 and np.array_equal(t.cpu().numpy(), a + i)
    with pytest.raises(SlmError):
        lk.arrays_to_device([np.arange(3)], "cuda")
    graph, y = torch.cuda.CUDAGraph(), torch.zeros(3, device="cuda")
    with torch.cuda.graph(graph):
        y.add_(1.0)
        with pytest.raises(SlmError):
            lk.arrays_to_device(ARRAYS, "cuda")


@pytest.mark.gpu
def test_handle_of_the_current_stream():
    assert kernels.current_stream_handle() == torch.cuda.current_stream().cuda_stream
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert kernels.current_stream_handle() == side.cuda_stream
