"""Uploads that the host does not wait for (utils/pinned.py)."""
import numpy as np
import pytest
import torch

from llm_weighted_consensus_amd.utils import pinned


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_arrays_of_several_types_and_sizes(device):
    arrays = [np.arange(7, dtype=np.int32), np.zeros(0, np.int64), np.arange(12).reshape(3, 4)[:, ::2], np.array([1.5], np.float32),
              np.arange(pinned.MOST_BYTES // 4, dtype=np.int32)]
    for n in (4, 5):   # (with the last, more than goes through pinned memory)
        got = pinned.to_device(device, *arrays[:n])
        for t, a in zip(got, arrays):
            assert t.device.type == device and t.shape == a.shape and np.array_equal(t.cpu().numpy(), a)


@pytest.mark.gpu
def test_host_arrays_may_change_behind_a_busy_stream(gpu):
    """Every upload holds what its array held when it was made, also where many are on their way."""
    x, got = torch.randn(4096, 4096, device=gpu).to(torch.bfloat16), []
    for i in range(24):
        for _ in range(4):
            x = (x @ x).clamp_(-1, 1)
        a = np.full(1000 << i % 8, i, np.int32)
        got.append(pinned.to_device(gpu, a)[0])
        a[:] = -1
    for i, t in enumerate(got):
        assert (t == i).all()
