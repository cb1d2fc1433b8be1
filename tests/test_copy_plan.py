"""BlockCopyPlan's host checks, in the order the copies were always refused: lengths, repeated
destinations, a destination that is also a source, ids outside the pool. On the CPU: the pools
are never touched (the GPU check of a pool is stood in for), no case reaches the upload."""
import pytest
import torch

from tinybatch_amd import _lib, ops


@pytest.fixture
def pools(monkeypatch):
    monkeypatch.setattr(_lib, "require_gpu_tensor", lambda name, t: None)
    return [torch.zeros(8, 2, 1, 4, 16) for _ in range(3)]


@pytest.mark.parametrize("src,dst,error", [
    ([0, 1], [2], ValueError), ([0, 1], [2, 2], ValueError), ([0, 1], [1, 2], ValueError),
    ([0, 8], [2, 3], IndexError), ([0, 1], [2, -1], IndexError), ([0, 1], [8, 8], ValueError),
    ([9, 1], [9, 2], ValueError)])
def test_refused_rounds(pools, src, dst, error):
    with pytest.raises(error):
        ops.BlockCopyPlan(pools, src, dst)


def test_refused_pools(pools):
    with pytest.raises(ValueError):
        ops.BlockCopyPlan([], [0], [1])
    with pytest.raises(ValueError):
        ops.BlockCopyPlan(pools + [torch.zeros(9, 2, 1, 4, 16)], [0], [1])
    with pytest.raises(ValueError):                              # not contiguous
        ops.BlockCopyPlan(pools + [torch.zeros(8, 2, 1, 16, 4).transpose(3, 4)], [0], [1])
