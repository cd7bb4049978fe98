"""Scratch rows of the fp32 head: what is taken, what is replaced, what is refused (CPU)."""
import pytest
import torch

from distributed_neural_networks_amd.ops import cifar as cops

K3 = 3 * 4096


def test_fc1_scratch():
    cpu = torch.device("cpu")
    own = torch.empty((3, K3), dtype=torch.bfloat16)
    assert cops._fc1_scratch(own, 3, cpu) is own and cops._fc1_scratch(own, 2, cpu) is own
    for other in (None, own[:, :4096], torch.empty((3, 2 * K3), dtype=torch.bfloat16)[:, :K3], own[:2]):
        got = cops._fc1_scratch(other, 3, cpu)
        assert got is not other and got.is_contiguous() and tuple(got.shape) == (3, K3) and got.dtype == torch.bfloat16
    for dt in (torch.uint8, torch.float16, torch.float32):  # the few-row head keeps 16 KB of partial sums a row in it
        with pytest.raises(TypeError):
            cops._fc1_scratch(torch.empty((3, K3), dtype=dt), 3, cpu)
