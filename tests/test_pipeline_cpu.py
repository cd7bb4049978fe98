"""Which inputs the colocated pipeline's first stage may read in place (CPU: the rule alone)."""
import torch

from distributed_neural_networks_amd.ops._lib import apart


def test_apart():
    m = torch.zeros(64)
    assert apart(m[:8], m[8:16]) and apart(m[8:16], m[:8])
    for a, b in ((m[:9], m[8:16]), (m, m[8:16]), (m[8:16], m), (m, m), (m, torch.from_dlpack(m))):
        assert not apart(a, b) and not apart(b, a)
    assert apart(m, torch.zeros(64))
