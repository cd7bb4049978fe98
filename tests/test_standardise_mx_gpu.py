"""Rows standardised and quantised without a gain: the bytes and scales of the kernel with a gain of ones."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("rms", [False, True])
@pytest.mark.parametrize("M,N", [(1, 8), (5, 504), (7, 512), (64, 768), (65, 1032), (257, 1600), (3, 2048), (9, 4096), (2, 8192)])
def test_no_gain_is_a_gain_of_ones(M, N, rms):
    from distributed_neural_networks_amd.ops import _lib
    from distributed_neural_networks_amd.ops.fp8 import kpad_of, mx_scale_bytes
    g = torch.Generator(device=DEV).manual_seed(N)
    rows = torch.zeros(M, N + 16, device=DEV, dtype=torch.bfloat16)
    x = rows[:, 8:8 + N]
    x.copy_(torch.randn(M, N, generator=g, device=DEV) * torch.logspace(-3, 3, M, device=DEV)[:, None] + 1)
    x[:, 3] = -0.0
    if M > 4:  # nothing, a constant, next to nothing in a block, an outlier
        x[0], x[1], x[2, :min(N, 128)], x[3, 7] = 0, 2.5, 1e-38, 3e4
    kp, ones, outs = kpad_of(N), torch.ones(N, device=DEV), []
    for w in (0, ones.data_ptr()):
        q, s = torch.full((M * kp,), 0x55, dtype=torch.uint8, device=DEV), torch.full((mx_scale_bytes(M, kp),), 0x55, dtype=torch.uint8, device=DEV)
        _lib.check(_lib.lib().layernorm_q8_mx(x.data_ptr(), x.stride(0), w, 0, q.data_ptr(), kp, s.data_ptr(), M, N, kp, 1e-5, int(rms),
                                              _lib.stream_ptr()), "layernorm_q8_mx")
        outs.append((q, s))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    assert outs[0][0].view(M, kp)[:, N:].count_nonzero() == 0 and outs[0][0].any() == bool(N > 1)


def test_refusals():
    from distributed_neural_networks_amd.ops import _lib
    t = torch.zeros(4096, dtype=torch.uint8, device=DEV)
    call = lambda ldx, b, at: _lib.lib().layernorm_q8_mx(t.data_ptr() + at, ldx, 0, b, t.data_ptr(), 128, t.data_ptr(), 1, 128, 128, 1e-5,  # noqa: E731
                                                         0, _lib.stream_ptr())
    assert call(128, t.data_ptr(), 0) == -1 and call(132, 0, 0) == -1 and call(128, 0, 2) == -1
