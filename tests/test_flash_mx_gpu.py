"""Prefill attention whose rows leave as MX e4m3: the bytes and scales of the
quantiser run over the plain kernel's rows."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,T,H,Hkv,pos0", [(1, 256, 25, 25, 0), (3, 129, 25, 25, 0), (2, 127, 12, 12, 70),
                                            (2, 200, 5, 5, 3), (1, 300, 1, 1, 0), (1, 65, 8, 2, 130), (5, 64, 6, 3, 1)])
def test_flash_mx_is_flash_then_quantiser(B, T, H, Hkv, pos0):
    from distributed_neural_networks_amd.ops import _lib
    from distributed_neural_networks_amd.ops import transformer_ops as T_
    from distributed_neural_networks_amd.ops.fp8 import kpad_of, mx_scale_bytes, quant_rows_mx
    hd, K, S, M = 64, H * 64, pos0 + T + 3, B * T
    g = torch.Generator(device=DEV).manual_seed(T * H)
    q = torch.randn(B, H, T, hd, generator=g, device=DEV).bfloat16()
    k, v = (torch.randn(B, Hkv, S, hd, generator=g, device=DEV).bfloat16() for _ in range(2))
    v[:, 0] *= 2.0 ** -9  # the two heads of a scale far apart
    v[0, -1, :, 5] = 0
    pos = torch.full((B,), pos0, dtype=torch.int32, device=DEV)
    rows = torch.empty((M, K), dtype=torch.bfloat16, device=DEV)
    T_.flash_attn(q.view(-1), k, v, rows, B, T, H, Hkv, hd, pos, one_group=True)
    kp = kpad_of(K)
    want, got = (torch.full((M * kp,), 0x7f, dtype=torch.uint8, device=DEV) for _ in range(2))
    s_want, s_got = (torch.full((mx_scale_bytes(M, kp),), 0xff, dtype=torch.uint8, device=DEV) for _ in range(2))
    quant_rows_mx(rows, want, s_want)
    _lib.check(_lib.lib().flash_attn_mx(q.data_ptr(), k.data_ptr(), v.data_ptr(), got.data_ptr(), kp, s_got.data_ptr(), B,
                                        T, H, Hkv, hd, S, pos.data_ptr(), 1 / math.sqrt(hd), _lib.stream_ptr()), "flash_attn_mx")
    assert torch.equal(got, want) and torch.equal(s_got, s_want)


def test_flash_mx_refuses(monkeypatch):
    from distributed_neural_networks_amd.ops import _lib
    t = torch.zeros(1 << 16, dtype=torch.uint8, device=DEV)
    call = lambda H, Hkv, hd, ld: _lib.lib().flash_attn_mx(*[t.data_ptr()] * 4, ld, t.data_ptr(), 1, 1, H, Hkv, hd, 8, 0,  # noqa: E731
                                                           1.0, _lib.stream_ptr())
    assert call(3, 2, 64, 256) == -1 and call(3, 3, 64, 128) == -1 and call(2, 2, 128, 256) == -3
    monkeypatch.setenv("DNN_FLASH_DB", "0")
    assert call(2, 2, 64, 128) == -3
