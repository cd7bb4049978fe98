"""Tiles with one epilogue against the tiles with all of them (rows at a distance that is no
multiple of 16 bytes): the same bits, on every tile, with waves past the columns and rows past the last."""
import math

import pytest
import torch
from torch.profiler import ProfilerActivity, profile

pytestmark = pytest.mark.gpu
DEV = "cuda"
KINDS = ["none", "bias", "xielu", "gelu_tanh", "res", "res_bias", "res_parts", "stat", "silu_stat", "gelu_norm", "gelu_parts"]


@pytest.mark.parametrize("tile", range(7))
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("M,N,K", [(65, 192, 128), (257, 320, 192), (129, 64, 64 * 7)])
def test_one_epilogue(tile, kind, M, N, K):
    from distributed_neural_networks_amd.ops import gemm as G
    g = torch.Generator(device=DEV).manual_seed(tile + M)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    x, w, kw = r(M, K).bfloat16(), (r(N, K) / math.sqrt(K)).bfloat16(), {}
    glu = kind in ("gelu_tanh", "silu_stat")
    act = {"xielu": G.ACT_XIELU, "gelu_tanh": G.ACT_GELU_TANH_MUL, "silu_stat": G.ACT_SILU_MUL}.get(kind, G.ACT_NONE)
    bias = r(N + 2 if kind == "xielu" else N) if kind in ("bias", "xielu", "res_bias", "res_parts") or "gelu_" in kind and not glu else None
    if kind.startswith("gelu_") and not glu:
        act, kw["colsum"] = G.ACT_GELU, r(N)
    if kind in ("stat", "silu_stat", "gelu_norm"):
        kw["rowstat"] = torch.stack([r(M).abs() + 0.5, r(M) if "colsum" in kw else torch.zeros(M, device=DEV)], 1).contiguous()
    if kind.startswith("res"):
        kw["residual"] = r(M, N).bfloat16()
    parts = G.parts_buffer(M, N, DEV)
    if kind == "gelu_parts":
        t = x.float().view(M, K // 32, 32)
        p = torch.stack([t.mean(-1), (t - t.mean(-1, keepdim=True)).square().sum(-1)], -1)
        kw["parts"] = (p.reshape(M, -1).contiguous(), 1e-5, 2)
    no, outs, names = N // 2 if glu else N, [], []
    G.lib().gemm_set_mid(tile, 1)
    try:
        for ld in (no, no + 4):
            out = torch.full((M + 1, ld), 7.0, device=DEV, dtype=torch.bfloat16)
            extra = {"parts_out": parts} if kind == "res_parts" and ld == no else {}
            with profile(activities=[ProfilerActivity.CUDA]) as p:
                G.linear(x, w, bias, act, out=out[:M, :no], **kw, **extra)
                torch.cuda.synchronize()
            names.append([e.key for e in p.key_averages() if "gemm_mid_kernel" in e.key])
            assert (out[M] == 7).all() and (out[:, no:] == 7).all()
            outs.append(out[:M, :no].clone())
    finally:
        G.lib().gemm_set_mid(-1, 1)
    assert [len(n) for n in names] == [1, 1] and "-1>" not in names[0][0] and "-1>" in names[1][0]  # MID_ANY
    assert torch.equal(*outs) and torch.isfinite(outs[0]).all() and outs[0].abs().max() > 0.1
    if kind == "res_parts":
        t = outs[0].float().view(M, N // 32, 32)
        assert torch.allclose(parts.view(M, N // 32, 2)[..., 0], t.mean(-1), rtol=0, atol=1e-5)
    if kind in ("none", "res"):  # of bf16 storage and fp32 sums
        ref = x.double() @ w.double().t() + (kw["residual"].double() if "residual" in kw else 0)
        assert ((outs[0].double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2.0 ** -17 * (x.double().abs() @ w.double().abs().t())).all()


@pytest.mark.parametrize("tile", range(5))
@pytest.mark.parametrize("M,N,K", [(256, 256, 128), (257, 320, 320), (300, 448, 640)])
def test_one_epilogue_of_e4m3(tile, M, N, K):
    from distributed_neural_networks_amd.ops import gemm as G
    from distributed_neural_networks_amd.ops.fp8 import kpad_of, linear_fp8, mx_scale_bytes, quantize_weight
    g = torch.Generator(device=DEV).manual_seed(tile + M)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    x, w, bias, res = r(M, K).bfloat16(), quantize_weight(r(N, K) / math.sqrt(K), DEV), r(N), r(M, N).bfloat16()
    q, sx = (torch.empty(n, dtype=torch.uint8, device=DEV) for n in (M * kpad_of(K), mx_scale_bytes(M, kpad_of(K))))
    outs, names = [], []
    G.lib().gemm_set_mid(tile, 1)
    try:
        for ld in (N, N + 4):
            out = torch.full((M + 1, ld), 7.0, device=DEV, dtype=torch.bfloat16)
            with profile(activities=[ProfilerActivity.CUDA]) as p:
                linear_fp8(x, w, bias, 0, res, out[:M, :N], q, None, sx=sx)
                torch.cuda.synchronize()
            names.append([e.key for e in p.key_averages() if "gemm_mid_fp8" in e.key])
            assert (out[M] == 7).all() and (out[:, N:] == 7).all()
            outs.append(out[:M, :N].clone())
    finally:
        G.lib().gemm_set_mid(-1, 1)
    assert [len(n) for n in names] == [1, 1] and names[0] != names[1]
    assert torch.equal(*outs)
    ref = x.double() @ (w.q[:, :K].double() * w.scale.double()[:, None]).t() + bias.double() + res.double()
    assert ((outs[0].double() - ref).norm() / ref.norm()).item() < 2.0 ** -4  # an activation's e4m3 rounding, at worst
