"""Decode projections laid out for one shape each, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _kernels(f):
    """Names of the kernels that ``f`` launches."""
    from torch.profiler import ProfilerActivity, profile
    f()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        f()
        torch.cuda.synchronize()
    return " ".join(e.key for e in p.key_averages())


def _err(y, ref, scale):
    """Largest error, of what bf16 storage (2^-9 of the value) and fp32 sums of bf16 products of size ``scale`` allow."""
    return ((y.double() - ref).abs() / (2.0 ** -8 * ref.abs() + 2.0 ** -17 * scale)).max().item()


@pytest.mark.parametrize("M", [1, 2, 15, 16, 17, 32, 33, 48, 49, 63, 64])
@pytest.mark.parametrize("K,N,w8,act", [(768, 2304, False, 0), (768, 3072, False, 2), (768, 48, False, 0), (1600, 4800, True, 0),
                                        (1600, 6400, True, 2), (1600, 80, True, 0)])
def test_norm_projection(M, K, N, w8, act):
    """Folded LayerNorm from merged partials: rows of a large mean, ragged rows, a column group that is not whole."""
    from distributed_neural_networks_amd.ops.gemm import attach_shuffled, fold_norm, linear_norm, rowstats_buffer
    g = torch.Generator(device=DEV).manual_seed(M * N)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    x = torch.zeros(M, K + 32, device=DEV, dtype=torch.bfloat16)[:, 8:8 + K]  # rows K + 32 apart
    x.copy_(r(M, K) * torch.logspace(-2, 2, M, device=DEV)[:, None] + 3)
    f = fold_norm(r(N, K) * 0.02, 1 + 0.1 * r(K), 0.1 * r(K), r(N), False, 1e-5, DEV, w8)
    attach_shuffled(f)
    rs = rowstats_buffer(M, K, DEV)
    t = x.float().reshape(M, K // 16, 16)
    rv = rs.view(M, -1, 2)
    rv[:, :K // 16, 0] = t.mean(-1)
    rv[:, :K // 16, 1] = (t - t.mean(-1, keepdim=True)).square().sum(-1)
    out = torch.full((M + 1, N + 4), 7.0, device=DEV, dtype=torch.bfloat16)
    call = lambda: linear_norm(x, f, act=act, out=out[:M, :N], rs_in=rs)  # noqa: E731
    assert "gemm_lean" in _kernels(call)
    xd = x.double()
    xd = (xd - xd.mean(-1, keepdim=True)) / (xd.var(-1, unbiased=False, keepdim=True) + 1e-5).sqrt()
    w = (f.w.q[:, :K].double() * f.w.scale.double()[:, None]) if w8 else f.w.double()
    z = xd @ w.t() + f.bias.double()
    ref = torch.nn.functional.gelu(z) if act else z
    # the mean's share of the sum is taken off behind it: products of the size of the row's largest values over its deviation
    scale = (x.double().abs().amax(-1, keepdim=True) / (x.double().var(-1, unbiased=False, keepdim=True) + 1e-5).sqrt()) * w.abs().sum(-1)
    assert _err(out[:M, :N], ref, scale) < 1
    assert (out[M:] == 7).all() and (out[:, N:] == 7).all()


@pytest.mark.parametrize("M", [1, 7, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("K,N,w8", [(768, 768, False), (3072, 768, False), (3072, 1040, False), (4096, 4096, False), (1600, 1600, True),
                                    (6400, 1600, True), (1600, 48, True)])
def test_residual_projection(M, K, N, w8):
    """In place on the residual, with the statistics of the stored rows."""
    from distributed_neural_networks_amd.ops.fp8 import linear_w8, quantize_weight
    from distributed_neural_networks_amd.ops.gemm import attach_shuffled, linear, rowstats_buffer, rowstats_written
    g = torch.Generator(device=DEV).manual_seed(M + K)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    x, h0, bias, W = r(M, K).bfloat16(), r(M + 1, N).bfloat16(), (None if K == 4096 else r(N)), r(N, K) * 0.02
    w = attach_shuffled(quantize_weight(W, DEV)) if w8 else W.bfloat16()
    ws = None if w8 else attach_shuffled(w)
    rs, h = rowstats_buffer(M, N, DEV), h0.clone()

    def call():
        h.copy_(h0)
        return (linear_w8(x, w, bias, 0, h[:M], h[:M], rs_out=rs) if w8
                else linear(x, w, bias, None, h[:M], h[:M], w_shuf=ws, rs_out=rs))
    assert "gemm_lean" in _kernels(call) and rowstats_written()
    wd = (w.q[:, :K].double() * w.scale.double()[:, None]) if w8 else w.double()
    ref = x.double() @ wd.t() + (0 if bias is None else bias.double()) + h0[:M].double()
    assert _err(h[:M], ref, x.double().abs() @ wd.abs().t()) < 1
    assert torch.equal(h[M], h0[M])
    t = h[:M].float().reshape(M, N // 16, 16)
    assert torch.allclose(rs.view(M, -1, 2)[:, :N // 16, 0], t.mean(-1), rtol=0, atol=2e-6 * t.abs().max().item())
    assert torch.allclose(rs.view(M, -1, 2)[:, :N // 16, 1], (t - t.mean(-1, keepdim=True)).square().sum(-1), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("M,N,act", [(m, n, 0) for m in (1, 9, 16, 17, 31, 32, 33, 48, 49, 64) for n in (6144, 5200)]
                         + [(9, 28672, 3), (16, 28672, 3), (13, 48, 3)])
def test_rms_projection(M, N, act):
    from distributed_neural_networks_amd.ops.gemm import attach_shuffled, fold_norm, linear_norm
    K = 4096
    g = torch.Generator(device=DEV).manual_seed(M)
    x = (torch.randn(M, K, generator=g, device=DEV) * torch.logspace(-2, 2, M, device=DEV)[:, None]).bfloat16()
    f = fold_norm(torch.randn(N, K, generator=g, device=DEV) * 0.02, torch.ones(K, device=DEV), None, None, True, 1e-5, DEV)
    attach_shuffled(f)
    NO = N // 2 if act else N
    out = torch.full((M + 1, NO + 4), 7.0, device=DEV, dtype=torch.bfloat16)
    assert "gemm_lean" in _kernels(lambda: linear_norm(x, f, act=act, out=out[:M, :NO]))
    xd = x.double() / (x.double().square().mean(-1, keepdim=True) + 1e-5).sqrt()
    z, size = xd @ f.w.double().t(), xd.abs() @ f.w.double().abs().t()
    if act:  # 8 gate columns, their 8 up columns; the derivative of silu is under 1.1
        (gate, up), (sg, su) = (t.view(M, -1, 2, 8).transpose(1, 2).reshape(M, 2, NO).unbind(1) for t in (z, size))
        z, size = torch.nn.functional.silu(gate) * up, 1.1 * sg * up.abs() + gate.abs() * su
    assert _err(out[:M, :NO], z, size) < 1
    assert (out[M:] == 7).all() and (out[:, NO:] == 7).all()


@pytest.mark.parametrize("M,N,lean", [(1, 4096, False), (1, 4112, True), (8, 6144, True), (8, 6160, False), (9, 4096, False),
                                      (9, 6160, True), (16, 8192, True), (17, 4096, False), (17, 6144, True), (17, 6160, False),
                                      (33, 2560, False), (48, 2576, True), (48, 6160, False), (49, 2048, False), (49, 2064, True),
                                      (64, 8192, True), (64, 64, False)])
def test_rms_projection_lines(M, N, lean):
    """Columns that leave CUs idle or start a second round stay with the general kernels."""
    from distributed_neural_networks_amd.ops.gemm import attach_shuffled, decode_workspace, fold_norm, linear_norm
    K = 4096
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    f = attach_shuffled(fold_norm(torch.randn(N, K, generator=g, device=DEV) * 0.02, torch.ones(K, device=DEV), None, None, True, 1e-5, DEV))
    out = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    assert ("gemm_lean" in _kernels(lambda: linear_norm(x, f, out=out, ws=decode_workspace(DEV, 7)))) == lean
    xd = x.double() / (x.double().square().mean(-1, keepdim=True) + 1e-5).sqrt()
    assert _err(out, xd @ f.w.double().t(), xd.abs() @ f.w.double().abs().t()) < 1


@pytest.mark.parametrize("M,N,lean", [(32, 64, True), (33, 1024, False), (33, 1040, True), (64, 64, False)])
def test_residual_projection_lines(M, N, lean):
    from distributed_neural_networks_amd.ops.gemm import decode_workspace, linear, shuffle_weight
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x, W = torch.randn(M, 4096, generator=g, device=DEV).bfloat16(), (torch.randn(N, 4096, generator=g, device=DEV) * 0.02).bfloat16()
    out, res, sh = (torch.empty(M, N, device=DEV, dtype=torch.bfloat16), torch.randn(M, N, generator=g, device=DEV).bfloat16(),
                    shuffle_weight(W))
    assert ("gemm_lean" in _kernels(lambda: linear(x, W, None, None, res, out, w_shuf=sh, ws=decode_workspace(DEV, 7)))) == lean
    assert _err(out, x.double() @ W.double().t() + res.double(), x.double().abs() @ W.double().abs().t()) < 1


def test_what_stays_with_the_general_kernels():
    """Rows off 16 bytes, outputs off 8, other widths and numbers of rows, no partials: the same results from elsewhere."""
    from distributed_neural_networks_amd.ops.gemm import attach_shuffled, linear
    g = torch.Generator(device=DEV).manual_seed(1)
    for M, K, N, off in ((8, 768, 770, 0), (65, 768, 768, 0), (8, 832, 768, 0), (8, 768, 768, 1), (65, 4096, 4096, 0)):
        x, W = torch.randn(M, K, generator=g, device=DEV).bfloat16(), (torch.randn(N, K, generator=g, device=DEV) * 0.02).bfloat16()
        out, res = torch.empty(M, N + off, device=DEV, dtype=torch.bfloat16)[:, off:], torch.randn(M, N, generator=g, device=DEV).bfloat16()
        call = lambda: linear(x, W, None, None, res, out, w_shuf=attach_shuffled(W))  # noqa: E731
        assert "gemm_lean" not in _kernels(call), (M, K, N, off)
        ref = x.double() @ W.double().t() + res.double()
        assert _err(out, ref, x.double().abs() @ W.double().abs().t()) < 1
