"""Prefill q | k | v with the rotation in the projection's epilogue: the bits of the projection's rows, split and rotated by a
pass of their own, on every tile."""
import pytest
import torch

pytestmark = pytest.mark.gpu
TILES = [("mid", t) for t in (2, 3, 4, 5, 6)] + [("tile", 256)]


@pytest.mark.parametrize("B,T,H,Hkv,K,S,at", [(1, 257, 2, 1, 64, 300, 7), (3, 143, 4, 2, 192, 160, 30), (1, 700, 32, 8, 4096, 704, 0),
                                              (2, 640, 3, 3, 512, 640, 0)])
@pytest.mark.parametrize("kind,tile", TILES)
def test_bits(kind, tile, B, T, H, Hkv, K, S, at):
    """Head counts whose columns no tile divides, rows past the cache's end (at + T > S), positions of their own."""
    from distributed_neural_networks_amd.ops import gemm as G_, transformer_ops as T_
    from distributed_neural_networks_amd.ops._lib import lib, stream_ptr
    g = torch.Generator().manual_seed(B * T + tile)
    hd, M, N = 128, B * T, (H + 2 * Hkv) * 128
    x, w = torch.randn(M, K, generator=g).bfloat16().cuda(), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16().cuda()
    pos = torch.tensor([max(0, at - 5 * b) for b in range(B)], dtype=torch.int32).cuda()
    ang = torch.arange(S)[:, None] * 500000.0 ** (-torch.arange(64) / 64.0)
    cos, sin = ang.cos().float().cuda(), ang.sin().float().cuda()
    stats, eps = torch.empty(M, 2, device="cuda"), 1e-5

    def outs():
        return (torch.full((B * H * T * hd,), 3.0, dtype=torch.bfloat16, device="cuda"),
                *(torch.full((B, Hkv, S, hd), 3.0, dtype=torch.bfloat16, device="cuda") for _ in range(2)))

    G_.set_gemm_mid(tile if kind == "mid" else -1)
    G_.set_gemm_tile(256 if kind == "tile" else 0)
    try:
        got = outs()
        rc = lib().gemm_bf16_qkv_rope(x.data_ptr(), K, w.data_ptr(), K, eps, stats.data_ptr(), *(t.data_ptr() for t in got),
                                      pos.data_ptr(), B, T, H, Hkv, hd, S, K, cos.data_ptr(), sin.data_ptr(), 0, stream_ptr())
        assert rc == 0
        want = outs()
        qkv = G_.linear(x, w, rowstat=stats)
        T_.qkv_split(qkv, want[0], want[1], want[2], B, T, H, Hkv, hd, pos, cos, sin)
    finally:
        G_.set_gemm_mid(-1)
        G_.set_gemm_tile(0)
    inside = (pos[:, None] + torch.arange(T, device="cuda") < S)[:, None, :, None]  # the pass drops rows past the cache
    q = [t.view(B, H, T, hd) * inside for t in (got[0], want[0])]
    assert torch.equal(q[0], q[1]) and torch.equal(got[1], want[1]) and torch.equal(got[2], want[2])
    r = x.double() * torch.rsqrt((x.double() ** 2).mean(1, keepdim=True) + eps)
    y = (r @ w.double().t()).view(B, T, H + 2 * Hkv, hd)
    p = (pos[:, None] + torch.arange(T, device="cuda")).clamp(max=S - 1).long()
    co, si = cos.double()[p][:, :, None], sin.double()[p][:, :, None]
    lo, hi = y[..., :64], y[..., 64:]
    rot = torch.cat([lo * co - hi * si, hi * co + lo * si], -1).transpose(1, 2)[:, :H]
    # two roundings to bf16, of the product and of the rotated pair: 2^-9 each, in norm under 2^-8
    assert ((q[0].double() - rot * inside).norm() / (rot * inside).norm()) < 2.0 ** -8


@pytest.mark.parametrize("B,T,H,Hkv,K,S", [(1, 1100, 96, 8, 512, 1100), (8, 512, 32, 8, 2048, 512), (1, 700, 32, 8, 4096, 710)])
def test_chosen(B, T, H, Hkv, K, S):
    """What the rule picks, columns in two launches too; every output against 64 bits."""
    from distributed_neural_networks_amd.ops._lib import lib, stream_ptr
    g = torch.Generator().manual_seed(T)
    hd, M, N = 128, B * T, (H + 2 * Hkv) * 128
    x, w = torch.randn(M, K, generator=g).bfloat16().cuda(), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16().cuda()
    pos = torch.arange(B, dtype=torch.int32).cuda() if S > T else torch.zeros(B, dtype=torch.int32).cuda()
    ang = torch.arange(S)[:, None] * 10000.0 ** (-torch.arange(64) / 64.0)
    cos, sin = ang.cos().float().cuda(), ang.sin().float().cuda()
    stats = torch.empty(M, 2, device="cuda")
    q = torch.full((B, H, T, hd), 3.0, dtype=torch.bfloat16, device="cuda")
    kc, vc = (torch.full((B, Hkv, S, hd), 3.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    assert lib().gemm_bf16_qkv_rope(x.data_ptr(), K, w.data_ptr(), K, 1e-5, stats.data_ptr(), q.data_ptr(), kc.data_ptr(),
                                    vc.data_ptr(), pos.data_ptr(), B, T, H, Hkv, hd, S, K, cos.data_ptr(), sin.data_ptr(), 0,
                                    stream_ptr()) == 0
    y = ((x.double() * torch.rsqrt((x.double() ** 2).mean(1, keepdim=True) + 1e-5)) @ w.double().t()).view(B, T, -1, hd)
    p = (pos[:, None] + torch.arange(T, device="cuda")).long()
    co, si = cos.double()[p][:, :, None], sin.double()[p][:, :, None]
    lo, hi = y[..., :64], y[..., 64:]
    rot = torch.cat([lo * co - hi * si, hi * co + lo * si], -1)
    for b in range(B):
        at = slice(pos[b].item(), pos[b].item() + T)
        for got, want in ((q[b], rot[b, :, :H]), (kc[b, :, at], rot[b, :, H:H + Hkv]), (vc[b, :, at], y[b, :, H + Hkv:])):
            want = want.transpose(0, 1)
            err = (got.double() - want).norm(dim=2) / want.norm(dim=2)  # row by row, as test_bits
            assert err.max() < 2.0 ** -7, err.max()
    assert (kc[:, :, :pos.min()] == 3).all() and (pos.max() + T >= S or (vc[:, :, pos.max() + T:] == 3).all())


def test_not_taken():
    """Tiles of 64 columns, heads of 64, rows the DMA cannot fetch: -3 and nothing launched."""
    from distributed_neural_networks_amd.ops import gemm as G_
    from distributed_neural_networks_amd.ops._lib import lib, stream_ptr
    x, w = torch.randn(300, 64).bfloat16().cuda(), torch.randn(512, 64).bfloat16().cuda()
    t = torch.full((1 << 18,), 3.0, device="cuda")
    pos = torch.zeros(1, dtype=torch.int32, device="cuda")

    def call(lda=64, H=2, hd=128):
        return lib().gemm_bf16_qkv_rope(x.data_ptr(), lda, w.data_ptr(), 64, 1e-5, t.data_ptr(), *(t.data_ptr(),) * 3,
                                        pos.data_ptr(), 1, 300, H, H // 2, hd, 300, 64, t.data_ptr(), t.data_ptr(), 0,
                                        stream_ptr())
    for tile in (0, 1):
        G_.set_gemm_mid(tile)
        try:
            assert call() == -3
        finally:
            G_.set_gemm_mid(-1)
    assert call(lda=63) == -3 and call(H=4, hd=64) == -3
    torch.cuda.synchronize()
    assert (t == 3).all()
