"""The token gate of K that eight waves hold, against fp64: rows and columns around the edges of its tiles."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [1024, 2048, 4096])
@pytest.mark.parametrize("M,n,np_", [(1, 64, 64), (16, 50, 64), (17, 256, 256), (256, 250, 256), (257, 256, 256), (512, 256, 256),
                                     (1000, 64, 64), (1030, 192, 192), (545, 512, 512)])
def test_token_gate(K, M, n, np_):
    from distributed_neural_networks_amd.ops._lib import check, lib, ptr, stream_ptr
    from distributed_neural_networks_amd.ops.gemm import shuffle_weight

    g = torch.Generator().manual_seed(K + M)
    V, off = 300, 7
    wide = torch.full((M, K + 64), float("nan"), dtype=torch.bfloat16)
    wide[:, :K] = torch.randn(M, K, generator=g)
    w = torch.randn(np_, K, generator=g).mul_(K ** -0.5).bfloat16()
    w[n:] = 0
    table = torch.randn(V, off + n + 1, generator=g).bfloat16()
    tok = torch.randint(0, V, (M,), generator=g).int()
    tok[0], tok[-1] = -3, V + 5  # clamped
    x, wd, td, kd = wide.cuda(), w.cuda(), table.cuda(), tok.cuda()
    out = torch.full((M + 1, np_ + 4), 7.0, device="cuda", dtype=torch.bfloat16)
    ws = shuffle_weight(wd)
    check(lib().token_gate(ptr(x), K + 64, ptr(wd), K, ptr(ws), K, ptr(td), off + n + 1, off, ptr(kd), V, ptr(out), np_ + 4, M,
                           n, np_, stream_ptr()), "token_gate")
    z = wide[:, :K].double() @ w.double().T
    e = table.double()[tok.long().clamp(0, V - 1), off:off + n]
    want = 0.5 * z * (1 + torch.tanh(0.797884560802865 * (z + 0.044715 * z ** 3)))
    want[:, :n] *= e
    want[:, n:] = 0
    got = out.double().cpu()
    assert (got[M:] == 7).all() and (got[:M, np_:] == 7).all()
    # the product in fp32 (sums of unit size: 1e-5 with the tanh), rounded once to bf16
    err = (got[:M, :np_] - want).abs()
    assert (err <= 2.0 ** -8 * want.abs() + 2e-5).all(), err.max()
