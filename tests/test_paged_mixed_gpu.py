"""Portions and single tokens of a step in one attention launch, against the float64
attention of the families' own tests; single tokens of more workgroups than CUs."""
import math

import pytest

import test_funepel_gpu as F
import test_kozusun_gpu as K
import test_lasizen_gpu as L

pytestmark = pytest.mark.gpu


@pytest.fixture
def mixed(monkeypatch):
    """The tests' two launches become one; returns the calls."""
    from distributed_neural_networks_amd.ops import decoder_ops as D_
    tiles, calls = [], []

    def decode(args, rows, n, splits, ws):
        calls.append((n, splits))
        D_.paged_mixed(args, tiles[0], rows, n, splits, ws)
    monkeypatch.setattr(D_, "paged_prefill", lambda args, t: tiles.append(t))
    monkeypatch.setattr(D_, "paged_decode", decode)
    return calls


@pytest.mark.parametrize("H,G,dk,dv", [(2, 2, 64, 64), (6, 2, 64, 128), (40, 1, 64, 64), (2, 1, 256, 256), (4, 4, 128, 128),
                                       (32, 8, 128, 128)])
@pytest.mark.parametrize("mask", [None, {"size": 50, "keep_first": 3}, {"size": 64, "keep_first": 64}])
def test_one_launch(mixed, H, G, dk, dv, mask):
    got, ref = K.run_attention("bf16", H, G, dk, dv, 1.2 / math.sqrt(dk), mask, K.SEQS, seed=H + dk)
    assert ((got - ref).norm(dim=1) / ref.norm(dim=1)).max().item() < 1.5e-2
    assert [s for _, s in mixed] == [1, 3]


@pytest.mark.parametrize("H,G,D,V,window", [(6, 2, 40, 24, 50), (40, 1, 128, 100, 64), (7, 1, 96, 72, 129)])
def test_one_launch_with_a_sink(mixed, H, G, D, V, window):
    got, ref = L.run_attention("bf16", H, G, D, V, window, L.SEQS, seed=H + D, scale=1.2 / math.sqrt(D))
    assert L.worst_row(got, ref) < 1e-2 and [s for _, s in mixed] == [1, 3, 7]


@pytest.mark.parametrize("H,G,dim,size", [(6, 2, 40, 50), (3, 1, 128, 1000)])
def test_one_launch_of_shared_keys(mixed, H, G, dim, size):
    got, ref = F.run_shared_attention("bf16", H, G, dim, size, F.SEQS, seed=H + dim)
    assert ((got - ref).flatten(1).norm(dim=1) / ref.flatten(1).norm(dim=1)).max().item() < 1.5e-2 and len(mixed) == 2


@pytest.mark.parametrize("n", [64, 65])
def test_single_tokens_beyond_a_workgroup_a_cu(n):
    """4 KV heads: 256 workgroups of eight waves, or 260 of four."""
    seqs = [(37 * i % 300, 1) for i in range(n)]
    got, ref = K.run_attention("bf16", 8, 4, 64, 64, 0.15, {"size": 130, "keep_first": 5}, seqs, seed=n)
    assert ((got - ref).norm(dim=1) / ref.norm(dim=1)).max().item() < 1.5e-2


def test_refusals():
    import torch
    from distributed_neural_networks_amd.ops import decoder_ops as D_
    t = torch.zeros(4, 4, dtype=torch.int32, device="cuda")
    for tiles, splits, ws in ((t[:, :3], 1, None), (t.float(), 1, None), (t, 2, None), (t, 2, t)):
        with pytest.raises(ValueError):
            D_.paged_mixed(None, tiles, t[0], 2, splits, ws)
