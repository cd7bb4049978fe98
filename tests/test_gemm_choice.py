"""Which rows take the decode kernels (the library's host side: no GPU needed)."""
import pytest

from distributed_neural_networks_amd.ops import gemm as G


@pytest.fixture
def max_m():
    from distributed_neural_networks_amd.ops._lib import lib
    try:
        lib()
    except RuntimeError as e:
        pytest.skip(f"kernel library: {e}")
    yield G.set_skinny_max_m
    G.set_skinny_max_m()


def test_set_skinny_max_m_governs_folded_norms(max_m):
    """Rows past the switch go by estimate, below 65 too: a head of 50304 columns is then the tiles'."""
    head = (50304, False, 768, True)
    assert all(G.skinny_rows(M, *head) for M in (1, 33, 48, 64)) and not G.skinny_rows(65, *head)
    max_m(32)
    assert G.skinny_rows(32, *head) and not any(G.skinny_rows(M, *head) for M in (33, 48, 64))
    assert G.skinny_rows(48, 768, False, 768, True)  # 16 workgroups of 128 x 128: still the decode kernels'
    max_m(64)
    assert G.skinny_rows(48, *head)  # no answer of the other setting is kept


def test_fp8_rows():
    assert G.skinny_rows(64, 50304, True) and G.skinny_rows(256, 12160, True) and not G.skinny_rows(65, 24576, True)
    assert not G.skinny_rows(257, 128, True)


def test_attention_that_quantises_is_for_short_prefill(max_m):
    """-3, nothing launched: long sequences, and launches of few or many workgroups of 769 tokens on, keep both launches."""
    from distributed_neural_networks_amd.ops._lib import lib
    call = lambda B, T, H: lib().flash_attn_mx(0, 0, 0, 0, -(-H // 2) * 128, 0, B, T, H, H, 64, T, 0, 0.125, 0)  # noqa: E731
    for B, T, H in ((1, 1025, 25), (4, 1280, 20), (1, 2048, 12), (16, 4096, 16),  # 3 to 14 % slower
                    (1, 769, 12), (1, 960, 16), (1, 1024, 12), (8, 960, 25), (16, 1024, 25), (8, 1024, 20)):
        assert call(B, T, H) == -3, (B, T, H)


def test_rotating_projection_leaves_other_shapes_to_the_rows(max_m):
    """-3, nothing launched, also for a K that its tiles do not take; pointers that no kernel could use stay refused."""
    from distributed_neural_networks_amd.ops._lib import lib
    call = lambda K=256, hd=128, M=300, cos=16: lib().gemm_bf16_qkv_rope(  # noqa: E731
        0, K, 0, K, 1e-5, 0, 0, 0, 0, 0, 1, M, 2, 1, hd, 512, K, cos, cos, 0, 0)
    assert call(K=96) == call(K=4128) == call(hd=64) == -3
    assert call(cos=0) == call(M=0) == -1
