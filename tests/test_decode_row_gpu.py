"""Decode steps of one or two rows by partial products against the step's own launches."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _stage(model, blocks, first, last, S, max_batch=4):
    from distributed_neural_networks_amd import checkpoint as ckpt
    from distributed_neural_networks_amd.runtime.transformer import TransformerStage
    sd = ckpt.random_stage_state_dict(model, 0, blocks - 1, first, last, 3, device=DEV, nontrivial=True)
    return TransformerStage(model, sd, 0, blocks - 1, first, last, DEV, max_batch=max_batch, max_seq=S)


def _steps(st, seed, B, b0, pos, n):
    """n tokens of sequences b0.. at positions ``pos`` on, over caches of noise: outputs, caches."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    for t in (st.kc, st.vc):
        t.copy_(torch.randn(t.shape, generator=g, device=DEV) * 0.5)
    p, outs = torch.tensor(pos, dtype=torch.int32, device=DEV), []
    for _ in range(n):
        x = (torch.randint(0, st.V, (B, 1), generator=g, device=DEV, dtype=torch.int32) if st.first
             else torch.randn(B, st.d, generator=g, device=DEV).bfloat16())
        y = st.step(x, p, B, 1, b0=b0)
        outs.append((y.probs if st.last else y).float().clone())
        p += 1
    return torch.stack(outs), st.kc.clone(), st.vc.clone()


@pytest.mark.parametrize("model,blocks,first,last,S,B,b0,pos", [
    ("gpt2", 2, True, True, 104, 1, 0, [0]), ("gpt2", 3, False, False, 400, 1, 3, [62]), ("gpt2", 1, True, False, 300, 1, 0, [255]),
    ("gpt2", 2, False, True, 1000, 2, 1, [995, 1]), ("gpt2-medium", 2, True, True, 130, 1, 2, [127]),
    ("gpt2-medium", 1, False, False, 66, 2, 2, [63, 64]), ("gpt2-tiny", 4, True, True, 200, 2, 0, [30, 31]),
    ("gpt2-tiny", 2, False, False, 40, 1, 0, [39])])  # the last: past the cache's end
def test_partial_products_against_the_launches(model, blocks, first, last, S, B, b0, pos, monkeypatch):
    """Both store bf16 at the same places and differ in the order of fp32 sums, so a stored value may round the other
    way: one unit, 2^-8 of it, of every value at worst, and what a block makes of it (the residual's share of it stays)."""
    st = _stage(model, blocks, first, last, S)
    native, calls = type(st)._decode_rows, []
    monkeypatch.setattr(type(st), "_decode_rows", lambda self, *a: calls.append(native(self, *a)) or calls[-1])
    got, k, v = _steps(st, 5, B, b0, pos, 3)
    assert calls == [True] * 3
    monkeypatch.setattr(type(st), "_decode_rows", lambda self, *a: False)
    want, k0, v0 = _steps(st, 5, B, b0, pos, 3)
    rel = lambda a, b: ((a.float() - b.float()).norm() / b.float().norm()).item()  # noqa: E731
    assert torch.isfinite(got).all() and rel(got, want) < 2.0 ** -8
    for a, b in ((k, k0), (v, v0)):
        assert rel(a, b) < 2.0 ** -8
        rows = torch.zeros(a.shape[1], a.shape[3], dtype=torch.bool, device=DEV)
        for i, p in enumerate(pos):
            rows[b0 + i, p:p + 3] = True
        assert torch.equal(a.transpose(2, 3)[:, ~rows], b.transpose(2, 3)[:, ~rows])  # nothing else is written
    again, k1, _ = _steps(st, 5, B, b0, pos, 3)
    monkeypatch.undo()
    one, k2, _ = _steps(st, 5, B, b0, pos, 3)
    assert torch.equal(one, got) and torch.equal(k2, k) and torch.equal(again, want)


def test_what_stays_with_the_launches():
    from distributed_neural_networks_amd.ops import _lib
    f = _lib.lib().decode_row_parts
    assert f(1, 768, 12, 12, 64, 1024) == 768 * 16 and f(2, 1024, 16, 16, 64, 2047) == 2 * 1024 * 20
    for args in ((3, 768, 12, 12, 64, 64), (0, 768, 12, 12, 64, 64), (1, 1280, 20, 20, 64, 64), (1, 768, 12, 6, 64, 64),
                 (1, 768, 6, 6, 128, 64), (1, 768, 12, 12, 64, 2048)):
        assert f(*args) == 0


def test_captured_step_follows_positions_and_weights():
    """A graph of the step, replayed with other positions, rows and changed weights, against eager steps."""
    from distributed_neural_networks_amd.runtime.graph import GraphedStep
    st = _stage("gpt2", 2, False, False, 64, 1)
    x, p = torch.zeros(1, st.d, device=DEV, dtype=torch.bfloat16), torch.zeros(1, dtype=torch.int32, device=DEV)
    step = GraphedStep(lambda: st.step(x, p, 1, 1), torch.device(DEV, 0))
    for i in range(4):
        x.copy_(torch.randn(1, st.d, generator=torch.Generator().manual_seed(i)))
        p.fill_(7 * i)
        if i == 2:
            st.layers[0].w_up.bias.mul_(2)
        got = step().clone()
        assert torch.equal(got, st.step(x, p, 1, 1))
