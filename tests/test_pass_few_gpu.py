"""Passes on a few images by one native call: when, and with the results of the stages' forwards."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _pipe(batch, monkeypatch, stages=None, **kw):
    from distributed_neural_networks_amd.models.cifar import NeuralNetwork
    from distributed_neural_networks_amd.ops import cifar as cops
    from distributed_neural_networks_amd.runtime.pipeline import ColocatedPipeline
    from distributed_neural_networks_amd.runtime.stages import CifarHipStage
    dev = torch.device("cuda", 0)
    torch.manual_seed(5)
    sd = NeuralNetwork().eval().state_dict()
    ranges = [(0, 1), (2, 3)] if stages is None else stages
    calls, native = [], cops.pass_few
    monkeypatch.setattr(cops, "pass_few", lambda *a: calls.append(1) or native(*a))
    return ColocatedPipeline([CifarHipStage(sd, a, b, dev, **kw) for a, b in ranges], batch), calls


def _check(pipe, x):
    got = pipe(x)
    probs, pred = got.probs.clone(), got.pred.clone()
    assert torch.equal(pipe.x, x)
    want = pipe()  # the stages' forwards on the copy that was left
    assert torch.equal(probs, want.probs) and torch.equal(pred, want.pred)


@pytest.mark.parametrize("batch,kw", [(1, {}), (64, {}), (65, {"boundary": "split"}), (512, {})])
def test_one_call(batch, kw, monkeypatch):
    pipe, calls = _pipe(batch, monkeypatch, **kw)
    for i in range(2):
        _check(pipe, torch.randn(batch, 3, 32, 32, device="cuda"))
    assert len(calls) == 2
    x = torch.randn(batch, 3, 32, 32, device="cuda")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # the current stream's
        _check(pipe, x)
    pipe.stages[1].wh.b_fc1.add_(0.5)  # weights as they are at the call
    torch.cuda.synchronize()
    _check(pipe, x)


@pytest.mark.parametrize("what", ["many", "ranges", "whole", "wrapped", "patched", "encoding", "output", "keep"])
def test_the_stages_decide(what, monkeypatch):
    from distributed_neural_networks_amd.runtime.stages import CifarHipStage
    batch = 513 if what == "many" else 8
    pipe, calls = _pipe(batch, monkeypatch, {"ranges": [(0, 2), (3, 3)], "whole": [(0, 3)]}.get(what))
    x = torch.randn(batch, 3, 32, 32, device="cuda")
    if what == "wrapped":
        class Wrapped(CifarHipStage):
            def forward(self, x, out=None, keep=None):
                return super().forward(x, out, keep)
        pipe.stages[1].__class__ = Wrapped
    if what == "patched":
        last = pipe.stages[1]
        last.forward = lambda x, out=None: CifarHipStage.forward(last, x, out)
    if what == "encoding":  # the stages disagree, and the forwards are what decides what comes of it
        pipe.stages[0].boundary = "split"
        got = [t.clone() for t in (pipe(x).probs, pipe.bufs[0])]
        pipe.x.copy_(x)
        assert all(torch.equal(a.nan_to_num(), b.nan_to_num()) for a, b in zip(got, (pipe().probs, pipe.bufs[0])))
        assert not calls
        return
    if what == "output":  # one at a time: test_pipeline_cpu.py
        pipe.bufs[0] = pipe.bufs[0].double()
        with pytest.raises(ValueError, match="bad output buffer"):
            pipe(x)
        assert not calls
        return
    if what == "keep":  # shares memory with the images
        pipe.x = torch.cat([x, x])[1:batch + 1]
        with pytest.raises(ValueError):
            pipe(pipe.x._base[:batch] if pipe.x._base is not None else pipe.x[:])
        assert not calls
        return
    _check(pipe, x)
    assert not calls
