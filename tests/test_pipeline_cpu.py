"""Which inputs the colocated pipeline's first stage may read in place (CPU: the rule alone)."""
import pytest
import torch


def test_input_apart_from_what_the_pass_writes():
    """One byte of the input buffer or of a stage's output is enough, on either side."""
    from distributed_neural_networks_amd.runtime.pipeline import ColocatedPipeline
    from distributed_neural_networks_amd.runtime.stages import TorchStage
    from distributed_neural_networks_amd.models.cifar import NeuralNetwork
    sd = NeuralNetwork().state_dict()
    pipe = ColocatedPipeline([TorchStage("cifar10", sd, 0, 1, True, False), TorchStage("cifar10", sd, 2, 3, False, True)], 2)
    n = pipe.x.nbytes
    for b in (pipe.x, *pipe.bufs):
        at = b.data_ptr()
        assert not any(pipe._apart(at + d) for d in (0, 1 - n, b.nbytes - 1, (b.nbytes - n) // 2))
    first, last = (f(b.data_ptr() + (f is max) * b.nbytes for b in (pipe.x, *pipe.bufs)) for f in (min, max))
    assert pipe._apart(first - n) and pipe._apart(last)


def test_keep_shares_no_byte_with_the_images(monkeypatch):
    from distributed_neural_networks_amd.models.cifar import NeuralNetwork
    from distributed_neural_networks_amd.ops import cifar as cops
    w = cops.pack_stage0(NeuralNetwork().state_dict(), torch.device("cpu"))
    launched = []
    monkeypatch.setattr(cops, "lib", lambda: type("L", (), {"cifar_stage0_x3": staticmethod(lambda *a: launched.append(a) or 0)}))
    monkeypatch.setattr(cops, "stream_ptr", lambda: 0)
    n = 2 * 3072
    m = torch.zeros(3 * n)
    x = m[n:2 * n].view(2, 3, 32, 32)
    for start in (n, 1, n - 1, n + 1, 2 * n - 1):
        with pytest.raises(ValueError, match="apart"):
            cops.stage0_forward(x, w, keep=m[start:start + n].view_as(x))
    for start in (0, 2 * n):
        cops.stage0_forward(x, w, keep=m[start:start + n].view_as(x))
    assert len(launched) == 2


def test_wrapped_forward_is_given_no_keep():
    from distributed_neural_networks_amd.models.cifar import NeuralNetwork
    from distributed_neural_networks_amd.runtime.stages import CifarHipStage
    sd = NeuralNetwork().state_dict()
    cpu = torch.device("cpu")

    class Wrapped(CifarHipStage):
        def forward(self, x, out=None):
            return super().forward(x, out)

    plain, patched = CifarHipStage(sd, 0, 1, cpu), CifarHipStage(sd, 0, 1, cpu)
    patched.forward = lambda x, out=None: out
    assert plain.keeps_input and not Wrapped(sd, 0, 1, cpu).keeps_input and not patched.keeps_input
    assert not CifarHipStage(sd, 2, 3, cpu).keeps_input and not CifarHipStage(sd, 0, 1, cpu, precision="bf16").keeps_input


def _two(monkeypatch, first, last):
    """A two-stage pipeline on the CPU whose first stage reads its input where it lies."""
    from distributed_neural_networks_amd.runtime.pipeline import ColocatedPipeline
    monkeypatch.setattr(ColocatedPipeline, "_reads", lambda self, x: True)
    return ColocatedPipeline([first, last], 2)


def test_a_first_stage_of_the_callers_own(monkeypatch):
    """keeps_input says that ``forward`` takes ``keep``, and nothing of passes by one call."""
    from distributed_neural_networks_amd.models.cifar import NeuralNetwork
    from distributed_neural_networks_amd.runtime.stages import TorchStage

    class Keeps(TorchStage):
        keeps_input = True

        def forward(self, x, out=None, keep=None):
            if keep is not None:
                keep.copy_(x)
            return super().forward(x, out)

    torch.manual_seed(2)
    net = NeuralNetwork().eval()
    sd = net.state_dict()
    pipe = _two(monkeypatch, Keeps("cifar10", sd, 0, 1, True, False), TorchStage("cifar10", sd, 2, 3, False, True))
    x = torch.randn(2, 3, 32, 32)
    got = pipe(x).probs.clone()
    assert torch.allclose(got, net(x), atol=1e-6) and torch.equal(pipe.x, x) and torch.equal(pipe().probs, got)


@pytest.mark.parametrize("what", ["class", "first", "last"])
def test_a_replaced_forward_is_not_passed_by(what, monkeypatch):
    """On the class or on a stage, on either side of the cut: the native call leaves the pass to the forwards."""
    from distributed_neural_networks_amd.models.cifar import NeuralNetwork
    from distributed_neural_networks_amd.ops import cifar as cops
    from distributed_neural_networks_amd.runtime.stages import CifarHipStage
    native = []
    monkeypatch.setattr(cops, "pass_few", lambda *a: native.append(1))
    sd, cpu = NeuralNetwork().state_dict(), torch.device("cpu")
    pipe = _two(monkeypatch, CifarHipStage(sd, 0, 1, cpu), CifarHipStage(sd, 2, 3, cpu))
    few = lambda: pipe.stages[0].pass_few(pipe.stages[1], torch.zeros(2, 3, 32, 32), *pipe.bufs, pipe.x)  # noqa: E731
    assert few() is not None and native == [1]  # as it is built
    at = {"class": CifarHipStage, "first": pipe.stages[0], "last": pipe.stages[1]}[what]
    monkeypatch.setattr(at, "forward", lambda *a, **kw: None)
    assert few() is None and native == [1]
    assert pipe.stages[0].keeps_input == (what == "last")


@pytest.mark.parametrize("buf", ["h", "probs", "keep"])
def test_the_native_call_writes_plain_buffers_only(buf, monkeypatch):
    """It checks nothing itself: each buffer by itself, of another type, shape or order, or a keep on the images."""
    from distributed_neural_networks_amd.models.cifar import NeuralNetwork
    from distributed_neural_networks_amd.ops import cifar as cops
    from distributed_neural_networks_amd.runtime.stages import CifarHipStage
    native = []
    monkeypatch.setattr(cops, "pass_few", lambda *a: native.append(1))
    sd, cpu = NeuralNetwork().state_dict(), torch.device("cpu")
    first, last = CifarHipStage(sd, 0, 1, cpu), CifarHipStage(sd, 2, 3, cpu)
    x, good = torch.zeros(4, 3, 32, 32), {"h": torch.zeros(4, 4096), "probs": torch.zeros(4, 10), "keep": torch.zeros(4, 3, 32, 32)}
    assert first.pass_few(last, x, **good) is not None and native == [1]
    t = good[buf]
    bad = [t.double(), t[:3], t[..., :-1], torch.zeros(8, *t.shape[1:])[::2], torch.zeros(t.shape[::-1]).permute(*range(t.dim())[::-1])]
    for b in bad + ([x, x.view(-1).as_strided(x.shape, x.stride())] if buf == "keep" else []):
        assert first.pass_few(last, x, **{**good, buf: b}) is None, (b.dtype, b.shape, b.stride())
    assert native == [1]


def test_a_sync_behind_every_kernel_needs_every_launch_by_itself(monkeypatch):
    """DNN_DEBUG_SYNC names the launch that a fault is of."""
    from distributed_neural_networks_amd.models.cifar import NeuralNetwork
    from distributed_neural_networks_amd.ops import _lib, cifar as cops
    from distributed_neural_networks_amd.runtime.stages import CifarHipStage
    native = []
    monkeypatch.setattr(cops, "pass_few", lambda *a: native.append(1))
    monkeypatch.setattr(_lib, "DEBUG_SYNC", True)
    sd, cpu = NeuralNetwork().state_dict(), torch.device("cpu")
    pipe = _two(monkeypatch, CifarHipStage(sd, 0, 1, cpu), CifarHipStage(sd, 2, 3, cpu))
    assert pipe.stages[0].pass_few(pipe.stages[1], torch.zeros(2, 3, 32, 32), *pipe.bufs, pipe.x) is None and not native
