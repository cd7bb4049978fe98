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
