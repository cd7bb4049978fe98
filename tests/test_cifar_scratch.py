"""Scratch rows of the fp32 head: what is taken, what is replaced, what is refused (CPU)."""
import pytest
import torch

from distributed_neural_networks_amd.ops import cifar as cops

K3 = 3 * 4096


def test_fc1_scratch():
    cpu = torch.device("cpu")
    own = torch.empty((3, K3), dtype=torch.bfloat16)
    assert cops._fc1_scratch(own, 3, cpu) is own and cops._fc1_scratch(own, 2, cpu) is own
    for other in (None, own[:, :4096], torch.empty((3, 2 * K3), dtype=torch.bfloat16)[:, :K3], own[:2]):
        got = cops._fc1_scratch(other, 3, cpu)
        assert got is not other and got.is_contiguous() and tuple(got.shape) == (3, K3) and got.dtype == torch.bfloat16
    for dt in (torch.uint8, torch.float16, torch.float32):  # the few-row head keeps 16 KB of partial sums a row in it
        with pytest.raises(TypeError):
            cops._fc1_scratch(torch.empty((3, K3), dtype=dt), 3, cpu)


@pytest.fixture
def fc1_calls(monkeypatch):
    """fc1_forward on tensors without memory: what it would launch, with the row distance of the output."""
    calls = []

    class Lib:
        def cifar_fc1_x3(self, a, lda, wh, wl, ldw, bias, c, ldc, *rest):
            calls.append(("fused", ldc, rest[5]))
            return 0

        def cifar_split3(self, *args):
            return 0

        def cifar_head_few(self, *args):
            calls.append(("few", 512, 1))
            return 0

    monkeypatch.setattr(cops, "lib", lambda: Lib())
    monkeypatch.setattr(cops, "stream_ptr", lambda: 0)

    def linear(x, w, bias, act, out):
        calls.append(("gemm", out.stride(0), 1))
        return out

    monkeypatch.setattr(cops, "linear", linear)
    return calls


def _head(device="meta"):
    bf = dict(dtype=torch.bfloat16, device=device)
    return cops.CifarHeadWeights("fp32", w_fc1=torch.empty((512, K3), **bf), w_fc1h=torch.empty((512, 4096), **bf),
                                 w_fc1l=torch.empty((512, 4096), **bf), b_fc1=torch.empty(512, device=device))


@pytest.mark.parametrize("B", [1, 512, 513, 8703, 8704, 9000, 16383, 16400, 65536])
def test_fc1_honours_its_output(B, fc1_calls):
    """Strided rows keep their distance, another type or layout is the GEMM's, on every side of the rules."""
    h, w = torch.empty((B, 4096), device="meta"), _head()
    wide = dict(device="meta")
    rows = {"plain": torch.empty((B, 512), **wide), "wide": torch.empty((B, 520), **wide)[:, :512],
            "odd": torch.empty((B, 517), **wide)[:, :512], "typed": torch.empty((B, 512), dtype=torch.bfloat16, **wide),
            "columns": torch.empty((512, B), **wide).t(), "more": torch.empty((B + 1, 512), **wide)}
    got = {}
    for name, out in rows.items():
        assert cops.fc1_forward(h, w, out=out) is out
        got[name] = fc1_calls.pop()
        assert not fc1_calls
    assert got["plain"][0] == ("few" if B <= 512 else "fused") and got["plain"][1] == 512
    if B > 1:  # one row has no distance
        assert got["wide"][:2] == ("fused" if B >= cops.FC1_X3_MIN_ROWS else "gemm", 520)
        assert got["odd"][:2] == ("gemm", 517) and got["columns"][0] == "gemm"
    assert got["wide"][2] == 1
    assert got["typed"][0] == "gemm" and got["more"][0] == "gemm"


@pytest.mark.parametrize("B", [513, 9000, 16400])
def test_fc1_rows_off_16_bytes(B, fc1_calls, monkeypatch):
    """Rows or weights that 16-byte LDS-DMA does not fetch are the GEMM's, whose split reads them with plain loads."""
    h, w = torch.empty((B, 4096), device="meta"), _head()
    for off in (None, h, w.w_fc1h, w.w_fc1l):
        monkeypatch.setattr(cops, "ptr", lambda t: 4 if t is not None and t is off else 0)
        cops.fc1_forward(h, w)
        assert fc1_calls.pop()[0] == ("fused" if off is None else "gemm")


@pytest.mark.parametrize("B", [1, 512, 513, 1000, 4096, 8703, 8704, 16384, 65536])
def test_fc1_scratch_rows(B, fc1_calls, monkeypatch):
    """What a stage keeps for its head is what the pass takes: nothing is allocated, and of more than
    512 rows no more than the parts of the ranges of K."""
    took = []
    scratch = cops._fc1_scratch
    monkeypatch.setattr(cops, "_fc1_scratch", lambda t, rows, dev: took.append((t, rows)) or scratch(t, rows, dev))
    rows = cops.fc1_scratch_rows(B)
    own = torch.empty((rows, K3), dtype=torch.bfloat16, device="meta") if rows else None
    cops.fc1_forward(torch.empty((B, 4096), device="meta"), _head(), scratch=own)
    assert took == ([(own, rows)] if rows else [])
    if B > 512:
        kind, _, splits = fc1_calls.pop()
        assert kind == "fused" and rows * K3 * 2 < (splits * B * 512 * 4 if splits > 1 else 0) + 2 * K3
