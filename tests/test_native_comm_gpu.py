"""Native RCCL data plane (csrc/comm/p2p.cpp, parallel/rccl.py) on one GPU.

A 1-rank loopback channel exercises the whole module on the 1-GPU box —
communicator bootstrap, the transfer stream and its ordering after the
caller's stream, completion tokens, HIP graph capture of a hop, counters —
and a 2-process pair channel on the same GPU runs the real pair bootstrap
through the TCP store (RCCL may refuse two ranks on one device; that refusal
must then surface as a clean init error, not a hang).  Cross-GPU hops over
xGMI run in the multi-GPU bench.
"""
import os
import socket
import subprocess
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def ch():
    from distributed_neural_networks_amd.parallel import rccl
    assert rccl.available(), "librccl did not resolve"
    c = rccl.loopback(torch.device("cuda", 0)).ready(60)
    yield c


@pytest.mark.parametrize("nbytes", [4, 16384, (3 << 20) + 7])
def test_loopback_roundtrip(ch, nbytes):
    from distributed_neural_networks_amd.parallel.rccl import RECV, SEND, Work
    dev = torch.device("cuda", 0)
    src = torch.randint(0, 256, (nbytes,), dtype=torch.uint8, device=dev)
    dst = torch.zeros_like(src)
    tok = ch.group([(SEND, src, 0), (RECV, dst, 0)])
    Work(ch, tok).wait()  # device-side: the check below runs after the transfer
    assert torch.equal(dst, src)
    ch.synchronize(tok, 30)
    assert ch.query(tok)


def test_loopback_ordered_after_producer(ch):
    """The transfer reads its buffer only after the work queued before the
    post (a long producer chain on the current stream)."""
    from distributed_neural_networks_amd.parallel.rccl import RECV, SEND, Work
    dev = torch.device("cuda", 0)
    a = torch.randn(2048, 2048, device=dev)
    src = torch.zeros(2048, 2048, device=dev)
    for _ in range(8):
        src = src + a @ a.T * 1e-3  # ~ms of queued work before the post
    final = src.clone()
    dst = torch.empty_like(src)
    w = Work(ch, ch.group([(SEND, src, 0), (RECV, dst, 0)]))
    w.wait()
    assert torch.equal(dst, final)


def test_loopback_graph_capture(ch):
    """A hop captured with the kernels around it replays as graph nodes."""
    from distributed_neural_networks_amd.parallel.rccl import RECV, SEND
    dev = torch.device("cuda", 0)
    x = torch.zeros(4096, device=dev)
    y = torch.empty_like(x)
    dst = torch.empty_like(x)
    out = torch.empty_like(x)
    s = torch.cuda.Stream(dev)
    s.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(s):  # warm the RCCL kernels outside the capture
        torch.mul(x, 2, out=y)
        ch.group([(SEND, y, 0), (RECV, dst, 0)], on_stream=True)
    torch.cuda.current_stream(dev).wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        torch.mul(x, 2, out=y)
        ch.group([(SEND, y, 0), (RECV, dst, 0)], on_stream=True)
        torch.add(dst, 1, out=out)
    for v in (1.0, -3.5, 7.25):
        x.fill_(v)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, torch.full_like(x, 2 * v + 1))


def test_loopback_token_ring_wraps(ch):
    """More ops than the channel's completion ring (1024) in one go."""
    from distributed_neural_networks_amd.parallel.rccl import RECV, SEND
    dev = torch.device("cuda", 0)
    src = torch.arange(256, device=dev, dtype=torch.int32)
    dst = torch.zeros_like(src)
    tok = 0
    for i in range(1100):
        tok = ch.group([(SEND, src, 0), (RECV, dst, 0)])
    ch.synchronize(tok, 60)
    assert torch.equal(dst, src)
    st = ch.stats()
    assert st["sent_msgs"] >= 1100 and st["recv_bytes"] >= 1100 * 1024


def test_post_validates(ch):
    from distributed_neural_networks_amd.parallel.rccl import SEND
    dev = torch.device("cuda", 0)
    t = torch.zeros(8, device=dev)
    with pytest.raises(RuntimeError, match="out of range"):
        ch.post(SEND, t, 1)
    with pytest.raises(ValueError):
        ch.post(SEND, torch.zeros(4, 4, device=dev).t(), 0)


def _free_port() -> int:
    with socket.socket() as s:
        s.bind(("127.0.0.1", 0))
        return s.getsockname()[1]


def _pair_results(tmp_path):
    port = str(_free_port())
    outs = [str(tmp_path / f"r{r}.txt") for r in range(2)]
    env = dict(os.environ, PYTHONPATH=ROOT)
    procs = [subprocess.Popen([sys.executable, "-u", os.path.join(ROOT, "tests", "rccl_pair_worker.py"), str(r), port,
                               outs[r]], env=env, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
             for r in range(2)]
    logs = []
    try:
        for p in procs:
            logs.append(p.communicate(timeout=150)[0].decode(errors="replace")[-2000:])
    finally:
        for p in procs:
            if p.poll() is None:
                p.kill()
    res = [open(o).read().strip() if os.path.exists(o) else "missing" for o in outs]
    print("pair channel results:", res)
    return res, logs


def test_pair_channel_two_processes(tmp_path):
    """Two processes, a pair channel bootstrapped through the TCP store,
    six messages up to 6 MiB each way, every byte checked.  On a 1-GPU box
    RCCL refuses two ranks on one device: that is reported as a SKIP (the
    data path did not run), never as a pass."""
    res, logs = _pair_results(tmp_path)
    assert all(r.startswith(("ok", "init_error")) for r in res), (res, logs)
    if any(r.startswith("init_error") for r in res):
        assert torch.cuda.device_count() < 2, (res, logs)  # with two GPUs the pair must work
        pytest.skip(f"RCCL refused the pair on one device: {res}")
    assert res == ["ok 0", "ok 0"], res  # both receivers got exactly the senders' bytes


def test_native_preflight_two_processes(tmp_path):
    """links.native_preflight on a 2-rank nccl group sharing GPU 0: RCCL
    refuses the pair, both ranks agree through the TCP store to fall back to
    ProcessGroupNCCL P2P (DNN_P2P=torch) with the failing rank's message
    (or, where RCCL accepts the pair, both report native)."""
    port = str(_free_port())
    outs = [str(tmp_path / f"p{r}.txt") for r in range(2)]
    env = dict(os.environ, PYTHONPATH=ROOT)
    env.pop("DNN_P2P", None)
    procs = [subprocess.Popen([sys.executable, "-u", os.path.join(ROOT, "tests", "preflight_worker.py"), str(r), port,
                               outs[r]], env=env, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
             for r in range(2)]
    logs = []
    try:
        for p in procs:
            logs.append(p.communicate(timeout=150)[0].decode(errors="replace")[-2000:])
    finally:
        for p in procs:
            if p.poll() is None:
                p.kill()
    res = [open(o).read().strip() if os.path.exists(o) else "missing" for o in outs]
    print("preflight results:", res)
    modes = [r.split("|")[0] for r in res]
    assert modes[0] == modes[1], (res, logs)
    if modes[0] == "native":
        assert all(r.endswith("|native") for r in res), res
    else:
        assert modes[0].startswith("torch (native preflight failed: rank"), (res, logs)
        assert all(r.endswith("|torch") for r in res), res
