"""Decode stream GEMM (csrc/kernels/gemm_stream.h): 17..64 rows, fragment-order
weights, A shared through LDS, K split across workgroups into a workspace.
Every variant (bf16 / W8A16 weights, no norm / RMS / LN folded pre-norm,
none / GELU / SwiGLU epilogues, residual, one slice / split-K) against the
fp32 torch reference of the same op, and bit-compared with itself across
workspace sizes where the slicing cannot change the sums' grouping."""
import math

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rel(a, b):
    return ((a.float() - b.float()).norm() / (b.float().norm() + 1e-12)).item()


@pytest.fixture(params=[1, 0], ids=["fold", "reduce"])
def force_stream(request):
    """Forced stream kernel on every eligible shape, however small, split or
    not; split-K combined in the launch (fold) or by the reduce launch."""
    from distributed_neural_networks_amd.ops.gemm import set_stream_gemm
    set_stream_gemm(2, 1, request.param)
    yield
    set_stream_gemm(1, 8 << 20, 0)


@pytest.mark.parametrize("M", [17, 32, 48, 64])
@pytest.mark.parametrize("N,K", [(640, 1024), (3072, 4096), (4096, 1536)])
@pytest.mark.parametrize("split", [False, True])
def test_stream_plain_bias_residual(force_stream, M, N, K, split):
    from distributed_neural_networks_amd.ops.gemm import decode_workspace, linear, shuffle_weight
    torch.manual_seed(M + N)
    x = torch.randn(M, K, device=DEV).bfloat16()
    W = (torch.randn(N, K, device=DEV) / math.sqrt(K)).bfloat16()
    b = torch.randn(N, device=DEV) * 0.1
    R = torch.randn(M, N, device=DEV).bfloat16()
    ref = x.float() @ W.float().t() + b + R.float()
    out = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    ws = decode_workspace(DEV, 7) if split else None
    linear(x, W, b, residual=R, out=out, w_shuf=shuffle_weight(W), ws=ws)
    torch.cuda.synchronize()
    assert _rel(out, ref) < 1e-2, _rel(out, ref)


@pytest.mark.parametrize("M", [24, 64])
@pytest.mark.parametrize("rms,act", [(True, "none"), (True, "silu_mul"), (False, "none"), (False, "gelu")])
@pytest.mark.parametrize("split", [False, True])
def test_stream_folded_norm(force_stream, M, rms, act, split):
    from distributed_neural_networks_amd.ops.gemm import (attach_shuffled, decode_workspace, fold_norm, linear_norm,
                                                          pack_gate_up)
    torch.manual_seed(9)
    K, N = 2048, 2048
    x = (torch.randn(M, K, device=DEV) * 2 + 3.0).bfloat16()  # |mean| >> 0: the LN shift matters
    gamma = torch.rand(K, device=DEV) + 0.5
    beta = None if rms else torch.randn(K, device=DEV) * 0.1
    W = torch.randn(N, K, device=DEV) / math.sqrt(K)
    bias = None if rms else torch.randn(N, device=DEV) * 0.1
    R = torch.randn(M, N, device=DEV).bfloat16() if act == "none" else None
    xf = x.float()
    xn = (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-5) * gamma if rms
          else F.layer_norm(xf, (K,), gamma, beta, 1e-5))
    if act == "silu_mul":
        g, u = W[: N // 2], W[N // 2:]
        Wk = pack_gate_up(g, u)
        ref = F.silu(xn @ g.t()) * (xn @ u.t())
    else:
        Wk = W
        ref = xn @ W.t() + (bias if bias is not None else 0)
        if act == "gelu":
            ref = F.gelu(ref)
    if R is not None:
        ref = ref + R.float()
    f = attach_shuffled(fold_norm(Wk, gamma, beta, bias, rms, 1e-5, DEV))
    out = torch.empty(ref.shape, device=DEV, dtype=torch.bfloat16)
    linear_norm(x, f, act=act, residual=R, out=out, ws=decode_workspace(DEV, 7) if split else None)
    torch.cuda.synchronize()
    assert _rel(out, ref) < 1.5e-2, _rel(out, ref)


@pytest.mark.parametrize("M", [20, 64])
@pytest.mark.parametrize("norm,act", [(0, 0), (2, 2), (1, 3)])
@pytest.mark.parametrize("split", [False, True])
def test_stream_w8(force_stream, M, norm, act, split):
    """Weight-only fp8 (e4m3 weights widened in registers): vs the same algebra
    in fp32 on the dequantised weights."""
    from distributed_neural_networks_amd.ops.fp8 import linear_w8, quantize_weight
    from distributed_neural_networks_amd.ops.gemm import attach_shuffled, decode_workspace, pack_gate_up
    torch.manual_seed(3)
    K, N = 1600, 6400
    x = (torch.randn(M, K, device=DEV) + (1.0 if norm == 2 else 0.0)).bfloat16()
    W = torch.randn(N, K, device=DEV) / math.sqrt(K)
    if act == 3:
        W = pack_gate_up(W[: N // 2], W[N // 2:])
    w8 = attach_shuffled(quantize_weight(W, DEV))
    wd = w8.q[:, :K].float() * w8.scale[:, None]
    xf = x.float()
    colsum = None
    if norm == 2:
        xs = F.layer_norm(xf, (K,), eps=1e-5)
        colsum = wd.sum(1).contiguous()
    elif norm == 1:
        xs = xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-5)
    else:
        xs = xf
    y = xs @ wd.t()
    bias = torch.randn(N, device=DEV) * 0.1 if act == 2 else None
    if act == 2:
        ref = F.gelu(y + bias)
    elif act == 3:
        y = y.view(M, N // 16, 2, 8)
        ref = (F.silu(y[:, :, 0]) * y[:, :, 1]).reshape(M, N // 2)
    else:
        ref = y
    out = torch.empty(ref.shape, device=DEV, dtype=torch.bfloat16)
    linear_w8(x, w8, bias, act, None, out, norm, colsum, 1e-5, ws=decode_workspace(DEV, 7) if split else None)
    torch.cuda.synchronize()
    assert _rel(out, ref) < 1e-2, _rel(out, ref)


def test_stream_matches_skinny_kernel_decode_shapes():
    """Llama-3 8B decode projections (M = 32) on the stream kernel equal the
    skinny kernel's output within bf16 rounding of the differently ordered
    sums, and the fp32 reference."""
    from distributed_neural_networks_amd.ops.gemm import decode_workspace, linear, set_stream_gemm, shuffle_weight
    torch.manual_seed(1)
    M = 32
    for N, K in ((6144, 4096), (4096, 14336)):
        x = torch.randn(M, K, device=DEV).bfloat16()
        W = (torch.randn(N, K, device=DEV) / math.sqrt(K)).bfloat16()
        ws_ = shuffle_weight(W)
        outs = []
        for on in (2, 0):
            set_stream_gemm(on, 8 << 20)
            o = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
            linear(x, W, out=o, w_shuf=ws_, ws=decode_workspace(DEV, 7))
            outs.append(o)
        set_stream_gemm(1, 8 << 20)
        torch.cuda.synchronize()
        ref = x.float() @ W.float().t()
        assert _rel(outs[0], ref) < 1e-2 and _rel(outs[0], outs[1]) < 1e-2


@pytest.mark.parametrize("norm", [0, 1, 2])
def test_stream_fold_matches_reduce_launch(norm):
    """The in-launch split-K combine (last-arriving workgroup per tile, sc1
    hand-off, self-re-arming tickets) gives bit-identical outputs to the
    separate reduce launch, call after call (the tickets must return to zero
    every launch, including when calls alternate between the two forms and
    between shapes with different slice counts)."""
    from distributed_neural_networks_amd.ops.gemm import (attach_shuffled, decode_workspace, fold_norm, linear,
                                                          linear_norm, set_stream_gemm, shuffle_weight)
    torch.manual_seed(norm)
    ws = decode_workspace(DEV, 5)
    outs = {0: [], 1: []}
    try:
        for it in range(3):
            for fold in (1, 0):
                set_stream_gemm(2, 1, fold)
                for (M, N, K) in ((32, 4096, 4096), (64, 1536, 2048)):
                    g = torch.Generator(device=DEV).manual_seed(N + it)
                    x = (torch.randn(M, K, device=DEV, generator=g) + 1).bfloat16()
                    W = torch.randn(N, K, device=DEV, generator=g) / math.sqrt(K)
                    o = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
                    if norm:
                        gamma = torch.rand(K, device=DEV, generator=g) + 0.5
                        f = attach_shuffled(fold_norm(W, gamma, None, None, norm == 1, 1e-5, DEV))
                        linear_norm(x, f, out=o, ws=ws)
                    else:
                        Wb = W.bfloat16()
                        R = torch.randn(M, N, device=DEV, generator=g).bfloat16()
                        linear(x, Wb, residual=R, out=o, w_shuf=shuffle_weight(Wb), ws=ws)
                    outs[fold].append(o)
        torch.cuda.synchronize()
    finally:
        set_stream_gemm(1, 8 << 20, 0)
    for a, b in zip(outs[1], outs[0]):
        assert torch.equal(a, b)
    tickets = ws[-4096:].view(torch.int32)
    assert int(tickets.abs().sum()) == 0  # every ticket re-armed


def _kernels(f):
    """Names of the kernels that ``f`` launches."""
    from torch.profiler import ProfilerActivity, profile
    f()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        f()
        torch.cuda.synchronize()
    return " ".join(e.key for e in p.key_averages())


@pytest.mark.parametrize("M,N,K,w8,form", [(17, 4096, 10240, False, "8, 512>"), (32, 4096, 11008, False, "8, 512>"),
                                           (32, 4096, 14336, False, "8, 256>"), (33, 4096, 10240, False, "8, 256>"),
                                           (17, 8192, 8192, True, "4, 512>"), (64, 4096, 14336, True, "4, 512>"),
                                           (64, 6144, 11008, True, "8, 256>")])
def test_split_forms(M, N, K, w8, form):
    """Waves and bytes of a row a step on both sides of a workgroup a CU, against float64: bf16 storage, and fp32 sums."""
    from distributed_neural_networks_amd.ops.fp8 import linear_w8, quantize_weight
    from distributed_neural_networks_amd.ops.gemm import attach_shuffled, decode_workspace, linear, shuffle_weight
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x, W = torch.randn(M, K, device=DEV, generator=g).bfloat16(), torch.randn(N, K, device=DEV, generator=g) / math.sqrt(K)
    R, out = torch.randn(M, N, device=DEV, generator=g).bfloat16(), torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    ws = decode_workspace(DEV, 7)
    if w8:
        w = attach_shuffled(quantize_weight(W, DEV))
        wd = w.q[:, :K].double() * w.scale.double()[:, None]
        run = lambda: linear_w8(x, w, None, 0, R, out, ws=ws)  # noqa: E731
    else:
        w = W.bfloat16()
        sh, wd = shuffle_weight(w), w.double()
        run = lambda: linear(x, w, residual=R, out=out, w_shuf=sh, ws=ws)  # noqa: E731
    names = _kernels(run)
    assert "gemm_stream_kernel" in names and "gemm_stream_reduce" in names and form in names, names
    ref = x.double() @ wd.t() + R.double()
    size = x.double().abs() @ wd.abs().t()
    assert ((out.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2.0 ** -17 * size).all()


@pytest.mark.parametrize("M,N,K,norm", [(17, 3072, 4096, 0), (64, 3072, 4096, 0), (32, 4096, 4096, 0), (32, 4096, 4096, 1),
                                        (64, 640, 1024, 0), (64, 2048, 2048, 2)])
@pytest.mark.parametrize("what", ["stream", "stream split", "stream fold", "one-shot", "one-shot pinned"])
def test_forced_kernels_run(M, N, K, norm, what):
    """A forced kernel is the one that runs, also for the shapes that kernels of their own are laid out for."""
    from distributed_neural_networks_amd.ops.gemm import (attach_shuffled, decode_workspace, fold_norm, linear, linear_norm,
                                                          set_oneshot_gemm, set_stream_gemm, shuffle_weight)
    g = torch.Generator(device=DEV).manual_seed(N + M)
    x, W = torch.randn(M, K, device=DEV, generator=g).bfloat16(), torch.randn(N, K, device=DEV, generator=g) / math.sqrt(K)
    R, xd = torch.randn(M, N, device=DEV, generator=g).bfloat16(), x.double()
    ws = decode_workspace(DEV, 7) if what != "stream" else None
    if norm:
        f = attach_shuffled(fold_norm(W, torch.ones(K, device=DEV), None, None, norm == 1, 1e-5, DEV))
        run = lambda: linear_norm(x, f, ws=ws)  # noqa: E731
        xd = xd if norm == 1 else xd - xd.mean(-1, keepdim=True)
        ref = xd / (xd.square().mean(-1, keepdim=True) + 1e-5).sqrt() @ W.bfloat16().double().t()
    else:
        Wb = W.bfloat16()
        sh = shuffle_weight(Wb)
        run = lambda: linear(x, Wb, residual=R, w_shuf=sh, ws=ws)  # noqa: E731
        ref = xd @ Wb.double().t() + R.double()
    try:
        if what.startswith("stream"):
            set_stream_gemm(2, 1, int(what == "stream fold"))
        elif what == "one-shot":
            set_oneshot_gemm(2)
        else:
            set_oneshot_gemm(1, 2, 1, 2, -(-K // 2048))
        names, y = _kernels(run), run()
        torch.cuda.synchronize()
    finally:
        set_stream_gemm(1, 8 << 20, 0)
        set_oneshot_gemm(1)
    assert ("gemm_stream_kernel" if what.startswith("stream") else "gemm_oneshot_kernel") in names, names
    if what == "stream split":
        assert "gemm_stream_reduce" in names, names
    # both round a sum of products of unit rows to bf16, which is 2^-9 of it at most; the rest is fp32
    assert ((y.double() - ref).norm() / ref.norm()).item() < 2.0 ** -8


# ---------------------------------------------------------------- one-shot decode GEMM (gemm_oneshot.h)
@pytest.mark.parametrize("M", [17, 32, 64])
@pytest.mark.parametrize("N,K,w8", [(2304, 768, False), (768, 3072, False), (4800, 1600, True), (1600, 6400, True),
                                    (6144, 4096, False), (200, 512, False)])
@pytest.mark.parametrize("epi", ["none", "bias_res", "ln_gelu", "rms_silu", "rms"])
def test_oneshot_matches_skinny(M, N, K, w8, epi):
    """The one-shot kernel (forced on every eligible shape, its planned and
    split-K configurations) against the existing decode path on the same
    fragment-order weights, for every epilogue the decode layers use: bias +
    residual, folded LayerNorm + GELU, folded RMSNorm + packed SwiGLU, folded
    RMSNorm; bf16 and W8A16 weights; partial M and N tiles."""
    from distributed_neural_networks_amd.ops.fp8 import linear_w8, quantize_weight
    from distributed_neural_networks_amd.ops.gemm import (FoldedLinear, decode_workspace, fold_norm, linear,
                                                          linear_norm, set_oneshot_gemm, shuffle_weight)
    if epi == "rms_silu" and N % 16:
        pytest.skip("packed gate|up needs N % 16 == 0")
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(M * 7 + N)
    x = (torch.randn(M, K, device=dev, generator=g) * 2 + 0.5).bfloat16()
    w = torch.randn(N, K, device=dev, generator=g) / K ** 0.5
    bias = torch.randn(N, device=dev, generator=g) if epi == "bias_res" else None
    res = torch.randn(M, N, device=dev, generator=g).bfloat16() if epi == "bias_res" else None
    ws = decode_workspace(dev)

    def run():
        if epi in ("ln_gelu", "rms_silu", "rms"):
            gam = torch.rand(K, device=dev, generator=g) + 0.5
            rms = epi != "ln_gelu"
            beta = None if rms else torch.randn(K, device=dev, generator=g) * 0.1
            f = fold_norm(w, gam, beta, None, rms, 1e-5, dev, w8)
            from distributed_neural_networks_amd.ops.gemm import attach_shuffled
            attach_shuffled(f)
            act = {"ln_gelu": "gelu", "rms_silu": "silu_mul", "rms": None}[epi]
            return linear_norm(x, f, act=act, ws=ws)
        if w8:
            q = quantize_weight(w, dev)
            q.shuf = shuffle_weight(q.q[:, :K])
            return linear_w8(x, q, bias, 0, res, ws=ws)
        return linear(x, w.bfloat16(), bias, None, res, w_shuf=shuffle_weight(w.bfloat16()), ws=ws)

    try:
        set_oneshot_gemm(0)
        g.manual_seed(M * 7 + N + 1)
        ref = run().float()
        set_oneshot_gemm(2)
        g.manual_seed(M * 7 + N + 1)
        got = run().float()
        torch.cuda.synchronize()
    finally:
        set_oneshot_gemm(1)
    err = ((got - ref).norm() / ref.norm()).item()
    assert err < 1e-2, err


@pytest.mark.parametrize("cfg", [(1, 1, 1, 1), (1, 4, 2, 3), (2, 2, 1, 2), (2, 4, 2, 1), (4, 1, 1, 1), (4, 4, 1, 4)])
def test_oneshot_pinned_configs(cfg):
    """Every (rows/16, column tiles, LDS steps, split-K) configuration the
    sweep explores computes the same product (W8A16 and bf16)."""
    from distributed_neural_networks_amd.ops._lib import lib, ptr, stream_ptr
    from distributed_neural_networks_amd.ops.fp8 import quantize_weight
    from distributed_neural_networks_amd.ops.gemm import decode_workspace, shuffle_weight
    dev = torch.device("cuda", 0)
    mt, ntw, steps, sk = cfg
    ws = decode_workspace(dev)
    for w8, (N, K) in ((False, (1000, 2048)), (True, (4800, 1600))):
        M = {1: 17, 2: 33, 4: 50}[mt]  # partial m-groups
        x = torch.randn(M, K, device=dev).bfloat16()
        w = torch.randn(N, K, device=dev)
        if w8:
            q = quantize_weight(w, dev)
            wsh, sw = shuffle_weight(q.q[:, :K]), q.scale
            wref = q.q[:, :K].float() * q.scale[:, None]
        else:
            wsh, sw = shuffle_weight(w.bfloat16()), None
            wref = w.bfloat16().float()
        out = torch.zeros(M, N, device=dev, dtype=torch.bfloat16)
        rc = lib().gemm_oneshot_sweep(ptr(x), K, ptr(wsh), ptr(sw), ptr(out), N, M, N, K, mt, ntw, steps, sk, int(w8),
                                      ptr(ws), ws.numel(), stream_ptr())
        if rc == -1:
            continue  # the config does not cover this K in one slice
        assert rc == 0
        torch.cuda.synchronize()
        ref = x.float() @ wref.T
        assert ((out.float() - ref).norm() / ref.norm()).item() < 1e-2, (cfg, w8)


@pytest.mark.parametrize("path", ["oneshot", "skinny"])
@pytest.mark.parametrize("N,K,w8", [(2304, 768, False), (768, 3072, False), (4800, 1600, True), (1600, 6400, True)])
@pytest.mark.parametrize("epi", ["bias_res", "ln_gelu"])
def test_epilogue_prefetch_bit_identical(path, N, K, w8, epi):
    """Epilogue operands issued with the first loads (gemm_oneshot.h /
    gemm_skinny_kernel ``pre``, the default) change when the channel scales,
    column sums, bias and residual arrive, not the operations: the prefetching
    launch is bit-identical from run to run (a first version let the activation
    image be read before its DMA landed, which showed only as run-to-run
    differences) and matches the late-load epilogue (``gemm_set_epi_prefetch(0)``)
    up to the compiler's mul-add contraction of the split-K combine (a
    straight-line scale-and-bias fuses into one fma: a bf16 step in a handful
    of the 102 400 outputs of the 1600 x 6400 shape, bias_res_w8 in
    profiles/r5_epi_prefetch_determinism.jsonl).  Every recorded call follows
    a launch on other activations (the LDS holds other bytes), which is what
    exposed the image-sync race (gemm_oneshot.h "Retiring the image")."""
    from distributed_neural_networks_amd.ops._lib import lib
    from distributed_neural_networks_amd.ops.fp8 import linear_w8, quantize_weight
    from distributed_neural_networks_amd.ops.gemm import (attach_shuffled, decode_workspace, fold_norm, linear,
                                                          linear_norm, set_oneshot_gemm, shuffle_weight)
    dev = torch.device("cuda", 0)
    M = 64
    g = torch.Generator(device=dev).manual_seed(N + K)
    x = (torch.randn(M, K, device=dev, generator=g) * 2 + 0.5).bfloat16()
    w = torch.randn(N, K, device=dev, generator=g) / K ** 0.5
    bias = torch.randn(N, device=dev, generator=g)
    res = torch.randn(M, N, device=dev, generator=g).bfloat16()
    ws = decode_workspace(dev)
    if epi == "ln_gelu":
        f = fold_norm(w, torch.rand(K, device=dev, generator=g) + 0.5, torch.randn(K, device=dev, generator=g) * 0.1,
                      bias, False, 1e-5, dev, w8)
        attach_shuffled(f)
        run = lambda a=x: linear_norm(a, f, act="gelu", ws=ws)  # noqa: E731
    elif w8:
        q = quantize_weight(w, dev)
        q.shuf = shuffle_weight(q.q[:, :K])
        run = lambda a=x: linear_w8(a, q, bias, 0, res, ws=ws)  # noqa: E731
    else:
        wb = w.bfloat16()
        wsh = shuffle_weight(wb)
        run = lambda a=x: linear(a, wb, bias, None, res, w_shuf=wsh, ws=ws)  # noqa: E731
    # each recorded call follows a launch on other activations, so an image read
    # before its LDS-DMA landed sees different stale bytes (bench/probes/epi_race_screen.py)
    x2 = (torch.randn(M, K, device=dev, generator=g) * 3 - 1.0).bfloat16()
    outs = []
    try:
        set_oneshot_gemm(2 if path == "oneshot" else 0)
        for on in (0, 1, 1, 1, 0):
            lib().gemm_set_epi_prefetch(on)
            run(x2)
            outs.append(run().clone())
        torch.cuda.synchronize()
    finally:
        lib().gemm_set_epi_prefetch(1)
        set_oneshot_gemm(1)

    def where(u, v):
        d = (u.float() - v.float()).abs()
        i = int(d.argmax())
        return (f"max {d.max().item()} at {divmod(i, N)} ({u.view(-1)[i].item()} vs {v.view(-1)[i].item()}), "
                f"{int((d > 0).sum())} differ")
    assert torch.equal(outs[0], outs[4]), "late-load epilogue not deterministic: " + where(outs[0], outs[4])
    for o in outs[2:4]:
        assert torch.equal(outs[1], o), "prefetching epilogue not deterministic: " + where(outs[1], o)
    a, b = outs[0].float(), outs[1].float()
    step = torch.maximum(torch.maximum(a.abs(), b.abs()), torch.full_like(b, 2.0 ** -126)) * 2.0 ** -7
    assert bool(((a - b).abs() <= step).all()), "on vs off: " + where(a, b)
    assert (a != b).float().mean().item() < 1e-3


@pytest.mark.parametrize("N,floor_kb", [(3072, 0), (2304, 0), (3072, 72)])
def test_oneshot_coresident_race_screen(N, floor_kb):
    """Regression: the forced one-shot LN + GELU grid with
    TWO workgroups per CU (LDS floor 0, or a 72 KB floor: padded but still two
    per CU), every call after a poisoning call on other activations, bit-
    identical to the settled reference in all 3000 calls.  The SLP build of
    the same kernel differed in ~1-2 % of these calls (one element of a row
    statistic summed unshifted in lanes 48-63, gemm_oneshot.h "The race of
    rounds 5-6"); tests/test_isa_lds_dma_order.py pins the build side (no
    cross-half packed FP32 in the product kernels)."""
    from distributed_neural_networks_amd.ops._lib import lib
    from distributed_neural_networks_amd.ops.gemm import (attach_shuffled, decode_workspace, fold_norm, linear_norm,
                                                          set_oneshot_gemm)
    dev = torch.device("cuda", 0)
    M, K = 64, 768
    g = torch.Generator(device=dev).manual_seed(N + K)
    x = (torch.randn(M, K, device=dev, generator=g) * 2 + 0.5).bfloat16()
    w = torch.randn(N, K, device=dev, generator=g) / K ** 0.5
    bias = torch.randn(N, device=dev, generator=g)
    x2 = (torch.randn(M, K, device=dev, generator=g) * 3 - 1.0).bfloat16()
    ws = decode_workspace(dev)
    f = fold_norm(w, torch.rand(K, device=dev, generator=g) + 0.5, torch.randn(K, device=dev, generator=g) * 0.1,
                  bias, False, 1e-5, dev, False)
    attach_shuffled(f)
    out = torch.empty((M, N), dtype=torch.bfloat16, device=dev)
    counts = {}
    try:
        set_oneshot_gemm(2, 2, 1, 1, 1)  # forced 2/1/1: N / 16 x 2 workgroups (> 256 CUs)
        lib().gemm_set_oneshot_lds_floor(floor_kb * 1024)
        assert lib().gemm_set_oneshot_probe(0, 0) == 0
        linear_norm(x, f, act="gelu", ws=ws, out=out)
        ref = linear_norm(x, f, act="gelu", ws=ws, out=out).clone()
        bad = 0
        for _ in range(3000):
            linear_norm(x2, f, act="gelu", ws=ws, out=out)
            o = linear_norm(x, f, act="gelu", ws=ws, out=out)
            bad += int(not torch.equal(o, ref))
        counts["product"] = bad
    finally:
        lib().gemm_set_oneshot_probe(0, 0)
        lib().gemm_set_oneshot_lds_floor(0)  # the library default
        set_oneshot_gemm(1)
    print(f"N={N} floor={floor_kb} KB: mismatched calls of 3000: {counts}")
    assert counts["product"] == 0, counts


@pytest.mark.parametrize("M", [17, 31, 33, 64])
@pytest.mark.parametrize("N,K", [(16, 64), (112, 192), (128, 576), (240, 4096), (2064, 320), (28672, 256)])
def test_stream_gated_seven_waves(force_stream, M, N, K):
    """Gate and up behind an RMS norm as tiles of 112 columns (seven waves): columns and K that no tile or step divides,
    nothing written past the rows, every value to the roundings."""
    from distributed_neural_networks_amd.ops.gemm import attach_shuffled, fold_norm, linear_norm, pack_gate_up
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn(M, K, device=DEV, generator=g).bfloat16()
    gate, up = (torch.randn(N // 2, K, device=DEV, generator=g) / math.sqrt(K) for _ in range(2))
    gamma = torch.rand(K, device=DEV, generator=g) + 0.5
    f = attach_shuffled(fold_norm(pack_gate_up(gate, up), gamma, None, None, True, 1e-5, DEV))
    out = torch.full((M + 1, N // 2 + 8), 5.0, device=DEV, dtype=torch.bfloat16)
    linear_norm(x, f, act="silu_mul", out=out[:M, :N // 2])
    assert (out[M] == 5).all() and (out[:, N // 2:] == 5).all()
    xd = x.double()
    w = f.w.double().view(N // 16, 2, 8, K)
    r = xd * torch.rsqrt((xd * xd).mean(1, keepdim=True) + 1e-5)
    zg, zu = (r @ w[:, i].reshape(-1, K).t() for i in (0, 1))
    ref = zg * torch.sigmoid(zg) * zu
    # one rounding to bf16; fp32 sums of K products of size about |r| |w|: 1e-5 of either factor, silu's slope is under 1.1
    size = [(r.abs() @ w[:, i].reshape(-1, K).abs().t()) for i in (0, 1)]
    bound = 2.0 ** -8 * ref.abs() + 1e-5 * (1.1 * size[0] * zu.abs() + size[1] * (zg * torch.sigmoid(zg)).abs()) + 1e-6
    assert ((out[:M, :N // 2].double() - ref).abs() <= bound).all()
