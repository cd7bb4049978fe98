"""Kozusun on the GPU kernels against the plain oracle (kozusun_oracle.py)."""
import io
import json
import math
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

import kozusun_oracle as O
from kozusun_cases import CASES, att, config, layer

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
F32_TOL = 2e-5
DT = {"float32": torch.float32, "bf16": torch.bfloat16}


def dev():
    return torch.device("cuda", 0)


def rel(got, ref):
    got, ref = got.double().cpu(), ref.double().cpu()
    return ((got - ref).norm() / ref.norm().clamp_min(1e-30)).item()


def worst_row(got, ref):
    """Largest relative error of a logits row (mean taken off)."""
    d = got.double().cpu() - ref
    d = d - d.mean(-1, keepdim=True)
    r = ref - ref.mean(-1, keepdim=True)
    return (d.norm(dim=-1) / r.norm(dim=-1)).max().item()


# ------------------------------------------------------------------ mechanisms alone
@pytest.mark.parametrize("dtype", ["bf16", "float32"])
@pytest.mark.parametrize("M,width,NP", [(1, 60, 64), (5, 200, 256), (300, 200, 256), (300, 520, 576), (3, 1100, 1152),
                                        (2, 4096, 4096), (2, 9000, 9024)])
def test_rows_update(dtype, M, width, NP):
    from distributed_neural_networks_amd.ops import decoder_ops as D_
    g = torch.Generator().manual_seed(M + NP)
    dt = DT[dtype]

    def mk(m, t):
        z = torch.zeros(m, NP)
        z[:, :width] = torch.randn(m, width, generator=g)
        return z.to(t)
    x, y, tab = mk(M, torch.float32), mk(M, dt), mk(9, dt)
    yw, nw = mk(1, torch.float32)[0], mk(1, torch.float32)[0]
    idx = torch.randint(0, 9, (M,), generator=g, dtype=torch.int32)
    to = lambda t: t.to(dev())  # noqa: E731
    eps, tol = 1e-2, 1e-6 if dt == torch.float32 else 4e-3
    # residual + normalised sublayer output -> residual, copy and the next norm
    xo, cp, h = to(torch.zeros(M, NP)), to(torch.zeros(M, 2 * NP, dtype=dt)), to(torch.zeros(M, NP, dtype=dt))
    D_.rows_update(M, width, x_in=to(x), y=to(y), mult=0.3, y_norm=to(yw), x_out=xo, copy=cp[:, NP:], norm=to(nw), h=h,
                   eps=eps)
    ref = x[:, :width].double() + 0.3 * O.rms_norm(y[:, :width].double(), eps) * yw[:width].double()
    assert rel(xo[:, :width], ref) < 1e-6 and rel(cp[:, NP:NP + width], ref) < tol
    assert rel(h[:, :width], O.rms_norm(ref, eps) * nw[:width].double()) < tol
    assert (cp[:, :NP] == 0).all() and (xo[:, width:] == 0).all() and (h[:, width:] == 0).all()
    # scaled gather (embedding), in place update, gathered norm (head rows)
    D_.rows_update(M, width, y=to(tab), yidx=to(idx), mult=2.5, x_out=xo, copy=cp[:, :NP], eps=eps)
    ref = 2.5 * tab[idx.long(), :width].double()
    assert rel(xo[:, :width], ref) < 1e-6 and rel(cp[:, :width], ref) < tol
    D_.rows_update(M, width, x_in=xo, y=to(y), mult=-1.0, x_out=xo, eps=eps)
    ref = ref - y[:, :width].double()
    assert rel(xo[:, :width], ref) < 1e-6
    rows = torch.arange(M - 1, -1, -1, dtype=torch.int32)
    D_.rows_update(M, width, x_in=xo, xidx=to(rows), norm=to(nw), h=h, eps=eps)
    assert rel(h[:, :width], (O.rms_norm(ref, eps) * nw[:width].double()).flip(0)) < tol


@pytest.mark.parametrize("dtype", ["bf16", "float32"])
@pytest.mark.parametrize("M", [1, 16, 17, 33, 64, 200, 257, 300, 4200])
@pytest.mark.parametrize("n,np_,K", [(25, 64, 64), (64, 64, 192), (130, 192, 448), (256, 256, 2624)])
def test_token_gate(dtype, M, n, np_, K):
    from distributed_neural_networks_amd.ops import decoder_ops as D_
    g = torch.Generator().manual_seed(M + n)
    dt = DT[dtype]
    x, tab = torch.randn(M, K + 64, generator=g).to(dt), torch.randn(11, n + 21, generator=g).to(dt)
    w = torch.zeros(np_, K)
    w[:n] = torch.randn(n, K, generator=g).bfloat16().float() * 2 / math.sqrt(K)
    ids = torch.randint(0, 11, (M,), generator=g, dtype=torch.int32)
    lin = D_.Linear(w, None, dt, dev())
    out = torch.ones(M, np_ + 8, dtype=dt, device=dev())
    D_.token_gate(x.to(dev())[:, :K], lin, tab.to(dev()), 20, ids.to(dev()), out[:, :np_], n,
                  torch.zeros(M, np_, device=dev()) if dtype == "float32" else None)
    ref = O.gelu_tanh(x[:, :K].double() @ lin.w.double().cpu()[:n].t()) * tab[ids.long(), 20:20 + n].double()
    err = ((out[:, :n].double().cpu() - ref).norm(dim=1) / ref.norm(dim=1)).max().item()
    assert err < (3e-6 if dtype == "float32" else 8e-3), err
    assert (out[:, n:np_] == 0).all() and (out[:, np_:] == 1).all()


def test_token_gate_rows_far_apart():
    """Rows whose distance times 64 passes 32 bits (4.9 GB of them), at a size that the tiles would take."""
    from distributed_neural_networks_amd.ops import decoder_ops as D_
    g = torch.Generator().manual_seed(0)
    M, n, K, ld = 70, 60, 64, 35_000_000
    xs, tab = torch.randn(M, K, generator=g).bfloat16(), torch.randn(11, n, generator=g).bfloat16()
    x = torch.empty(M * ld, dtype=torch.bfloat16, device=dev()).as_strided((M, K), (ld, 1))
    x.copy_(xs)
    w, ids = torch.zeros(64, K), torch.randint(0, 11, (M,), generator=g, dtype=torch.int32)
    w[:n] = torch.randn(n, K, generator=g).bfloat16().float() / math.sqrt(K)
    lin, out = D_.Linear(w, None, torch.bfloat16, dev()), torch.empty(M, 64, dtype=torch.bfloat16, device=dev())
    D_.token_gate(x, lin, tab.to(dev()), 0, ids.to(dev()), out, n)
    ref = O.gelu_tanh(xs.double() @ lin.w.double().cpu()[:n].t()) * tab[ids.long()].double()
    assert ((out[:, :n].double().cpu() - ref).norm(dim=1) / ref.norm(dim=1)).max().item() < 8e-3


@pytest.mark.parametrize("M", [64, 65, 500, 2049, 4100])
@pytest.mark.parametrize("n,np_", [(60, 64), (300, 320)])
def test_token_gate_long_rows(M, n, np_):
    """Rows of 4096: the few-row kernel beyond 256 rows and the 64x64 tiles, either side of the rule."""
    test_token_gate("bf16", M, n, np_, 4096)


@pytest.mark.parametrize("M,N,K", [(1, 6, 64), (33, 200, 128), (70, 331, 192), (129, 64, 1024)])
def test_linear_f32(M, N, K):
    from distributed_neural_networks_amd.ops import decoder_ops as D_
    g = torch.Generator().manual_seed(N)
    x, w, b = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g), torch.randn(N, generator=g)
    out = torch.full((M, N + 3), 7.0, device=dev())
    D_.linear_f32(x.to(dev()), w.to(dev()), b.to(dev()), out[:, :N])
    err = rel(out[:, :N], x.double() @ w.double().t() + b.double())
    assert err < 4e-8 * math.sqrt(K) and (out[:, N:] == 7).all()  # fp32 rounding of a K-term running sum


@pytest.mark.parametrize("dtype", ["bf16", "float32"])
@pytest.mark.parametrize("M", [1, 8, 17, 40, 64, 100, 300, 1000])
@pytest.mark.parametrize("F,K", [(192, 128), (1024, 768)])
def test_gated_tanh_gelu(dtype, M, F, K):
    """Packed gate|up projection with the activation in the epilogue, at decode and prefill sizes."""
    from distributed_neural_networks_amd.ops import decoder_ops as D_
    from distributed_neural_networks_amd.ops.gemm import ACT_GELU_TANH_MUL, decode_workspace, pack_gate_up
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).to(DT[dtype])
    gate, up = (torch.randn(F, K, generator=g).bfloat16().float() / math.sqrt(K) * 2 for _ in range(2))
    lin = D_.Linear(pack_gate_up(gate, up), None, DT[dtype], dev(), ACT_GELU_TANH_MUL)
    out = torch.zeros(M, F + 64, dtype=DT[dtype], device=dev())
    lin(x.to(dev()), out[:, 64:], decode_workspace(dev()) if M <= 64 else None,
        torch.zeros(M, 2 * F, device=dev()) if dtype == "float32" else None)
    xd = x.double()
    rd = (lambda t: t.to(DT[dtype]).double())
    ref = O.gelu_tanh(xd @ rd(gate).t()) * (xd @ rd(up).t())
    assert rel(out[:, 64:], ref) < (2e-6 if dtype == "float32" else 5e-3) and (out[:, :64] == 0).all()


def attention_ref(q, k, v, gate, n_new, scale, mask):
    """q (T, H, dk), k (T, G, dk), v (T, G, dv): outputs of the last n_new positions, (n_new, H * dv)."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    ok = O.visible(T, mask)
    outs = [O.masked_softmax(O.attention_scores(q[:, h], k[:, h // (H // G)], scale), ok) @ v[:, h // (H // G)]
            * torch.sigmoid(gate[:, h:h + 1]) for h in range(H)]
    return torch.cat(outs, 1)[-n_new:]


def run_attention(dtype, H, G, dk, dv, scale, mask, seqs, seed=0, standout=None, pages_extra=3):
    """One launch over sequences (cached length, new tokens) whose pages are
    scattered over a pool with garbage in it; ``standout``: {(sequence, key): factor}
    multiplies that key by a copy of the last query.  Returns (got, ref)."""
    from distributed_neural_networks_amd.ops import decoder_ops as D_
    from distributed_neural_networks_amd.runtime.paging import PAGE, PageTable, build_batch, pages_for
    g = torch.Generator().manual_seed(seed)
    dt, R = DT[dtype], H // G
    n_pages = sum(pages_for(a + b) for a, b in seqs) + pages_extra
    table = PageTable(n_pages, len(seqs))
    order = torch.randperm(n_pages, generator=g).tolist()
    table._free_pages = order
    kp = torch.randn(n_pages, G, PAGE, dk, generator=g).to(dt).to(dev()) * 3
    vp = torch.randn(n_pages, G, PAGE, dv, generator=g).to(dt).to(dev()) * 3
    qkv_rows, refs, entries = [], [], []
    for s, (old, new) in enumerate(seqs):
        T = old + new
        q, k, v, gt = (torch.randn(T, n, d, generator=g).to(dt).double()
                       for n, d in ((H, dk), (G, dk), (G, dv), (H, 1)))
        for (sq, key), f in (standout or {}).items():
            if sq == s:
                for c in range(G):
                    k[key, c] = (q[T - 1, c * R] * f / q[T - 1, c * R].norm()).to(dt).double()
        slot = table.admit()
        table.reserve(slot, T)
        for j in range(old):
            p = table.table[slot, j // PAGE]
            kp[p, :, j % PAGE], vp[p, :, j % PAGE] = k[j].to(dt).to(dev()), v[j].to(dt).to(dev())
        qkv_rows.append(torch.cat([t[old:].reshape(new, -1) for t in (q, k, v, gt)], 1))
        refs.append(attention_ref(q, k, v, gt[..., 0], new, scale, mask))
        entries.append(([1] * new, old, slot, []))
    b = build_batch(entries, table.table, [R], dev())
    rows = torch.cat(qkv_rows)
    qkv = torch.zeros(b.M, -(-rows.shape[1] // 16) * 16, dtype=dt)
    qkv[:, :rows.shape[1]] = rows.to(dt)
    out = torch.full((b.M, H * dv + 64), 5.0, dtype=dt, device=dev())
    qkv = qkv.to(dev())  # the arguments hold its address, not the tensor
    args = D_.paged_args(qkv, kp, vp, b.table, b.slots, b.pos, out[:, :H * dv], b.M, H, scale,
                         None if mask is None else mask["size"], 0 if mask is None else mask["keep_first"],
                         (H + G) * dk + G * dv)
    if dtype == "float32":
        D_.paged_write(args, True)
        D_.paged_attn_f32(args)
    else:
        if b.chunks:
            D_.paged_write(args, False)
            D_.paged_prefill(args, b.tiles[R])
        if b.n_dec:
            for splits in (1, 3):
                ws = torch.empty(b.n_dec * H * splits * (dv + 2), device=dev()) if splits > 1 else None
                D_.paged_decode(args, b.dec_rows, b.n_dec, splits, ws)
                if splits == 1:
                    one = out.clone()
            assert rel(out, one) < 5e-3  # split or not, the same attention
    torch.cuda.synchronize()
    assert (out[:, H * dv:] == 5).all()
    # what the launch wrote to the cache
    for (toks, old, slot, _), r in zip(entries, torch.split(rows, [len(e[0]) for e in entries])):
        for t in (0, len(toks) - 1):
            p, o = table.table[slot, (old + t) // PAGE], (old + t) % PAGE
            assert torch.equal(kp[p, :, o].cpu().double().view(-1), r[t, H * dk:(H + G) * dk])
            assert torch.equal(vp[p, :, o].cpu().double().view(-1), r[t, (H + G) * dk:(H + G) * dk + G * dv])
    return out[:, :H * dv].cpu().double(), torch.cat(refs)


SEQS = [(0, 1), (0, 2), (63, 1), (64, 1), (65, 2), (127, 3), (0, 130), (200, 1), (130, 77), (191, 65)]


@pytest.mark.parametrize("dtype", ["bf16", "float32"])
@pytest.mark.parametrize("H,G,dk,dv", [(2, 2, 64, 64), (6, 2, 64, 128), (3, 1, 128, 64), (40, 1, 64, 64),
                                       (2, 1, 256, 256), (4, 4, 128, 128), (5, 1, 64, 256), (2, 2, 256, 64)])
@pytest.mark.parametrize("mask", [None, {"size": 1, "keep_first": 0}, {"size": 50, "keep_first": 3},
                                  {"size": 64, "keep_first": 64}, {"size": 100, "keep_first": 70}])
def test_paged_attention(dtype, H, G, dk, dv, mask):
    got, ref = run_attention(dtype, H, G, dk, dv, 1.2 / math.sqrt(dk), mask, SEQS, seed=H + dk)
    err = ((got - ref).norm(dim=1) / ref.norm(dim=1)).max().item()
    assert err < (2e-6 if dtype == "float32" else 1.5e-2), err


@pytest.mark.parametrize("dtype", ["bf16", "float32"])
@pytest.mark.parametrize("new", [1, 2, 40])
@pytest.mark.parametrize("size,keep", [(32, 5), (64, 0), (65, 64), (90, 17), (128, 33)])
def test_window_edges_stand_out(dtype, new, size, keep):
    """One key that draws nearly all the weight of the last query, just inside
    and just outside the window and the kept keys, and at page borders."""
    T = 300
    last = T - 1
    for key in sorted({last - size + 1, last - size, keep - 1, keep, 0, 63, 64, 127, 128, last, last - 1} - {-1}):
        if key >= T - new and key != last:
            continue
        got, ref = run_attention(dtype, 3, 1, 64, 64, 0.25, {"size": size, "keep_first": keep}, [(T - new, new)],
                                 seed=key, standout={(0, key): 60.0})
        assert rel(got[-1], ref[-1]) < (2e-6 if dtype == "float32" else 1.5e-2), key


# ------------------------------------------------------------------ whole models
_MODELS = {}


def model(name, dtype, num_pages=12, stages=1, max_batch=1, max_seq=768, **kw):
    """(config, oracle weights in float64, stages)"""
    from distributed_neural_networks_amd.models import kozusun
    from distributed_neural_networks_amd.runtime.decoder import DecoderStage
    d = CASES[name]
    if name not in _MODELS:
        W = O.random_weights(d, 11, gain=1.5)
        _MODELS[name] = (W, {k: v.double() for k, v in W.items()})
    W, Wd = _MODELS[name]
    c = kozusun.parse_config(d)
    n = c.n_layer
    cuts = [round(i * n / stages) for i in range(stages + 1)]
    st = []
    for i in range(stages):
        a, b, f, l = cuts[i], cuts[i + 1] - 1, i == 0, i == stages - 1
        sd = {k: W[k] for k in kozusun.stage_key_map(c, a, b, f, l)}
        st.append(DecoderStage(name, sd, a, b, f, l, dev(), max_batch=max_batch, max_seq=max_seq, dtype=dtype,
                               num_pages=num_pages, cfg=c, **kw))
    return d, Wd, st


def engine(name, dtype, **kw):
    from distributed_neural_networks_amd.runtime.engine import Engine
    d, W, st = model(name, dtype, **kw)
    return d, W, Engine(st, max_slots=4)


def tokens(d, n, seed=0):
    return torch.randint(0, d["vocab"], (n,), generator=torch.Generator().manual_seed(seed)).tolist()


_REFS = {}


def reference(name, toks):
    key = (name, tuple(toks))
    if key not in _REFS:
        _REFS[key] = O.forward(torch.tensor(toks), CASES[name], _MODELS[name][1])
    return _REFS[key]


_ROUNDING = {}


def tol(name, dtype):
    """Logits tolerance of a model: fp32 rounding, or three times the error that
    bf16 projections alone make in the oracle."""
    if dtype == "float32":
        return F32_TOL
    if name not in _ROUNDING:
        d, toks = CASES[name], tokens(CASES[name], 210)
        got = O.forward(torch.tensor(toks), d, _MODELS[name][1], rnd=O.bf16)
        _ROUNDING[name] = 3 * worst_row(got, reference(name, toks))
    assert _ROUNDING[name] < 0.2
    return _ROUNDING[name]


def feed(eng, sid, toks, sizes):
    """All logits of one sequence brought in portions of ``sizes`` (the last repeats)."""
    from distributed_neural_networks_amd.runtime.engine import Entry
    out, p, i = [], 0, 0
    while p < len(toks):
        n = min(sizes[min(i, len(sizes) - 1)], len(toks) - p)
        out.append(eng.step([Entry(sid, toks[p:p + n], range(n))]).float().cpu())
        p, i = p + n, i + 1
    return torch.cat(out)


@pytest.mark.parametrize("dtype", ["float32", "bf16"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_portions_match_oracle(name, dtype):
    """The same logits however the prompt is cut: whole, token by token, portions
    of 2, 3, 7, 64, 65, and a prompt followed by long decoding."""
    d, W, eng = engine(name, dtype)
    toks = tokens(d, 210)
    ref = reference(name, toks)
    for i, sizes in enumerate([[210], [1], [2], [3], [7, 1], [64], [65], [63, 1, 66, 2], [20, 1]]):
        got = feed(eng, i, toks, sizes)
        assert worst_row(got, ref) < tol(name, dtype), (sizes, worst_row(got, ref))
        eng.end(i)


@pytest.mark.parametrize("dtype", ["float32", "bf16"])
@pytest.mark.parametrize("name", ["plain", "mixed"])
def test_mixed_batches_and_reused_pages(name, dtype):
    """Unequal sequences together — portions beside single tokens, sequences left
    out of steps, pages and slots given back and used again — against each alone."""
    from distributed_neural_networks_amd.runtime.engine import Entry
    d, W, eng = engine(name, dtype, num_pages=9)
    g = torch.Generator().manual_seed(4)
    lengths = [1, 130, 67, 5, 190, 64, 90, 2, 128, 33]
    seqs = {i: tokens(d, n, 100 + i) for i, n in enumerate(lengths)}
    waiting, live, got, slots_seen = list(seqs), {}, {i: [] for i in seqs}, set()
    from distributed_neural_networks_amd.runtime.paging import pages_for
    while waiting or live:
        while waiting and len(live) < 4 and \
                sum(pages_for(lengths[i]) for i in live) + pages_for(lengths[waiting[0]]) <= 9:
            live[waiting.pop(0)] = 0
        entries = []
        for i, p in live.items():
            r = int(torch.randint(0, 6, (1,), generator=g))
            if r == 0 and len(live) > 1:
                continue  # left out of this step
            n = min([1, 1, 2, 9, 64][r - 1], lengths[i] - p) if r else 1
            entries.append(Entry(i, seqs[i][p:p + n], range(n)))
        if not entries:
            continue
        y = eng.step(entries).float().cpu()
        slots_seen |= {eng.live[e.id].slot for e in entries}
        for e, part in zip(entries, torch.split(y, [len(e.tokens) for e in entries])):
            got[e.id].append(part)
            live[e.id] += len(e.tokens)
            if live[e.id] == lengths[e.id]:
                eng.end(e.id)
                del live[e.id]
    assert slots_seen == {0, 1, 2, 3} and eng.table.free_pages == 9
    for i in seqs:
        err = worst_row(torch.cat(got[i]), reference(name, seqs[i]))
        assert err < tol(name, dtype), (i, lengths[i], err)


def standout_model(far_bias):
    """One attention layer whose score is (almost) one-hot on marked tokens:
    token 1 is the marked key, its value large along one direction."""
    d = config([layer(att(2, 1, 64, 64, 0.125, 80, 6), 64), layer(att(2, 1, 64, 64, 0.125, 80, 6), 64)], 64, 64,
               embed=1.0, mult=1.0)
    W = {k: v for k, v in O.random_weights(d, 3).items()}
    for i in (0, 1):
        W[f"l{i}.mix.q"] *= 0
        W[f"l{i}.mix.q.b"] = torch.ones(128).bfloat16().float() * 4
        mark = torch.zeros(64)
        mark[5] = 1
        W[f"l{i}.mix.k"] = torch.outer(torch.ones(64), mark) * far_bias
        W[f"l{i}.mix.k.b"] *= 0
    W["embed"][:, 5] = 0
    W["embed"][1, 5] = 4
    return d, {k: v.bfloat16().float() for k, v in W.items()}


@pytest.mark.parametrize("dtype", ["float32", "bf16"])
def test_far_key_through_the_model(dtype):
    """A marked token moves through the window's edge, the kept keys' edge and the
    page borders while the model decodes past it: its weight must vanish exactly
    where the mask says."""
    from distributed_neural_networks_amd.models import kozusun
    from distributed_neural_networks_amd.runtime.decoder import DecoderStage
    from distributed_neural_networks_amd.runtime.engine import Engine
    d, W = standout_model(0.5)
    Wd = {k: v.double() for k, v in W.items()}
    c = kozusun.parse_config(d)
    st = DecoderStage("standout", W, 0, 1, True, True, dev(), max_batch=1, max_seq=512, dtype=dtype, num_pages=8, cfg=c)
    eng = Engine([st], max_slots=2)
    base = [t if t != 1 else 2 for t in tokens(d, 300, 9)]
    plain = O.forward(torch.tensor(base), d, Wd)
    for n, key in enumerate([0, 5, 6, 63, 64, 100, 127, 128]):
        toks = list(base)
        toks[key] = 1
        ref = O.forward(torch.tensor(toks), d, Wd)
        bf16_tol = 3 * worst_row(O.forward(torch.tensor(toks), d, Wd, rnd=O.bf16), ref)
        if key == 100:  # the marked key shows while it is in the window, and is gone after two windows
            shift = (ref - plain).norm(dim=1) / plain.norm(dim=1)
            assert shift[101:180].min() > 0.05 and shift[100 + 2 * 79 + 1:].max() < 1e-12
        for sizes in ([300], [70, 1], [64, 2]):
            err = worst_row(feed(eng, n, toks, sizes), ref)
            assert err < (F32_TOL if dtype == "float32" else bf16_tol), (key, sizes, err)
            eng.end(n)


def greedy(name, prompt, steps):
    """Oracle greedy continuation; also the smallest top-2 gap on the way."""
    seq, gap = list(prompt), 1e9
    for _ in range(steps):
        y = O.forward(torch.tensor(seq), CASES[name], _MODELS[name][1])[-1]
        top = y.topk(2).values
        gap = min(gap, ((top[0] - top[1]) / y.std()).item())
        seq.append(int(y.argmax()))
    return seq[len(prompt):], gap


@pytest.mark.parametrize("stages", [1, 2])
@pytest.mark.parametrize("name", ["plain", "mixed"])
def test_greedy_generation(name, stages):
    """Greedy tokens of the oracle from the engine (unequal prompts, queueing,
    several budgets) and from the decode ring (graphs, microbatches, chunks)."""
    from distributed_neural_networks_amd.runtime.engine import Engine
    from distributed_neural_networks_amd.runtime.scheduler import DecodeRing, RingLinks
    d, W, st = model(name, "float32", num_pages=6, stages=stages, max_batch=2, max_seq=96)
    prompts = [tokens(d, n, 40 + n) for n in (1, 66, 30, 2, 5)]
    want, gaps = zip(*(greedy(name, p, 12) for p in prompts))
    assert min(gaps) > 1e-4  # fp32 cannot flip a greedy choice
    eng = Engine(st, max_slots=3)
    for budget in (0, 40, 3):
        assert eng.generate(prompts, 12, budget) == list(want)
    d, W, st = model(name, "float32", num_pages=None, stages=stages, max_batch=4, max_seq=96, max_tokens=160)
    same = [tokens(d, 33, 70 + i) for i in range(4)]
    want = [greedy(name, p, 20)[0] for p in same]
    for M, B, chunk in ((1, 4, 0), (2, 2, 10)):
        ring = DecodeRing(st, RingLinks(), 1, M, B)
        got = ring.generate([torch.tensor(same[m * B:(m + 1) * B]) for m in range(M)], 33, 20, chunk)
        assert got.tolist() == want, (M, B, chunk)


def test_ring_graph_replays_match_eager():
    from distributed_neural_networks_amd.runtime.scheduler import DecodeRing, RingLinks
    d, W, st = model("plain", "bf16", num_pages=None, max_batch=3, max_seq=300)
    prompt = torch.tensor([tokens(d, 70, i) for i in range(3)])
    a = DecodeRing(st, RingLinks(), 1, 1, 3, use_graphs=False).generate([prompt], 70, 200)
    for _ in range(2):
        b = DecodeRing(st, RingLinks(), 1, 1, 3, multi_step=4).generate([prompt], 70, 200)
        assert torch.equal(a, b)


def test_forward_all_positions_and_sampling():
    d, W, st = model("mixed", "bf16", num_pages=None, stages=2, max_batch=2, max_seq=128, temperature=0.8, top_k=20,
                     seed=5)
    toks = torch.tensor([tokens(d, 90, i) for i in (1, 2)])
    h = st[0].forward(toks)
    assert h.shape == (2, 90, st[0].d) and h.dtype == torch.float32
    y = st[1].forward(h.cpu())
    for i in (0, 1):
        assert worst_row(y.probs[i].float(), reference("mixed", toks[i].tolist())) < tol("mixed", "bf16")
    from distributed_neural_networks_amd.runtime.engine import Engine
    eng = Engine(st, max_slots=2)
    p = [t.tolist() for t in toks]
    a = eng.generate(p, 10)
    assert a == eng.generate(p, 10) and all(0 <= t < d["vocab"] for r in a for t in r)  # counter-based: reproducible
    assert a != Engine(model("mixed", "bf16", num_pages=None, stages=2, max_batch=2, max_seq=128)[2],
                       max_slots=2).generate(p, 10)  # not the greedy tokens


def _node_config(tmp_path, folder, parts, **kw):
    cfg = {"nodes": [{"id": f"n{i}", "address": f"127.0.0.1:{50750 + i}", "part_index": i} for i in range(parts)],
           "model_weights": folder, "num_parts": parts, "transport": "colocated", "model": folder, **kw}
    p = tmp_path / "node.json"
    p.write_text(json.dumps(cfg))
    return str(p)


def _run_cli(args, capsys):
    from distributed_neural_networks_amd import cli
    assert cli.main(args) == 0
    text = capsys.readouterr().out
    return json.loads(next(ln for ln in text.splitlines() if "generated tokens:" in ln).split("generated tokens:")[1])


@pytest.mark.parametrize("parts", [1, 3])
def test_cli_generation(tmp_path, capsys, parts):
    """node.py on a model folder: one prompt through the decode ring, several
    unequal ones through the engine; greedy tokens equal the oracle's."""
    d, W, _ = model("plain", "float32")
    O.save_model(str(tmp_path), d, _MODELS["plain"][0])
    prompts = [tokens(d, n, 40 + n) for n in (1, 66, 30)]
    want = [greedy("plain", p, 8)[0] for p in prompts]
    text = [",".join(map(str, p)) for p in prompts]
    cfg = _node_config(tmp_path, str(tmp_path), parts, dtype="float32", decode_steps=8, micro_batch_size=2,
                       prefill_chunk=16)
    assert _run_cli(["--node_id", "n0", "--config", cfg, "--prompt", ";".join(text)], capsys) == want
    assert _run_cli(["--node_id", "n0", "--config", cfg, "--prompt", text[1]], capsys) == [want[1]] * 2


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_trace_runner(tmp_path, dtype):
    """bin/trace_run as a program: a pool of live tokens only, logits per step."""
    d, W, _ = model("mixed", "float32")
    O.save_model(str(tmp_path), d, _MODELS["mixed"][0])
    seqs = {i: tokens(d, n, 7 + i) for i, n in enumerate((70, 64, 100))}
    steps = [([(0, 0, 69), (1, 0, 2)], []), ([(0, 69, 70), (1, 2, 40)], [0]), ([(2, 0, 100), (1, 40, 41)], []),
             ([(1, 41, 64)], [1, 2])]
    lines, refs = [], []
    for n, (parts, end) in enumerate(steps):
        lines.append(json.dumps({"step": n, "end": [f"s{i}" for i in end], "entries": [
            {"id": f"s{i}", "tokens": seqs[i][a:b], "want": list(range(b - a))} for i, a, b in parts]}))
        refs.append(torch.cat([reference("mixed", seqs[i])[a:b] for i, a, b in parts]))
    out = tmp_path / "out"
    r = subprocess.run([os.path.join(ROOT, "bin", "trace_run"), "--model", str(tmp_path), "--dtype", dtype, "--out",
                        str(out), "--max-tokens", "192"], input="\n".join(lines) + "\n", capture_output=True, text=True,
                       timeout=110)
    assert r.returncode == 0, r.stderr[-2000:]
    assert [ln for ln in r.stdout.splitlines() if ln.startswith("done")] == [f"done {n}" for n in range(4)]
    for n, ref in enumerate(refs):
        got = torch.from_numpy(np.fromfile(out / f"{n}.f32", dtype="<f4").reshape(-1, d["vocab"]))
        assert got.shape == ref.shape and worst_row(got, ref) < tol("mixed", "float32" if dtype == "float32" else "bf16")


def test_refusals():
    from distributed_neural_networks_amd.models import kozusun
    from distributed_neural_networks_amd.runtime.decoder import DecoderStage
    from distributed_neural_networks_amd.runtime.engine import Engine
    d, W, st = model("plain", "bf16", num_pages=2, max_seq=64)
    with pytest.raises(ValueError, match="dtype"):
        model("plain", "fp8")
    with pytest.raises(ValueError, match="GPU"):
        DecoderStage("plain", {}, 0, 0, True, False, "cpu", cfg=kozusun.parse_config(d))
    with pytest.raises(ValueError):
        Engine(st, num_pages=3)
    with pytest.raises(ValueError, match="holds"):
        st[0].step(torch.zeros((2, 1), dtype=torch.int32, device=dev()),
                   torch.zeros(2, dtype=torch.int32, device=dev()), 2, 1)


@pytest.mark.parametrize("tokens", [1, 70])
def test_build_batch_does_not_wait_and_keeps_its_own_rows(tokens):
    """Batches built one behind the other while the stream is busy: the host does not
    wait for it, and each arrives with its own ids, positions and wanted rows."""
    from distributed_neural_networks_amd.runtime.paging import PageTable, build_batch
    table = PageTable(16, 4)
    slot = table.admit()
    build_batch([([1] * tokens, 0, slot, [])], table.table, [1], dev())  # the pinned block exists
    a = torch.randn(8192, 8192, device=dev())
    torch.cuda.synchronize()
    for _ in range(20):
        a @ a
    busy = torch.cuda.Event()
    busy.record()
    got = [build_batch([([7 * i + j for j in range(tokens)], 3 * i, slot, [tokens - 1])], table.table, [1], dev())
           for i in range(12)]
    assert not busy.query()
    torch.cuda.synchronize()
    for i, b in enumerate(got):
        assert b.ids.tolist() == [7 * i + j for j in range(tokens)]
        assert b.pos.tolist() == list(range(3 * i, 3 * i + tokens))
        assert b.want_pos.tolist() == [3 * i + tokens - 1] == b.pos[b.want.long()].tolist()
