"""Rows of 1024, 2048 and 4096 in bf16, a workgroup each with nothing but the asked parts: equal to the general kernel
(which takes more rows than 2048) bit for bit where both add in one order, and to fp64 within the roundings."""
import pytest
import torch

pytestmark = pytest.mark.gpu

FORMS = ["table", "table-last", "join", "join-norm", "join-copy", "y-norm", "y-norm-norm", "y-norm-copy", "rows", "rows-in-place"]


@pytest.mark.parametrize("NP,N", [(1024, 1000), (1024, 1024), (2048, 2048), (4096, 4096), (4096, 3997)])
@pytest.mark.parametrize("form", FORMS)
def test_rows_lean(form, NP, N):
    from distributed_neural_networks_amd.ops import decoder_ops as D_

    g = torch.Generator().manual_seed(NP + N + FORMS.index(form))
    R = 2049
    cols = torch.arange(NP) < N

    def noise(rows, std=1.0):
        return (torch.randn(rows, NP, generator=g) * std * cols).cuda()

    x, y = noise(R + 3), noise(R + 3, 3.0).bfloat16()
    yw, nw = noise(1)[0], noise(1)[0]
    idx = torch.randint(0, R + 3, (R,), generator=g).int()
    idx[0], idx[1] = -5, R + 9  # clamped
    at = idx.long().clamp(0, R + 2)
    idx = idx.cuda()

    def call(M):
        out = {k: torch.full((M + 1, NP), 7.0, device="cuda", dtype=d) for k, d in
               (("x_out", torch.float32), ("copy", torch.bfloat16), ("h", torch.bfloat16))}
        kw = {k: v[:M] for k, v in out.items()}
        use = set()
        if form.startswith("table"):
            kw.update(y=y, yidx=idx[-M:] if form == "table-last" else idx[:M], mult=1.7)
            use = {"x_out", "h"}
        elif form.startswith("rows"):
            kw.update(x_in=x if form == "rows" else x[:M], xidx=idx[:M] if form == "rows" else None)
            use = {"h"}
        else:
            kw.update(x_in=x[:M], y=y[:M], mult=0.6)
            if form.startswith("y-norm"):
                kw["y_norm"] = yw
            use = {"x_out"} | ({"copy"} if form.endswith("copy") else {"h"} if form in ("join-norm", "y-norm-norm") else set())
        if "h" in use:
            kw["norm"] = nw
        kw = {k: v for k, v in kw.items() if k not in out or k in use}
        D_.rows_update(M, N, eps=1e-5, **kw)
        for k, v in out.items():
            assert (v[M:] == 7).all() and (k in use or (v == 7).all())
        return {k: out[k][:M] for k in use}

    whole = call(R)  # more rows than one launch has workgroups for: the general kernel
    for M in (1, 5, 2048):
        got = call(M)
        for k, v in got.items():
            if NP > 1024 and form != "table-last":
                assert torch.equal(v, whole[k][:M]), (k, M)
        xd, yd = x.double().cpu(), y.double().cpu()
        if form.startswith("table"):
            z = 1.7 * yd[at[-M:] if form == "table-last" else at[:M]]
        elif form.startswith("rows"):
            z = xd[at[:M]] if form == "rows" else xd[:M]
        else:
            z = yd[:M]
            if form.startswith("y-norm"):
                z = z * torch.rsqrt((z * z).sum(1, keepdim=True) / N + 1e-5) * yw.double().cpu()
            z = xd[:M] + 0.6 * z
        # fp32 sums of <= 16 terms a thread and six steps over the wave, twice: under 1e-5; a bf16 result another 2^-8
        want = {"x_out": z, "copy": z, "h": z * torch.rsqrt((z * z).sum(1, keepdim=True) / N + 1e-5) * nw.double().cpu()}
        for k, v in got.items():
            tol = 1e-5 if k == "x_out" else 2.0 ** -8 + 1e-5
            err = (v.double().cpu() - want[k]).abs()
            assert (err <= tol * want[k].abs() + 2e-5).all(), (k, M, err.max())


@pytest.mark.parametrize("NP,N", [(1024, 1000), (2048, 2048), (4096, 3997), (4096, 4096)])
@pytest.mark.parametrize("form", ["table", "join", "y-norm"])
@pytest.mark.parametrize("lengths", [(1,), (1, 1, 1, 1, 1), (3, 1, 250, 2), (1, 640, 7, 1399, 1)])
def test_rows_shift(form, NP, N, lengths):
    """The token shift, a workgroup a row: as the general kernel (more than 2048 rows) forms the same sequences, bit for bit
    where both add in one order, fp64 otherwise; the states of fresh and going sequences before and after."""
    from distributed_neural_networks_amd.ops import decoder_ops as D_

    g = torch.Generator().manual_seed(NP + N + len(lengths) + len(form))
    cols = torch.arange(NP) < N
    M, S = sum(lengths), len(lengths)
    assert M <= 2048
    R = M + 2049

    def noise(rows, std=1.0):
        return (torch.randn(rows, NP, generator=g) * std * cols).cuda()

    x, y, state0 = noise(R), noise(R, 3.0).bfloat16(), noise(S + 3)
    yw, nw, mu = noise(1)[0], noise(1)[0], noise(1)[0]
    ids = torch.randint(-2, R + 2, (R,), generator=g).int().cuda()  # clamped
    slots = torch.randperm(S + 1, generator=g)[:S]
    rows = [torch.zeros(R, dtype=torch.int32) for _ in range(4)]  # first, last row, slot, position
    at = 0
    for i, n in enumerate(list(lengths) + [R - M]):
        slot, p0 = (slots[i].item(), 0 if i % 2 else 40 + i) if i < S else (S + 2, 5)
        for t, v in zip(rows, (at, at + n - 1, slot, p0)):
            t[at:at + n] = v
        rows[3][at:at + n] += torch.arange(n, dtype=torch.int32)
        at += n
    rows = [t.cuda() for t in rows]

    def call(M):
        xo, h = torch.full((M + 1, NP), 7.0, device="cuda"), torch.full((M + 1, NP), 7.0, device="cuda", dtype=torch.bfloat16)
        state = state0.clone()
        kw = dict(y=y, yidx=ids[:M], mult=1.7) if form == "table" else dict(x_in=x[:M], y=y[:M], mult=0.6)
        D_.rows_update(M, N, x_out=xo[:M], norm=nw, h=h[:M], y_norm=yw if form == "y-norm" else None, eps=1e-5,
                       shift=D_.TokenShift(mu, state, *(t[:M].contiguous() for t in rows)), **kw)
        assert (xo[M:] == 7).all() and (h[M:] == 7).all()
        return xo[:M], h[:M], state

    whole, got = call(R), call(M)
    assert torch.equal(got[2][S + 1:], state0[S + 1:])
    if NP > 1024:
        for a, b in zip(got[:2], whole[:2]):
            assert torch.equal(a, b[:M])
        assert torch.equal(got[2][:S + 1], whole[2][:S + 1])
    xd, yd = x.double().cpu(), y.double().cpu()
    if form == "table":
        z = 1.7 * yd[ids[:M].long().clamp(0, R - 1).cpu()]
    else:
        z = yd[:M]
        if form == "y-norm":
            z = z * torch.rsqrt((z * z).sum(1, keepdim=True) / N + 1e-5) * yw.double().cpu()
        z = xd[:M] + 0.6 * z
    hn = z * torch.rsqrt((z * z).sum(1, keepdim=True) / N + 1e-5) * nw.double().cpu()
    prev, want_state, at = torch.cat([hn[:1], hn[:-1]]), state0.double().cpu(), 0
    for i, n in enumerate(lengths):
        prev[at] = 0 if i % 2 else want_state[slots[i]]
        at += n
    at = 0
    for i, n in enumerate(lengths):
        at += n
        want_state[slots[i]] = hn[at - 1]
    want = hn + (prev - hn) * mu.double().cpu()
    # as above; the shift is one more rounding of values up to |prev| + |h|
    assert ((got[0].double().cpu() - z).abs() <= 1e-5 * z.abs() + 2e-5).all()
    assert ((got[2].double().cpu() - want_state).abs() <= 1e-5 * want_state.abs() + 2e-5).all()
    size = hn.abs() + (prev.abs() + hn.abs()) * mu.double().cpu().abs()
    assert ((got[1].double().cpu() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5 * size + 2e-5).all()
