"""Layers of the paged decoder stages (``runtime/decoder.py``): packed weights,
the caches or states of a layer run, and its launches.

A *layer* holds the weights of one layer of the model; a layer that runs several
times (a loop) has one object and a cache per run (``new_cache``).  It describes
what it needs (``buffers``: scratch columns by name, ``groups``: query heads per
KV head) and adds its launches in ``run``, which reads the normed input from
``st.h`` and leaves the updated residual in ``st.x`` together with what the next
run asks for (``nxt``, keyword arguments of ``rows_update``).

* ``JointLayer`` (Kozusun): attention and feed-forward side by side behind one
  norm, one output projection for both.
* ``SequentialLayer`` (Funepel): a mixer, then a mixture of experts, each behind
  a norm of its own.
  ``Mamba2Mixer``: convolution and state-space recurrence, state by slot.
  ``AttentionRetentionMixer``: paged attention whose values are its keys, and a
  retention state, on the same input, by one projection.
* ``PostNormLayer`` (Tizalorn): a mixer, then a feed-forward, each with a norm on
  its output; the sublayers read the residual itself.
  ``WkvMixer``: mixes with the token before, recurrence with a decay per key
  channel, states by slot.  ``LatentAttentionMixer``: every head over one cached
  latent per token.  ``PolyNormFeedForward``: powers normed over the row.
* ``SandwichLayer`` (Lasizen): a mixer on the shifted norm of the residual, then a
  feed-forward, each with a norm before it and a norm on its output.
  ``DeltaMixer``: convolution and gated delta rule, state by slot.
  ``HeadNormAttentionMixer``: rotation and norm per head, paged attention with a
  sink.  ``XieluFeedForward``: the activation in the projection's epilogue.
* ``MixtureOfExperts``: both routers and expert activations of ``MoEConfig``.
* ``TokenInput``: the per-layer input looked up by token, shared by both.

All padding happens here, once: widths, feed-forward and side sizes to multiples
of 64, attention heads to 64 / 128 / 256, states to 32 / 64 / 128 / 256 x
multiples of 64, with zeros, so kernels see aligned shapes.
"""
from __future__ import annotations

import math
from typing import Dict, List, Optional

import torch

from ..models import funepel, lasizen, tizalorn
from ..ops import decoder_ops as D_
from ..models.decoder_config import MoEConfig
from ..ops import mixer_ops as M_
from ..ops.gemm import ACT_CLAMP_MUL, ACT_GELU_TANH_MUL, ACT_SILU_MUL, ACT_XIELU, pack_gate_up
from .paging import PAGE, LatentHeads, StepBatch


def pad(t: torch.Tensor, *shape: int) -> torch.Tensor:
    """``t`` in the leading corner of a zero tensor of ``shape``."""
    if tuple(t.shape) == shape:
        return t
    out = t.new_zeros(shape)
    out[tuple(slice(0, n) for n in t.shape)] = t
    return out


def pad_heads(w: torch.Tensor, heads: int, dim: int, to: int) -> torch.Tensor:
    """Rows of ``heads`` groups of ``dim`` -> groups of ``to``, zeros between."""
    w = w.reshape(heads, dim, *w.shape[1:])
    return pad(w, heads, to, *w.shape[2:]).reshape(heads * to, *w.shape[2:])


def pad16(n: int) -> int:
    return -(-n // 16) * 16


class Weights:
    """A layer's tensors as padded fp32 on the device, and packed projections."""

    def __init__(self, cfg, prefix: str, sd: Dict[str, torch.Tensor], dtype, device):
        self.cfg, self.prefix, self.sd, self.dtype, self.device = cfg, prefix, sd, dtype, device
        self.width, self.wp = cfg.n_embd, D_.pad64(cfg.n_embd)

    def sub(self, name: str) -> "Weights":
        return Weights(self.cfg, self.prefix + name, self.sd, self.dtype, self.device)

    def __call__(self, name: str) -> torch.Tensor:
        return self.sd[self.prefix + name].to(device=self.device, dtype=torch.float32)

    def has(self, name: str) -> bool:
        return self.prefix + name in self.sd

    def rows(self, name: str, n: int) -> torch.Tensor:
        """A projection from the width: (n padded rows, padded width)."""
        return pad(self(name), n, self.wp)

    def vec(self, name: str) -> torch.Tensor:
        return pad(self(name), self.wp)

    def linear(self, w: torch.Tensor, bias=None, act: int = 0, consts=None) -> D_.Linear:
        return D_.Linear(w, bias, self.dtype, self.device, act, consts=consts)

    def gate_up(self, n: int) -> torch.Tensor:
        return pack_gate_up(self.rows("gate", n), self.rows("up", n))


class TokenInput:
    """y = W_proj (gelu_tanh(W_gate x) * the layer's part of the token's row), RMS-normed."""

    def __init__(self, ld: Weights, i: int, dim: int):
        sp = D_.pad64(dim)
        self.off = i * dim
        self.w_gate, self.w_proj = ld.linear(ld.rows("gate", sp)), ld.linear(pad(ld("proj"), ld.wp, sp))
        self.norm = ld.vec("norm")

    def run(self, st, s: slice, ids, gws, nxt: dict, up) -> None:
        """The residual's copy is in ``st.cat``; the update prepares ``nxt``."""
        x, y = st.x[s], st.y[s]
        D_.token_gate(st.cat[s, :st.wp], self.w_gate, st.side_embed, self.off, ids, st.g[s], st.side, st.z)
        self.w_proj(st.g[s], y, gws)
        up(x_in=x, y=y, mult=st.mult, y_norm=self.norm, x_out=x, **nxt)


def attention_cache(st, heads: int, dk: int, dv: Optional[int]):
    """Key and value page pools (``dv`` None: keys only)."""
    z = lambda d: torch.zeros((st.num_pages, heads, PAGE, d), dtype=st.dtype, device=st.device)  # noqa: E731
    return z(dk), None if dv is None else z(dv)


def run_attention(st, args, b: StepBatch, group: int, splits: int, ws, write: bool = True) -> None:
    """The attention launches of one step: fp32, or bf16 portions and single tokens."""
    if st.f32:
        if write:
            D_.paged_write(args, True)
        D_.paged_attn_f32(args)
        return
    if b.chunks:
        if write:
            D_.paged_write(args, False)
        if b.n_dec:
            D_.paged_mixed(args, b.tiles[group], b.dec_rows, b.n_dec, splits, ws)
        else:
            D_.paged_prefill(args, b.tiles[group])
    elif b.n_dec:
        D_.paged_decode(args, b.dec_rows, b.n_dec, splits, ws)


# ---------------------------------------------------------------------- Kozusun
class JointLayer:
    """Attention and feed-forward on one normed input, one projection for their sum."""

    def __init__(self, cfg, i: int, sd: Dict[str, torch.Tensor], dtype, device):
        ld = Weights(cfg, f"l{i}.", sd, dtype, device)
        L, m, wp = cfg.layers[i], cfg.layers[i].mixer, ld.wp
        self.mix, self.ff = m, L.ff
        self.dk, self.dv = D_.pad_dim(m.dim), D_.pad_dim(m.vdim)
        self.group = m.heads // m.kv_heads
        self.groups = [self.group]
        self.norm1 = pad(1 + ld("norm1"), wp)
        self.norm1[cfg.n_embd:] = 0
        heads = ((m.heads, m.dim, self.dk, "q"), (m.kv_heads, m.dim, self.dk, "k"), (m.kv_heads, m.vdim, self.dv, "v"))
        w = [pad_heads(ld.rows(f"mix.{n}", h * d), h, d, p) for h, d, p, n in heads]
        b = [pad_heads(ld(f"mix.{n}.b"), h, d, p) for h, d, p, n in heads]
        self.gate_col = sum(t.shape[0] for t in w)
        self.n_qkv = pad16(self.gate_col + m.heads)
        self.w_qkv = ld.linear(pad(torch.cat(w + [ld.rows("mix.g", m.heads)]), self.n_qkv, wp),
                               pad(torch.cat(b), self.n_qkv))
        wo = ld("mix.o").view(cfg.n_embd, m.heads, m.vdim)
        outs = [pad(pad(wo, cfg.n_embd, m.heads, self.dv).reshape(cfg.n_embd, -1), wp, m.heads * self.dv)]
        self.n_att, self.n_ff = m.heads * self.dv, 0
        self.w_up = None
        if L.ff is not None:
            self.n_ff = D_.pad64(L.ff)
            self.w_up = ld.linear(ld.sub("mlp.").gate_up(self.n_ff), act=ACT_GELU_TANH_MUL)
            outs.append(pad(ld("mlp.down"), wp, self.n_ff))
        self.w_out = ld.linear(torch.cat(outs, 1))
        self.side = TokenInput(ld.sub("side."), i, cfg.side_dim) if cfg.side_dim else None

    def prep(self, h: torch.Tensor, cache, b: StepBatch) -> dict:
        """What the residual update before a run of this layer also produces."""
        return {"norm": self.norm1, "h": h}

    def buffers(self, f32: bool) -> Dict[str, int]:
        b = {"qkv": self.n_qkv, "af": self.n_att + self.n_ff}
        if f32 and self.n_ff:
            b["gu"] = 2 * self.n_ff
        return b

    def new_cache(self, st):
        return attention_cache(st, self.mix.kv_heads, self.dk, self.dv)

    def splits(self, n: int, keys: int) -> int:
        m = self.mix
        return D_.paged_splits(n, m.heads, m.kv_heads, keys, m.window, m.keep_first)

    def ws_need(self, n: int, keys: int) -> int:
        """fp32 partials the decode launches of ``n`` sequences need."""
        s = self.splits(n, keys)
        return n * self.mix.heads * s * (self.dv + 2) if s > 1 else 0

    def run(self, st, cache, b: StepBatch, ids, s: slice, gws, ws, nxt: dict, up) -> None:
        m, x, h, y, (kp, vp) = self.mix, st.x[s], st.h[s], st.y[s], cache
        qkv, af = st.buf["qkv"][s, :self.n_qkv], st.buf["af"][s, :self.n_att + self.n_ff]
        self.w_qkv(h, qkv, gws)
        if self.w_up is not None:
            self.w_up(h, af[:, self.n_att:], gws, st.buf["gu"][s, :2 * self.n_ff] if st.f32 else None)
        args = D_.paged_args(qkv, kp, vp, b.table, b.slots, b.pos, af[:, :self.n_att], b.M, m.heads, m.scale, m.window,
                             m.keep_first, self.gate_col)
        run_attention(st, args, b, self.group, self.splits(b.n_dec, b.max_len) if b.n_dec else 1, ws)
        self.w_out(af, y, gws)
        if self.side is None:
            up(x_in=x, y=y, mult=st.mult, x_out=x, **nxt)
            return
        up(x_in=x, y=y, mult=st.mult, x_out=x, copy=st.cat[s, :st.wp])
        self.side.run(st, s, ids, gws, nxt, up)


# ---------------------------------------------------------------------- Funepel
class DynamicTanh:
    """tanh(alpha x) * w + b, as keyword arguments of ``rows_update``."""

    def __init__(self, ld: Weights, name: str):
        self.w, self.b, self.alpha = ld.vec(name), ld.vec(name + ".b"), float(ld(name + ".alpha"))

    def prep(self, h: torch.Tensor) -> dict:
        return {"norm": self.w, "norm_b": self.b, "alpha": self.alpha, "h": h}


class Mamba2Mixer:
    """Projection rows [x | B | C | z | dt]: the convolved channels first, heads
    of x padded to multiples of 64 columns, groups of B and C to a state size."""

    def __init__(self, ld: Weights, m: funepel.Mamba2Config):
        self.m, self.groups = m, []
        H, P, N, G = m.heads, m.vdim, m.state, m.groups
        self.np, self.vp = M_.pad_state(N), D_.pad64(P)
        self.C = H * self.vp + 2 * G * self.np
        self.ip = D_.pad64(m.inner)
        self.z_col, self.dt_col = self.C, self.C + self.ip
        self.n_in = pad16(self.dt_col + H)

        def channels(t):  # [x | B | C] rows, padded
            x, B, C = t.split([m.inner, G * N, G * N])
            return torch.cat([pad_heads(x, H, P, self.vp), pad_heads(B, G, N, self.np), pad_heads(C, G, N, self.np)])
        w = pad(ld("in"), m.inner * 2 + 2 * G * N + H, ld.wp)
        z, xbc, dt = w.split([m.inner, m.inner + 2 * G * N, H])
        self.w_in = ld.linear(pad(torch.cat([channels(xbc), pad(z, self.ip, ld.wp), dt]), self.n_in, ld.wp))
        self.conv = M_.ConvWeights(channels(ld("conv")).t().contiguous(), channels(ld("conv.b")).contiguous(),
                                   ld("dt_bias").contiguous(), ld("A_log").contiguous())
        self.D, self.norm = ld("D").contiguous(), ld("norm").contiguous()
        self.w_o = ld.linear(pad(ld("o"), ld.wp, self.ip))
        x1 = H * self.vp
        self.cols = (x1 + G * self.np, x1, 0)  # q = C, k = B, v = x

    def buffers(self, f32: bool) -> Dict[str, int]:
        return {"in": self.n_in, "conv": self.C, "mix": self.ip, "mixn": self.ip, "dt": self.m.heads, "la": self.m.heads}

    def new_cache(self, st):
        return {"ring": torch.zeros((st.num_slots, self.m.conv, self.C), dtype=st.dtype, device=st.device),
                "state": torch.zeros((st.num_slots, self.m.heads, self.vp, self.np), dtype=torch.float32,
                                     device=st.device)}

    def ws_need(self, n: int, keys: int) -> int:
        return 0

    def run(self, st, cache, b: StepBatch, s: slice, gws, ws) -> dict:
        """Returns the mixer's part of the residual update."""
        m, M, B = self.m, b.M, st.buf
        rows = self.w_in(st.h[s], B["in"][s, :self.n_in], gws)
        cv, y, yn = B["conv"][s, :self.C], B["mix"][s, :self.ip], B["mixn"][s, :self.ip]
        dt, la = st.flat("dt", s, m.heads), st.flat("la", s, m.heads)
        M_.conv(rows, self.conv, cache["ring"], cv, dt, la, self.dt_col, b.start, b.slots, b.pos, b.ent,
                len(b.chunks), M)
        M_.scan(cv, self.cols, cache["state"], y, m.vdim, m.heads // m.groups, b.pos, b.ent, len(b.chunks), b.n_dec, M,
                dt=dt, la=la, D=self.D)
        M_.gated_norm(y, rows[:, self.z_col:], yn, M, m.inner, m.norm_groups, st.eps, self.norm, gate_first=True)
        return {"y": self.w_o(yn, st.y[s], gws), "mult": 1.0}


class AttentionRetentionMixer:
    """One projection for both sides: [q | k | attention gate | retention q | k
    | v | gate].  The key norm's weight is folded into the query's, its factor
    per key is kept beside the pages, and the pages hold the keys as projected:
    keys and values share one pool."""

    def __init__(self, ld: Weights, m: funepel.ParallelConfig):
        self.m = m
        a, r = m.left, m.right
        self.dk, self.np, self.vp = D_.pad_dim(a.dim), M_.pad_state(r.dim), D_.pad64(r.vdim)
        self.group = a.heads // a.kv_heads
        self.groups = [self.group]
        self.n_att, self.n_ret = a.heads * self.dk, D_.pad64(r.heads * r.vdim)
        wp, left, right = ld.wp, ld.sub("left."), ld.sub("right.")

        def side(w, name, heads, dim, to):
            return pad_heads(w.rows(name, heads * dim), heads, dim, to)
        parts = [side(left, "q", a.heads, a.dim, self.dk), side(left, "k", a.kv_heads, a.dim, self.dk),
                 side(left, "g", a.heads, a.dim, self.dk), side(right, "q", r.heads, r.dim, self.np),
                 side(right, "k", r.heads, r.dim, self.np), side(right, "v", r.heads, r.vdim, self.vp),
                 right.rows("g", self.n_ret)]
        col = [0]
        for p in parts:
            col.append(col[-1] + p.shape[0])
        self.gate_col, self.cols, self.rg_col = col[2], (col[3], col[4], col[5]), col[6]
        self.n_in = pad16(col[-1])
        self.w_in = ld.linear(pad(torch.cat(parts), self.n_in, wp))
        qn, kn = (pad_heads(left(f"{n}.norm"), h, a.dim, self.dk) for n, h in (("q", a.heads), ("k", a.kv_heads)))
        self.qw = (qn.view(a.kv_heads, self.group, self.dk) * kn.view(a.kv_heads, 1, self.dk)).reshape(-1).contiguous()
        f = dict(dtype=torch.float32, device=ld.device)
        self.slopes = torch.tensor([2.0 ** (-8.0 * (h + 1) / a.heads) for h in range(a.heads)], **f)
        self.la = torch.tensor([max(math.log(d), -88.0) if d > 0 else -88.0 for d in r.decay], **f)
        wo = pad(left("o").view(ld.width, a.heads, a.dim), ld.width, a.heads, self.dk)
        self.w_left = ld.linear(pad(wo.reshape(ld.width, -1), wp, self.n_att))
        self.w_right = ld.linear(pad(right("o"), wp, self.n_ret))
        self.left_out, self.right_out = left.vec("out"), right.vec("out")

    def buffers(self, f32: bool) -> Dict[str, int]:
        return {"in": self.n_in, "mix": max(self.n_att, self.n_ret), "mixn": self.n_ret, "y2": None}

    def new_cache(self, st):
        r = self.m.right
        return {"kp": attention_cache(st, self.m.left.kv_heads, self.dk, None)[0],
                "kscale": torch.zeros((st.num_pages, PAGE), dtype=torch.float32, device=st.device),
                "state": torch.zeros((st.num_slots, r.heads, self.vp, self.np), dtype=torch.float32, device=st.device)}

    def splits(self, n: int, keys: int) -> int:
        a = self.m.left
        return D_.paged_splits(n, a.heads, a.kv_heads, keys, a.window, a.keep_first)

    def ws_need(self, n: int, keys: int) -> int:
        s = self.splits(n, keys)
        return n * self.m.left.heads * s * (self.dk + 2) if s > 1 else 0

    def run(self, st, cache, b: StepBatch, s: slice, gws, ws) -> dict:
        a, r, M, B = self.m.left, self.m.right, b.M, st.buf
        rows = self.w_in(st.h[s], B["in"][s, :self.n_in], gws)
        # retention
        o, on = B["mix"][s, :self.n_ret], B["mixn"][s, :self.n_ret]
        M_.scan(rows, self.cols, cache["state"], o, r.vdim, 1, b.pos, b.ent, len(b.chunks), b.n_dec, M, la_h=self.la,
                dt_c=r.dim ** -0.5)
        M_.gated_norm(o, rows[:, self.rg_col:], on, M, r.heads * r.vdim, r.heads, st.eps)
        y2 = self.w_right(on, B["y2"][s], gws)
        # attention
        M_.qk_norm(rows, cache["kp"], cache["kscale"], self.qw, b.table, b.slots, b.pos, M, a.heads, a.heads * a.dim,
                   a.kv_heads * a.dim, st.eps, a.temp_every, a.temp_coef)
        out = B["mix"][s, :self.n_att]
        args = D_.paged_args(rows, cache["kp"], cache["kp"], b.table, b.slots, b.pos, out, M, a.heads, a.scale, a.window,
                             a.keep_first, self.gate_col, True, cache["kscale"], self.slopes)
        run_attention(st, args, b, self.group, self.splits(b.n_dec, b.max_len) if b.n_dec else 1, ws, write=False)
        y = self.w_left(out, st.y[s], gws)
        return {"y": y, "y_norm": self.left_out, "y2": y2, "y2_norm": self.right_out, "mult": 0.5}


class MixtureOfExperts:
    def __init__(self, ld: Weights, m: MoEConfig):
        self.m, self.fp, self.ep = m, D_.pad64(m.ff), pad16(m.experts)
        self.w_router = ld.linear(ld.rows("router", self.ep))
        experts = [ld.sub(f"e{e}.") for e in range(m.experts)]
        act = (ACT_SILU_MUL, None) if m.limit is None else (ACT_CLAMP_MUL, (m.limit, m.alpha, m.shift))
        self.w_up = M_.ExpertLinear([e.gate_up(self.fp) for e in experts], ld.dtype, ld.device, *act)
        self.routing = {"sigmoid": m.sigmoid, "group_top": m.group_top, "normalise": m.normalise,
                        "correction": ld("correction").contiguous() if m.correction else None}
        self.w_down = M_.ExpertLinear([pad(e("down"), ld.wp, self.fp) for e in experts], ld.dtype, ld.device)
        self.sp = D_.pad64(m.shared_ff) if m.shared_ff else 0
        if self.sp:
            sh = ld.sub("shared.")
            self.w_sup = ld.linear(sh.gate_up(self.sp), act=ACT_SILU_MUL)
            self.w_sdown = ld.linear(pad(sh("down"), ld.wp, self.sp))

    def buffers(self, f32: bool) -> Dict[str, int]:
        b = {"sff": self.sp, "router": self.ep}
        if f32:
            b["gu"] = 2 * self.sp
        return b

    def run(self, st, s: slice, gws) -> dict:
        """Returns the feed-forward's part of the residual update."""
        m, h, B = self.m, st.h[s], st.buf
        r0, M = s.start, s.stop - s.start
        z = self.w_router(h, B["router"][s, :self.ep], gws)
        rt, up, down = st.experts(m.experts, m.top, self.fp)
        M_.route(z, rt, M, m.groups, m.keep, r0, **self.routing)
        e = slice(r0 * m.top, (r0 + M) * m.top)
        gu = up[e, :self.fp]
        self.w_up(h, M * m.top, gu, rt, m.top, r0, st.expert_scratch(2 * self.fp, e) if st.f32 else None, clear=True)
        ys = self.w_down(gu, M * m.top, down[e], rt, 0, r0)
        part = {"ys": ys, "ysi": rt.place[e], "ysw": rt.w[e], "top": m.top, "mult": 1.0}
        if self.sp:
            f = self.w_sup(h, B["sff"][s, :self.sp], gws, B["gu"][s, :2 * self.sp] if st.f32 else None)
            part["y"] = self.w_sdown(f, st.y[s], gws)
        return part


class SequentialLayer:
    """Mixer, then experts, then the token input, each with its own residual update."""

    def __init__(self, cfg, i: int, sd: Dict[str, torch.Tensor], dtype, device):
        ld = Weights(cfg, f"l{i}.", sd, dtype, device)
        L = cfg.layers[i]
        self.norm1 = DynamicTanh(ld, "norm1")
        mixer = Mamba2Mixer if isinstance(L.mixer, funepel.Mamba2Config) else AttentionRetentionMixer
        self.mixer = mixer(ld.sub("mix."), L.mixer)
        self.groups: List[int] = self.mixer.groups
        self.ff = self.norm2 = None
        if L.mlp is not None:
            self.norm2, self.ff = DynamicTanh(ld, "norm2"), MixtureOfExperts(ld.sub("mlp."), L.mlp)
        self.side = TokenInput(ld.sub("side."), i, cfg.side_dim) if cfg.side_dim else None

    def prep(self, h: torch.Tensor, cache, b: StepBatch) -> dict:
        return self.norm1.prep(h)

    def buffers(self, f32: bool) -> Dict[str, int]:
        b = dict(self.mixer.buffers(f32))
        for k, v in (self.ff.buffers(f32) if self.ff else {}).items():
            b[k] = max(b.get(k, 0), v)
        return b

    def new_cache(self, st):
        return self.mixer.new_cache(st)

    def ws_need(self, n: int, keys: int) -> int:
        return self.mixer.ws_need(n, keys)

    def run(self, st, cache, b: StepBatch, ids, s: slice, gws, ws, nxt: dict, up) -> None:
        x = st.x[s]
        last = nxt if self.side is None else {"copy": st.cat[s, :st.wp]}
        part = self.mixer.run(st, cache, b, s, gws, ws)
        if self.ff is None:
            up(x_in=x, x_out=x, **part, **last)
        else:
            up(x_in=x, x_out=x, **part, **self.norm2.prep(st.h[s]))
            part = self.ff.run(st, s, gws)
            up(x_in=x, x_out=x, **part, **last)
        if self.side is not None:
            self.side.run(st, s, ids, gws, nxt, up)


# ---------------------------------------------------------------------- Tizalorn
class ScalarNorm:
    """RMS norm of a sublayer's output times one number, as keyword arguments of ``rows_update``."""

    def __init__(self, ld: Weights, name: str):
        self.w = torch.zeros(ld.wp, dtype=torch.float32, device=ld.device)
        self.w[:ld.width] = ld(name)

    @property
    def joined(self) -> dict:
        """... of the whole sum, where weighted rows join the output."""
        return {"y_norm": self.w, "y_joined": True}

    def of(self, part: dict) -> dict:
        return dict(part, **(self.joined if "ys" in part else {"y_norm": self.w}))


class WkvMixer:
    """r, k, v and the gate in one launch (four projections of operands of their
    own), heads of r, k and v padded to a state size; the decay by way of its
    low-rank projection in fp32."""
    groups: List = []
    reads_copy = False  # it reads the fp32 residual

    def __init__(self, ld: Weights, m: tizalorn.WkvConfig):
        self.m = m
        self.np = max(64, M_.pad_state(m.dim))
        self.n, self.inner, self.ip = m.heads * self.np, m.inner, D_.pad64(m.inner)
        self.mu = torch.stack([ld.vec("mu." + n) for n in "rkvgw"]).contiguous()
        heads = [pad_heads(ld.rows(n, m.inner), m.heads, m.dim, self.np) for n in "rkv"]
        self.w_in = M_.ExpertLinear(heads + [ld.rows("g", self.n)], ld.dtype, ld.device)
        w1, w2 = ld("w1"), ld("w2")
        if w1.shape[0] != w2.shape[1]:
            raise ValueError(f"{ld.prefix}: w1 {tuple(w1.shape)} does not fit w2 {tuple(w2.shape)}")
        self.rank = D_.pad64(w1.shape[0])
        self.w1 = ld.linear(pad(w1, self.rank, ld.wp))
        self.w2 = pad(pad_heads(w2, m.heads, m.dim, self.np), self.n, self.rank).to(ld.dtype).contiguous()
        self.w0 = pad_heads(ld("w0"), m.heads, m.dim, self.np).contiguous()
        self.u = pad(ld("u"), m.heads, self.np).contiguous()
        self.norm = ld("norm").contiguous()
        self.w_o = ld.linear(pad(ld("o"), ld.wp, self.ip))

    def buffers(self, f32: bool) -> Dict[str, int]:
        return {"mixes": 5 * self.mu.shape[1], "rkvg": 4 * self.n, "lowrank": self.rank, "la": self.n, "mix": self.ip,
                "mixn": self.ip}

    def new_cache(self, st):
        f = dict(dtype=torch.float32, device=st.device)
        return {"shift": torch.zeros((st.num_slots, st.wp), **f),
                "state": torch.zeros((st.num_slots, self.m.heads, self.np, self.np), **f)}

    def ws_need(self, n: int, keys: int) -> int:
        return 0

    def run(self, st, cache, b: StepBatch, s: slice, gws, ws) -> dict:
        m, M, B, wp = self.m, b.M, st.buf, st.wp
        mixes = st.flat("mixes", s, 5 * wp).view(5, M, wp)
        M_.token_shift(st.x[s], self.mu, cache["shift"], mixes, b.start, b.last, b.slots, b.pos, M)
        rkvg = self.w_in.each(mixes[:4], st.flat("rkvg", s, 4 * self.n).view(4, M, self.n))
        la = st.flat("la", s, self.n)
        M_.decay(self.w1(mixes[4], B["lowrank"][s, :self.rank], gws), self.w2, self.w0, la, M)
        o, on = B["mix"][s, :self.ip], B["mixn"][s, :self.ip]
        M_.wkv(rkvg, la, self.u, cache["state"], o, m.dim, b.pos, b.ent, len(b.chunks), b.n_dec, M)
        M_.gated_norm(o, rkvg[3], on, M, self.inner, m.heads, st.eps, self.norm)
        return {"y": self.w_o(on, st.y[s], gws), "mult": 1.0}


class LatentAttentionMixer:
    """One projection to [query latent | latent | key part | gate]; the heads'
    query projection to [unrotated | rotated] parts.  Over latents: the key
    projection applied to the query and the value projection to the summed
    latents, both head by head.  Over keys (long portions): both applied to the
    sequence's gathered latents, one projection."""
    reads_copy = True

    def __init__(self, ld: Weights, m: tizalorn.LatentAttentionConfig):
        self.m = m
        H, D, R, V = m.heads, m.dim, m.rot_dim, m.vdim
        self.cp, self.rp = D_.pad_to(m.kv_rank, D_.LATENT_DIMS, "latent size"), D_.pad_to(R, D_.LATENT_ROT, "rotated size")
        self.dp, self.vp, self.qp = D_.pad64(D), D_.pad64(V), D_.pad64(m.q_rank)
        self.hs = self.dp + self.rp
        by_keys = ld.dtype == torch.bfloat16 and self.dp in D_.LATENT_KEYS and self.vp in D_.LATENT_KEYS
        self.tiles = LatentHeads(H, self.cp, self.dp, self.vp, by_keys)
        self.groups: List = [self.tiles]
        kv = ld("dkv")
        parts = [ld.rows("dq", self.qp), pad(kv[:m.kv_rank], self.cp, ld.wp), pad(kv[m.kv_rank:], self.rp, ld.wp),
                 ld.rows("g", H)]
        self.gate_col = self.qp + self.cp + self.rp
        self.n_in = pad16(self.gate_col + H)
        self.w_in = ld.linear(pad(torch.cat(parts), self.n_in, ld.wp))
        self.qw, self.cw = pad(ld("dq.norm"), self.qp).contiguous(), pad(ld("dkv.norm"), self.cp).contiguous()
        uq = ld("uq").view(H, D + R, m.q_rank)
        uq = torch.cat([pad(uq[:, :D], H, self.dp, self.qp), pad(uq[:, D:], H, self.rp, self.qp)], 1)
        self.w_uq = ld.linear(uq.reshape(H * self.hs, self.qp))
        uk, uv = ld("uk").view(H, D, m.kv_rank), ld("uv").view(H, V, m.kv_rank)
        self.w_uk = M_.ExpertLinear([pad(w.t().contiguous(), self.cp, self.dp) for w in uk], ld.dtype, ld.device)
        self.w_uv = M_.ExpertLinear([pad(w, self.vp, self.cp) for w in uv], ld.dtype, ld.device)
        if by_keys:
            ukv = torch.cat([pad(uk, H, self.dp, self.cp), pad(uv, H, self.vp, self.cp)], 1)
            self.w_ukv = ld.linear(ukv.reshape(-1, self.cp))
        self.w_o = ld.linear(pad(pad(ld("o").view(ld.width, H, V), ld.width, H, self.vp).reshape(ld.width, -1), ld.wp,
                                 H * self.vp))
        self.rope = D_.Rope(*m.rot.frequencies(), ld.device)

    def buffers(self, f32: bool) -> Dict[str, int]:
        H = self.m.heads
        return {"in": self.n_in, "q": H * self.hs, "qlat": H * self.cp, "olat": H * self.cp, "mix": H * self.vp}

    def new_cache(self, st):
        return {"kp": torch.zeros((st.num_pages, PAGE, self.cp + self.rp), dtype=st.dtype, device=st.device)}

    def splits(self, n: int, keys: int) -> int:
        return D_.latent_splits(n, self.tiles.per_token, keys)

    def ws_need(self, n: int, keys: int) -> int:
        return D_.latent_ws(n, self.m.heads, self.splits(n, keys), self.cp)

    def run(self, st, cache, b: StepBatch, s: slice, gws, ws) -> dict:
        m, H, M, B, kp, g = self.m, self.m.heads, b.M, st.buf, cache["kp"], self.tiles
        rows = self.w_in(st.h[s], B["in"][s, :self.n_in], gws)
        D_.latent_prep(rows, kp, self.qw, self.cw, self.rope, b.table, b.slots, b.pos, M, m.q_rank, m.kv_rank, self.cp,
                       st.eps)
        q = self.w_uq(rows[:, :self.qp], B["q"][s, :H * self.hs], gws)
        D_.rope_rows(q, M, H, self.hs, self.dp, self.rp, b.pos, self.rope)
        out, gate = B["mix"][s, :H * self.vp], rows[:, self.gate_col:]
        over, ones, keys = (b.tiles.get((g, k)) for k in ("chunks", "ones", "keys"))
        if st.f32 or over is not None or ones is not None:
            heads = lambda t, n: t.unflatten(1, (H, n)).transpose(0, 1)  # noqa: E731  (M, H n) -> (H, M, n)
            qlat, olat = (B[k][s, :H * self.cp] for k in ("qlat", "olat"))
            self.w_uk.each(heads(q, self.hs)[..., :self.dp], heads(qlat, self.cp))
            args = D_.latent_args(qlat, q, self.dp, self.hs, kp, b.table, b.slots, b.pos, olat, M, H, self.cp, m.scale, gate)
            if st.f32:
                D_.latent_attn_f32(args)
            if not st.f32 and over is not None:
                D_.latent_attn(args, over, D_.LATENT_ROWS[1])
            if not st.f32 and ones is not None:
                D_.latent_attn(args, ones, g.rows, self.splits(b.n_dec, b.max_len), g.per_token, ws)
            self.w_uv.each(heads(olat, self.cp), heads(out, self.vp))
        if keys is not None:  # after the others: every row of `out` is written above
            pages = b.tiles[g, "pages"]
            n = pages.shape[0] * PAGE
            lat = st.scratch("latents", n, self.cp + self.rp)
            D_.latent_gather(kp, b.table, pages, lat)
            kv = self.w_ukv(lat[:, :self.cp], st.scratch("keys", n, H * (self.dp + self.vp)))
            D_.latent_prefill(q, kv, lat[:, self.cp:], b.pos, out, M, H, self.dp, self.vp, m.scale, keys, gate)
        return {"y": self.w_o(out, st.y[s], gws), "mult": 1.0}


class PolyNormFeedForward:
    def __init__(self, ld: Weights, m: tizalorn.DenseConfig):
        self.m, self.fp = m, D_.pad64(m.ff)
        self.w_up, self.w_down = ld.linear(ld.rows("up", self.fp)), ld.linear(pad(ld("down"), ld.wp, self.fp))
        self.act = ld("act").contiguous()

    def buffers(self, f32: bool) -> Dict[str, int]:
        return {"ff": self.fp}

    def run(self, st, s: slice, gws) -> dict:
        z = self.w_up(st.h[s], st.buf["ff"][s, :self.fp], gws)
        D_.poly_norm(z, self.act, s.stop - s.start, self.m.ff, st.eps)
        return {"y": self.w_down(z, st.y[s], gws), "mult": 1.0}


class PostNormLayer:
    """x += N(mixer(x)) g1, x += N(feed-forward(x)) g2."""
    side = None

    def __init__(self, cfg, i: int, sd: Dict[str, torch.Tensor], dtype, device):
        ld = Weights(cfg, f"l{i}.", sd, dtype, device)
        L = cfg.layers[i]
        mixer = WkvMixer if isinstance(L.mixer, tizalorn.WkvConfig) else LatentAttentionMixer
        self.mixer, self.norm1 = mixer(ld.sub("mix."), L.mixer), ScalarNorm(ld, "norm1")
        self.groups: List = self.mixer.groups
        self.ff = self.norm2 = None
        if L.mlp is not None:
            ff = PolyNormFeedForward if isinstance(L.mlp, tizalorn.DenseConfig) else MixtureOfExperts
            self.ff, self.norm2 = ff(ld.sub("mlp."), L.mlp), ScalarNorm(ld, "norm2")

    def prep(self, h: torch.Tensor, cache, b: StepBatch) -> dict:
        return {"copy": h} if self.mixer.reads_copy else {}

    def buffers(self, f32: bool) -> Dict[str, int]:
        b = dict(self.mixer.buffers(f32))
        for k, v in (self.ff.buffers(f32) if self.ff else {}).items():
            b[k] = max(b.get(k, 0), v)
        return b

    def new_cache(self, st):
        return self.mixer.new_cache(st)

    def ws_need(self, n: int, keys: int) -> int:
        return self.mixer.ws_need(n, keys)

    def run(self, st, cache, b: StepBatch, ids, s: slice, gws, ws, nxt: dict, up) -> None:
        x = st.x[s]
        part = self.norm1.of(self.mixer.run(st, cache, b, s, gws, ws))
        if self.ff is None:
            up(x_in=x, x_out=x, **part, **nxt)
            return
        up(x_in=x, x_out=x, **part, copy=st.h[s])
        up(x_in=x, x_out=x, **self.norm2.of(self.ff.run(st, s, gws)), **nxt)


# ---------------------------------------------------------------------- Lasizen
class DeltaMixer:
    """Projection rows [q | k | v | gate | b | a]: the convolved channels first,
    heads of q and k padded to a state size, heads of v to multiples of 64."""
    groups: List = []

    def __init__(self, ld: Weights, m: lasizen.DeltaConfig):
        self.m = m
        H, G, self.np, self.vp = m.heads, m.kv_heads, M_.pad_state(m.dim), D_.pad64(m.vdim)
        self.ip = D_.pad64(m.inner)
        heads = (("q", G, m.dim, self.np), ("k", G, m.dim, self.np), ("v", H, m.vdim, self.vp))
        w = torch.cat([pad_heads(ld.rows(n, h * d), h, d, p) for n, h, d, p in heads])
        self.C = w.shape[0]
        self.b_col, self.a_col = self.C + self.ip, self.C + self.ip + H
        self.n_in = pad16(self.a_col + H)
        self.w_in = ld.linear(pad(torch.cat([w, ld.rows("g", self.ip), ld.rows("b", H), ld.rows("a", H)]), self.n_in, ld.wp))
        taps = torch.cat([pad_heads(ld(n + ".conv"), h, d, p) for n, h, d, p in heads])
        self.conv = M_.ConvWeights(taps.t().contiguous(), taps.new_zeros(self.C), ld("dt_bias").contiguous(),
                                   ld("A_log").contiguous())
        self.cols = (0, G * self.np, 2 * G * self.np)
        self.norm = ld("norm").repeat(H).contiguous()
        self.w_o = ld.linear(pad(ld("o"), ld.wp, self.ip))

    def buffers(self, f32: bool) -> Dict[str, int]:
        H = self.m.heads
        return {"in": self.n_in, "conv": self.C, "mix": self.ip, "mixn": self.ip, "dt": H, "la": H}

    def new_cache(self, st):
        m = self.m
        return {"ring": torch.zeros((st.num_slots, m.conv, self.C), dtype=st.dtype, device=st.device),
                "state": torch.zeros((st.num_slots, m.heads, self.vp, self.np), dtype=torch.float32, device=st.device)}

    def ws_need(self, n: int, keys: int) -> int:
        return 0

    def run(self, st, cache, b: StepBatch, s: slice, gws, ws) -> dict:
        m, M, B, H = self.m, b.M, st.buf, self.m.heads
        rows = self.w_in(st.h[s], B["in"][s, :self.n_in], gws)
        cv, y, yn = B["conv"][s, :self.C], B["mix"][s, :self.ip], B["mixn"][s, :self.ip]
        beta, la = st.flat("dt", s, H), st.flat("la", s, H)
        M_.conv(rows, self.conv, cache["ring"], cv, beta, la, self.a_col, b.start, b.slots, b.pos, b.ent, len(b.chunks), M,
                self.b_col)
        M_.delta(cv, self.cols, beta, la, cache["state"], y, m.vdim, H // m.kv_heads, b.pos, b.ent, len(b.chunks), b.n_dec, M,
                 m.dim ** -0.5, lasizen.UNIT_EPS)
        M_.gated_norm(y, rows[:, self.C:], yn, M, m.inner, H, st.eps, self.norm)
        return {"y": self.w_o(yn, st.y[s], gws), "mult": 1.0}


class HeadNormAttentionMixer:
    """One projection [q | k | v]; rotation, norm and cache write in one launch,
    then attention.  The sink is a score of zero per head."""

    def __init__(self, ld: Weights, m: lasizen.AttentionConfig):
        self.m = m
        self.dk, self.dv = D_.pad_dim(m.dim), D_.pad_dim(m.vdim)
        self.group = m.heads // m.kv_heads
        self.groups: List = [self.group]
        heads = (("q", m.heads, m.dim, self.dk), ("k", m.kv_heads, m.dim, self.dk), ("v", m.kv_heads, m.vdim, self.dv))
        w = torch.cat([pad_heads(ld.rows(n, h * d), h, d, p) for n, h, d, p in heads])
        self.n_in, self.n_out = w.shape[0], m.heads * self.dv
        self.w_in = ld.linear(w)
        wo = pad(ld("o").view(ld.width, m.heads, m.vdim), ld.width, m.heads, self.dv)
        self.w_o = ld.linear(pad(wo.reshape(ld.width, -1), ld.wp, self.n_out))
        self.rope = D_.Rope(*(m.rot.frequencies() if m.rot else ([], 1.0)), ld.device)
        self.sinks = torch.zeros(m.heads, dtype=torch.float32, device=ld.device)

    def buffers(self, f32: bool) -> Dict[str, int]:
        return {"in": self.n_in, "mix": self.n_out}

    def new_cache(self, st):
        kp, vp = attention_cache(st, self.m.kv_heads, self.dk, self.dv)
        return {"kp": kp, "vp": vp}

    def splits(self, n: int, keys: int) -> int:
        m = self.m
        return D_.paged_splits(n, m.heads, m.kv_heads, keys, m.window, 0)

    def ws_need(self, n: int, keys: int) -> int:
        s = self.splits(n, keys)
        return n * self.m.heads * s * (self.dv + 2) if s > 1 else 0

    def run(self, st, cache, b: StepBatch, s: slice, gws, ws) -> dict:
        m, M, kp, vp = self.m, b.M, cache["kp"], cache["vp"]
        rows = self.w_in(st.h[s], st.buf["in"][s, :self.n_in], gws)
        D_.qk_heads(rows, kp, vp, self.rope, b.table, b.slots, b.pos, M, m.heads, m.dim, st.eps)
        out = st.buf["mix"][s, :self.n_out]
        args = D_.paged_args(rows, kp, vp, b.table, b.slots, b.pos, out, M, m.heads, m.scale, m.window, 0, sinks=self.sinks,
                             written=True)
        run_attention(st, args, b, self.group, self.splits(b.n_dec, b.max_len) if b.n_dec else 1, ws, write=False)
        return {"y": self.w_o(out, st.y[s], gws), "mult": 1.0}


class XieluFeedForward:
    """W_down act(W_up h); the layer's numbers (p, q) enter as softplus(p) and softplus(q) + 1/2."""

    def __init__(self, ld: Weights, m: lasizen.DenseConfig):
        self.fp = D_.pad64(m.ff)
        c = torch.nn.functional.softplus(ld("act").double(), threshold=1e9) + torch.tensor([0.0, 0.5], device=ld.device)
        self.w_up = ld.linear(ld.rows("up", self.fp), act=ACT_XIELU, consts=c)
        self.w_down = ld.linear(pad(ld("down"), ld.wp, self.fp))

    def buffers(self, f32: bool) -> Dict[str, int]:
        return {"ff": self.fp}

    def run(self, st, s: slice, gws) -> dict:
        z = self.w_up(st.h[s], st.buf["ff"][s, :self.fp], gws)
        return {"y": self.w_down(z, st.y[s], gws), "mult": 1.0}


class SandwichLayer:
    """x += N(mixer(shift(N(x)))), x += N(feed-forward(N(x))).  The update that
    makes the next layer's shifted input reads rows of other threads, so the
    residual goes from ``st.x`` to a second buffer and back."""
    side = None

    def __init__(self, cfg, i: int, sd: Dict[str, torch.Tensor], dtype, device):
        ld = Weights(cfg, f"l{i}.", sd, dtype, device)
        L = cfg.layers[i]
        mixer = DeltaMixer if isinstance(L.mixer, lasizen.DeltaConfig) else HeadNormAttentionMixer
        self.mixer = mixer(ld.sub("mix."), L.mixer)
        self.groups: List = self.mixer.groups
        self.norm1, self.norm1b, self.mu = ld.vec("norm1"), ld.vec("norm1b"), ld.vec("shift")
        self.ff = None
        if L.mlp is not None:
            self.ff, self.norm2, self.norm2b = XieluFeedForward(ld.sub("mlp."), L.mlp), ld.vec("norm2"), ld.vec("norm2b")

    def prep(self, h: torch.Tensor, cache, b: StepBatch) -> dict:
        return {"norm": self.norm1, "h": h, "shift": D_.TokenShift(self.mu, cache["shift"], b.start, b.last, b.slots, b.pos)}

    def buffers(self, f32: bool) -> Dict[str, int]:
        b = dict(self.mixer.buffers(f32), x2=None)
        for k, v in (self.ff.buffers(f32) if self.ff else {}).items():
            b[k] = max(b.get(k, 0), v)
        return b

    def new_cache(self, st):
        return {"shift": torch.zeros((st.num_slots, st.wp), dtype=torch.float32, device=st.device), **self.mixer.new_cache(st)}

    def ws_need(self, n: int, keys: int) -> int:
        return self.mixer.ws_need(n, keys)

    def run(self, st, cache, b: StepBatch, ids, s: slice, gws, ws, nxt: dict, up) -> None:
        x, x2 = st.x[s], st.buf["x2"][s]
        part = self.mixer.run(st, cache, b, s, gws, ws)
        if self.ff is None:
            up(x_in=x, x_out=x2, y_norm=self.norm1b, **part)
            up(x_in=x2, x_out=x, **nxt)
            return
        up(x_in=x, x_out=x2, y_norm=self.norm1b, **part, norm=self.norm2, h=st.h[s])
        part = self.ff.run(st, s, gws)
        up(x_in=x2, x_out=x, y_norm=self.norm2b, **part, **nxt)


LAYERS = {"kozusun": JointLayer, "funepel": SequentialLayer, "tizalorn": PostNormLayer, "lasizen": SandwichLayer}
