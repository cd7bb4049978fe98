"""Decoder stages with an fp32 residual over paged caches and recurrent states
(the families of ``models.DECODERS``).

A stage runs a range of layer *runs* (a looped layer counts once per pass; every
run has its own cache or state, weights are shared).  What a layer is made of is
in ``runtime/decoder_layers.py``.  One forward pass serves both callers:

* ``step_batch(StepBatch)`` — the engine's step (``runtime/engine.py``): tokens
  of any number of sequences, portions of prompts beside single tokens;
* ``step(x, pos, B, T, b0)`` — ``TransformerStage.step``'s contract for the
  decode ring (``runtime/scheduler.py``): B sequences of T tokens on cache rows
  [b0, b0 + B), each with its own fixed pages, so a decode step is one HIP
  graph whose positions live on the device.

Keys live in pages (``runtime/paging.py``), recurrent states by slot; a portion
that begins at position 0 starts from a zero state.  The residual, norms,
scores, softmax, routers and everything of a recurrence but its projections are
fp32.  ``dtype="float32"`` runs the same sequence with fp32 weights,
activations, cache and matrix products (``ops/decoder_ops.py``).

Stage boundary: rows ``[residual | token id | padding]`` of fp32 (the token id
as its bits): later stages need the tokens for their per-layer inputs, and the
embedding output at a loop's entry.
"""
from __future__ import annotations

import math
from typing import Dict, List, Optional

import torch

from ..models import DECODERS, model_info
from ..ops import decoder_ops as D_
from ..ops import mixer_ops as M_
from ..ops import transformer_ops as T_
from ..ops.gemm import decode_workspace, prefill_workspace
from .decoder_layers import LAYERS, DynamicTanh, ScalarNorm, Weights, pad
from .paging import LatentHeads, StepBatch, pages_for, tile_lists
from .stages import StageCompute, StageOutput

DTYPES = {None: torch.bfloat16, "bf16": torch.bfloat16, "bfloat16": torch.bfloat16, "fp32": torch.float32,
          "float32": torch.float32}
STATES = ("state", "ring", "shift", "prev")  # tensors by slot that a step advances
F32_BUFFERS = ("dt", "la", "router", "lowrank", "x2")
HOP_IDS = 4  # fp32 columns after the residual at a stage boundary: the token id's bits, padding


class DecoderStage(StageCompute):
    act_dtype = torch.float32  # stage-boundary rows

    def __init__(self, model: str, sd: Dict[str, torch.Tensor], start: int, end: int, first: bool, last: bool,
                 device, max_batch: int = 8, max_seq: int = 1024, max_tokens: Optional[int] = None,
                 dtype: Optional[str] = None, temperature: float = 0.0, top_k: int = 0, seed: int = 0,
                 num_pages: Optional[int] = None, cfg=None, num_slots: Optional[int] = None):
        """``max_batch`` x ``max_seq``: the ring's cache rows (and the default
        ``num_pages`` / ``num_slots``).  ``num_pages``: the page pool of an
        engine, ``num_slots``: its sequences' states.  ``max_tokens``: rows of
        one step.  ``cfg`` overrides the registry's configuration."""
        if dtype not in DTYPES:
            raise ValueError(f"dtype {dtype!r}: this model runs in bf16 or float32")
        self.model = model
        self.cfg = c = cfg if cfg is not None else model_info(model).cfg
        self.family = next(f for f, mod in DECODERS.items() if type(c).__module__ == mod.__name__)
        self.start, self.end, self.first, self.last = start, end, first, last
        self.device = dev = torch.device(device)
        if dev.type != "cuda":
            raise ValueError("DecoderStage runs on the GPU kernels only")
        self.dtype = dt = DTYPES[dtype]
        self.f32 = dt == torch.float32
        self.temperature, self.top_k, self.seed = float(temperature), int(top_k), int(seed)
        self.max_batch, self.max_seq = max_batch, max_seq
        self.row_pages = pages_for(max_seq)
        self.num_pages = num_pages or max_batch * self.row_pages
        self.num_slots = max(num_slots or 0, max_batch)
        self.max_tokens = max(max_tokens or max_batch * max_seq, max_batch)
        self.width, self.wp = c.n_embd, D_.pad64(c.n_embd)
        self.V = c.vocab_size
        self.Vpad = D_.pad64(self.V)
        self.eps, self.mult = c.norm_eps, getattr(c, "residual_mult", 1.0)
        self.runs = c.runs[start:end + 1]
        self.side = c.side_dim
        self.enters = any(r.enters for r in self.runs)
        koz, tiz = self.family == "kozusun", self.family == "tizalorn"
        self.entry_projects = koz  # a loop's entry: a projection of [x | x0], or the sum x + x0
        self.embed_mult = getattr(c, "embed_scale", 1.0)

        def table(name, cols):  # gathered rows; columns padded so every row is aligned
            t = sd[name].to(device=dev, dtype=dt)
            return pad(t, t.shape[0], cols).contiguous()
        self.embed = table("embed", self.wp) if (first or self.enters) else None
        self.freq: Optional[torch.Tensor] = None  # sinusoidal position vector: turns per position
        if self.family == "funepel":
            i = torch.arange(-(-self.width // 2), dtype=torch.float64)
            self.freq = (10000.0 ** (-2.0 * i / self.width) / (2.0 * math.pi)).to(dev)
        self.pairs = c.bigram if tiz and first else None  # a table of token pairs joins the embedding, normed
        if self.pairs is not None:
            self.pair_embed = table("bigram", self.wp)
            self.embed_norm = ScalarNorm(Weights(c, "", sd, dt, dev), "embed.norm")
        if self.side:
            self.side_embed = sd["side.embed"].to(device=dev, dtype=dt).contiguous()
        if self.enters and self.entry_projects:
            w = sd["loop.in"].to(device=dev, dtype=torch.float32)
            w = torch.cat([pad(w[:, :self.width], self.wp, self.wp), pad(w[:, self.width:], self.wp, self.wp)], 1)
            self.w_loop = D_.Linear(w, None, dt, dev)
        layers = {i: LAYERS[self.family](c, i, sd, dt, dev) for i in sorted({r.layer for r in self.runs})}
        self.layers: List = [layers[r.layer] for r in self.runs]
        if last:
            ld = Weights(c, "", sd, dt, dev)
            if koz:
                w = pad(1 + ld("final.norm"), self.wp)
                w[self.width:] = 0
                self.final_norm = {"norm": w}
            elif tiz:
                self.final_norm = {"norm": ScalarNorm(ld, "final.norm").w}
            elif self.family == "lasizen":
                self.final_norm = {"norm": ld.vec("final.norm") * c.logit_scale}
            else:
                self.final_norm = DynamicTanh(ld, "final.norm").prep(None)
            self.w_head = ld.linear(ld.rows("head", self.V))
        self.groups = sorted({g for L in self.layers for g in L.groups}, key=str)
        self._alloc()
        self._ring: Dict[tuple, dict] = {}
        self._ring_table: Optional[torch.Tensor] = None
        self._ring_ws: Optional[torch.Tensor] = None

    def _alloc(self):
        dev, dt, n = self.device, self.dtype, self.max_tokens
        z = lambda cols, t=dt: torch.zeros((n, cols), dtype=t, device=dev)  # noqa: E731
        self.x = z(self.wp, torch.float32)
        self.cat = z(2 * self.wp)                     # [residual copy | embedding output]
        self.h, self.y = z(self.wp), z(self.wp)
        # scratch rows by name, as wide as the widest layer asks for
        cols: Dict[str, int] = {}
        for L in self.layers:
            for k, v in L.buffers(self.f32).items():
                cols[k] = max(cols.get(k, 0), self.wp if v is None else v)
        self.buf = {k: z(v, torch.float32 if k in F32_BUFFERS else dt) for k, v in cols.items() if v}
        self._experts: Dict[tuple, M_.Routing] = {}
        self._expert_rows: Dict[str, torch.Tensor] = {}
        self._flat: Dict[str, torch.Tensor] = {}
        if self.side:
            self.g = z(D_.pad64(self.side))
            self.z = z(D_.pad64(self.side)) if self.f32 else None
        if self.enters:
            if self.entry_projects:
                self.y32 = self.y if self.f32 else z(self.wp, torch.float32)
            else:
                self.x0 = z(self.wp, torch.float32)
        if self.pairs is not None:
            self.pair_row = torch.zeros((n,), dtype=torch.int32, device=dev)
            self.ones = torch.ones((n,), dtype=torch.float32, device=dev)
            self.prev = torch.zeros((self.num_slots,), dtype=torch.int32, device=dev)
        if not self.first:
            self.ids_in = torch.zeros((n,), dtype=torch.int32, device=dev)
        self.caches = [L.new_cache(self) for L in self.layers]
        if self.last:
            self.hn = z(self.wp)
            self.logits = torch.zeros((max(self.max_batch, 1), self.Vpad), dtype=dt, device=dev)
            self.next_ids = torch.zeros((max(self.max_batch, 1),), dtype=torch.int32, device=dev)
            self.amx_part = torch.empty((max(self.max_batch, 1) * 2 * T_.ARGMAX_PART_PER_ROW,), dtype=torch.int32,
                                        device=dev)
        self.ws: Optional[torch.Tensor] = None        # decode-attention partials (engine steps)
        widest = max(w.shape[1] for w in (self.h, *self.buf.values()))
        self.pws = None if self.f32 else prefill_workspace(n, widest, dev)  # K splits of steps of more than 64 rows

    def flat(self, name: str, s: slice, cols: int) -> torch.Tensor:
        """Rows ``s`` of a scratch buffer as dense rows of ``cols`` (buffers of
        concurrent microbatches do not overlap: a row has at least ``cols``)."""
        w = self.buf[name].shape[1]
        return self.buf[name].view(-1)[s.start * w:s.start * w + (s.stop - s.start) * cols]

    def experts(self, experts: int, top: int, ff: int):
        """Routing buffers, and the rows of (token, choice) between and after the experts' projections."""
        key, rows = (experts, top), self.max_tokens * top
        if key not in self._experts:
            self._experts[key] = M_.Routing(self.max_tokens, experts, top, self.device)
        return self._experts[key], self._grown("up", rows, ff), self._grown("down", rows, self.wp)

    def expert_scratch(self, cols: int, s: slice) -> torch.Tensor:
        return self._grown("gu", s.stop, cols)[s, :cols]

    def scratch(self, name: str, rows: int, cols: int) -> torch.Tensor:
        """Dense rows that no graph and no concurrent microbatch uses (prefill)."""
        t = self._flat.get(name)
        if t is None or t.numel() < rows * cols:
            t = self._flat[name] = torch.empty((rows * cols,), dtype=self.dtype, device=self.device)
        return t[:rows * cols].view(rows, cols)

    def _grown(self, name: str, rows: int, cols: int) -> torch.Tensor:
        t = self._expert_rows.get(name)
        if t is None or t.shape[0] < rows or t.shape[1] < cols:
            have = (0, 0) if t is None else t.shape
            t = self._expert_rows[name] = torch.zeros((max(rows, have[0]), max(cols, have[1])), dtype=self.dtype,
                                                      device=self.device)
        return t

    # ------------------------------------------------------------------ specs
    @property
    def d(self) -> int:
        """Columns of a stage-boundary row."""
        return self.wp + HOP_IDS

    def in_spec(self, batch: int, T: int = 1):
        return ((batch, T), torch.int32) if self.first else ((batch * T, self.d), torch.float32)

    def out_spec(self, batch: int, T: int = 1):
        return ((batch,), torch.int32) if self.last else ((batch * T, self.d), torch.float32)

    @property
    def fuses_step_tail(self) -> bool:
        """Greedy last stage: the argmax launch writes the next input ids and advances the positions."""
        return self.last and not self.temperature > 0

    def _cache_tensors(self):
        if self.pairs is not None:
            yield "prev", self.prev
        for c in self.caches:
            yield from ((k, t) for k, t in (c.items() if isinstance(c, dict) else zip(("kp", "vp"), c)))

    def reset(self):
        for _, t in self._cache_tensors():
            t.zero_()

    def save_states(self) -> List[torch.Tensor]:
        """Copies of the recurrent states (a step that is run twice advances them twice)."""
        return [t.clone() for k, t in self._cache_tensors() if k in STATES]

    def restore_states(self, saved: List[torch.Tensor]) -> None:
        for t, v in zip((t for k, t in self._cache_tensors() if k in STATES), saved):
            t.copy_(v)

    @property
    def recurrent(self) -> bool:
        return any(k in STATES for k, _ in self._cache_tensors())

    # ------------------------------------------------------------------ layers
    def _prep(self, k: int, r0: int, b: StepBatch) -> dict:
        """What the residual update before run ``k`` also produces."""
        s = slice(r0, r0 + b.M)
        if k == len(self.runs):
            return {}
        if not self.runs[k].enters:
            return self.layers[k].prep(self.h[s], self.caches[k], b)
        if self.entry_projects:
            return {"copy": self.cat[s, :self.wp]}
        return {"x_add": self.x0[s], **self.layers[k].prep(self.h[s], self.caches[k], b)}

    def _ws_need(self, n: int, keys: int) -> int:
        """fp32 partials the decode launches of ``n`` sequences need."""
        return max((L.ws_need(n, keys) for L in self.layers), default=0)

    def _layers(self, b: StepBatch, ids: torch.Tensor, r0: int, gws, ws) -> None:
        """Residual rows [r0, r0 + M) through this stage's runs (``self.x`` holds
        the incoming residual on a later stage)."""
        M, wp, w, s = b.M, self.wp, self.width, slice(r0, r0 + b.M)
        x = self.x[s]
        up = lambda **kw: D_.rows_update(M, w, eps=self.eps, **kw)  # noqa: E731
        emb = {"y": self.embed, "yidx": ids, "mult": self.embed_mult}
        if self.freq is not None:
            emb.update(pos=b.pos, freq=self.freq)
        if self.pairs is not None:
            p, rows = self.pairs, self.pair_row[s]
            M_.pair_rows(ids, self.prev, rows, b.start, b.last, b.slots, b.pos, M, p.mul_prev, p.mul_cur, p.buckets)
            emb.update(ys=self.pair_embed, ysi=rows, ysw=self.ones[s], top=1, **self.embed_norm.joined)
        if not self.enters:
            up(**(dict(emb, x_out=x) if self.first else {"x_in": x}), **self._prep(0, r0, b))
        elif self.entry_projects:  # the embedding output, kept for the loop's passes
            up(**emb, x_out=x if self.first else None, copy=self.cat[s, wp:])
            up(x_in=x, **self._prep(0, r0, b))
        else:
            up(**emb, x_out=self.x0[s])
            up(x_in=self.x0[s] if self.first else x, x_out=x, **self._prep(0, r0, b))
        for k, (run, L) in enumerate(zip(self.runs, self.layers)):
            if run.enters and self.entry_projects:
                up(y=self.w_loop(self.cat[s], self.y32[s], gws), x_out=x, **L.prep(self.h[s], self.caches[k], b))
            L.run(self, self.caches[k], b, ids, s, gws, ws, self._prep(k + 1, r0, b), up)

    def _head(self, r0: int, M: int, rows: torch.Tensor, n: int, logits: torch.Tensor, gws=None) -> torch.Tensor:
        """Logits of ``n`` rows (``rows``: their places among the M of the step)."""
        hn = self.hn[r0:r0 + n]
        D_.rows_update(n, self.width, x_in=self.x[r0:r0 + M], xidx=rows, eps=self.eps, **dict(self.final_norm, h=hn))
        self.w_head(hn, logits[:, :self.V], gws)
        return logits

    # ------------------------------------------------------------------ engine step
    def step_batch(self, b: StepBatch, x: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
        """One step of an engine.  First stage: ``b.ids``; later ones: ``x``, the
        previous stage's rows.  Returns boundary rows, or on the last stage the
        logits of the wanted rows (n_want, V) (None when nothing is wanted)."""
        if b.M > self.max_tokens:
            raise ValueError(f"stage buffers hold {self.max_tokens} tokens, the step brings {b.M}")
        if not self.f32 and b.n_dec:
            need = self._ws_need(b.n_dec, b.max_len)
            if need and (self.ws is None or self.ws.numel() < need):
                self.ws = torch.empty((need,), dtype=torch.float32, device=self.device)
        ids = self._enter(x, b.ids, 0, b.M)
        gws = decode_workspace(self.device) if not self.f32 and b.M <= 64 else None
        self._layers(b, ids, 0, self.pws if gws is None else gws, self.ws)
        if not self.last:
            return self._leave(ids, 0, b.M, None)
        if not b.n_want:
            return None
        lg = torch.empty((b.n_want, self.Vpad), dtype=self.dtype, device=self.device)
        return self._head(0, b.M, b.want, b.n_want, lg, gws if b.n_want <= 64 else None)[:, :self.V]

    def sample(self, logits: torch.Tensor, pos: torch.Tensor) -> torch.Tensor:
        """Next token of every logits row (int32), ``pos``: its position (sampling counter)."""
        n = logits.shape[0]
        out = torch.empty((n,), dtype=torch.int32, device=self.device)
        if self.temperature > 0:
            T_.sample_topk(logits if logits.dtype == torch.bfloat16 else logits.bfloat16(), out, self.V,
                           self.temperature, self.top_k, self.seed, step=pos)
        else:
            T_.argmax_rows(logits, out, n=self.V)
        return out

    def _enter(self, x, ids, r0: int, M: int) -> torch.Tensor:
        """Token ids of the step; a later stage takes the residual from ``x``."""
        if self.first:
            return ids
        if x.dtype != torch.float32 or x.dim() != 2 or x.shape[0] < M or x.shape[1] != self.d:
            raise ValueError(f"stage input {tuple(x.shape)} {x.dtype}: need ({M}, {self.d}) fp32 rows")
        self.x[r0:r0 + M].copy_(x[:M, :self.wp])
        ids_in = self.ids_in[r0:r0 + M]
        ids_in.copy_(x[:M, self.wp:].view(torch.int32)[:, 0])
        return ids_in

    def _leave(self, ids, r0: int, M: int, out: Optional[torch.Tensor]) -> torch.Tensor:
        if out is None:
            out = torch.empty((M, self.d), dtype=torch.float32, device=self.device)
        o = out.view(M, self.d)
        o[:, :self.wp].copy_(self.x[r0:r0 + M])
        o[:, self.wp:].view(torch.int32).copy_(ids.view(M, 1).expand(M, HOP_IDS))
        return out

    # ------------------------------------------------------------------ ring step
    def _tiles(self, chunks, ones, starts=None) -> Dict[object, torch.Tensor]:
        return {k: torch.tensor(v, dtype=torch.int32, device=self.device)
                for k, v in tile_lists(self.groups, chunks, ones, starts).items()}

    def _ring_batch(self, pos: torch.Tensor, B: int, T: int, b0: int) -> StepBatch:
        """B sequences of T tokens on cache rows [b0, b0 + B), each with fixed pages."""
        dev, W = self.device, self.row_pages
        if self._ring_table is None:
            if self.num_pages < self.max_batch * W:
                raise ValueError(f"the page pool ({self.num_pages}) does not hold {self.max_batch} rows of {W} pages")
            self._ring_table = torch.arange(self.max_batch * W, dtype=torch.int32, device=dev).view(self.max_batch, W)
        c = self._ring.get((B, T, b0))
        if c is None:
            slots = torch.arange(b0, b0 + B, dtype=torch.int32, device=dev)
            first = torch.arange(0, B * T, T, dtype=torch.int32, device=dev)
            ent = torch.stack([first, torch.full_like(first, T), slots, torch.zeros_like(first)], 1).contiguous()
            c = {"slots": slots.repeat_interleave(T).contiguous(), "ent": ent,
                 "start": first.repeat_interleave(T).contiguous(),
                 "last": torch.arange(T - 1, B * T, T, dtype=torch.int32, device=dev),
                 "ends": (first + (T - 1)).repeat_interleave(T).contiguous(),
                 "rows": torch.arange(B * T, dtype=torch.int32, device=dev), "chunks": []}
            seqs = [(i * T, T, b0 + i) for i in range(B)]
            if T > 1:
                c["chunks"] = seqs
                c["steps"] = torch.arange(T, dtype=torch.int32, device=dev)
            else:
                c["tiles"] = self._tiles([], seqs)
            self._ring[(B, T, b0)] = c
        p = pos
        if T > 1:
            p = (pos.view(B, 1) + c["steps"]).view(-1).contiguous()
            starts = pos.tolist() if any(isinstance(g, LatentHeads) for g in self.groups) else None
            if c.get("starts", ()) != starts:  # tiles over a latent cache depend on the portions' places
                c["tiles"], c["starts"] = self._tiles(c["chunks"], [], starts), starts
        return StepBatch(M=B * T, pos=p, slots=c["slots"], table=self._ring_table,
                         dec_rows=c["rows"] if T == 1 else None, n_dec=B if T == 1 else 0, chunks=c["chunks"],
                         max_len=self.max_seq, ent=c["ent"], start=c["start"], last=c["ends"], tiles=c["tiles"])

    def step(self, x: torch.Tensor, pos: torch.Tensor, B: int, T: int, b0: int = 0,
             out: Optional[torch.Tensor] = None, last_only: bool = True, advance=None):
        """``TransformerStage.step``'s contract (ids (B, T) on the first stage,
        else boundary rows; ``pos`` (B,) device int32)."""
        if advance is not None and not (self.fuses_step_tail and last_only):
            raise ValueError("step(advance=...) needs a greedy last stage with last_only")
        M, r0 = B * T, b0 if T == 1 else 0
        if r0 + M > self.max_tokens or b0 + B > self.max_batch:
            raise ValueError(f"step of {B} x {T} tokens at row {b0}: the stage holds {self.max_tokens} tokens, "
                             f"{self.max_batch} sequences")
        if self.first and (x.dtype != torch.int32 or tuple(x.shape) != (B, T)):
            raise ValueError(f"first stage expects int32 ids ({B},{T}), got {x.dtype} {tuple(x.shape)}")
        b = self._ring_batch(pos, B, T, b0)
        ws = None
        if T == 1 and not self.f32:
            need = self._ws_need(B, self.max_seq)
            if need:  # one slice per concurrent microbatch
                per = -(-need // B)
                if self._ring_ws is None or self._ring_ws.numel() < per * self.max_batch:
                    self._ring_ws = torch.empty((per * self.max_batch,), dtype=torch.float32, device=self.device)
                ws = self._ring_ws[per * b0:]
        ids = self._enter(x, x.view(-1) if self.first else None, r0, M)
        gws = decode_workspace(self.device, b0 // B) if T == 1 and not self.f32 else None
        self._layers(b, ids, r0, self.pws if gws is None else gws, ws)
        if not self.last:
            return self._leave(ids, r0, M, out)
        c = self._ring[(B, T, b0)]
        if last_only:
            n, rows, q0 = B, c["last"], r0 if T == 1 else b0
            lg, nxt = self.logits[q0:q0 + n], self.next_ids[q0:q0 + n]
        else:
            n, rows = M, c["rows"]
            lg = torch.empty((n, self.Vpad), dtype=self.dtype, device=self.device)
            nxt = torch.empty((n,), dtype=torch.int32, device=self.device)
        self._head(r0, M, rows, n, lg, gws)
        if self.temperature > 0 and last_only:
            T_.sample_topk(lg if not self.f32 else lg.bfloat16(), nxt, self.V, self.temperature, self.top_k, self.seed,
                           step=pos)
            if out is not None:
                out.copy_(nxt)
            return StageOutput(lg[:, :self.V], nxt)
        dst = out if (last_only and out is not None) else nxt
        also, adv, hist = (None, None, None) if advance is None else (tuple(advance) + (None,))[:3]
        part = self.amx_part[q0 * 2 * T_.ARGMAX_PART_PER_ROW:] if last_only and not self.f32 else None
        T_.argmax_rows(lg, dst, n=self.V, also=also, advance=adv, part=part, hist=hist)
        return StageOutput(lg[:, :self.V], dst)

    def forward(self, x: torch.Tensor, out: Optional[torch.Tensor] = None):
        """Full-prefix forward of one request (``TransformerStage.forward``)."""
        B, T = x.shape[0], x.shape[1]
        if B > self.max_batch or T > self.max_seq:
            raise ValueError(f"request (B={B}, T={T}) exceeds the stage cache ({self.max_batch}, {self.max_seq})")
        if self.first:
            h = x.to(device=self.device, dtype=torch.int32).contiguous()
        else:
            h = x.to(device=self.device, dtype=torch.float32).reshape(B * T, self.d).contiguous()
        y = self.step(h, torch.zeros((B,), dtype=torch.int32, device=self.device), B, T, last_only=False)
        if not self.last:
            return y.view(B, T, self.d)
        return StageOutput(y.probs.reshape(B, T, self.V), y.pred.view(B, T)[:, -1].contiguous())
