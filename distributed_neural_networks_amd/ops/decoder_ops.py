"""Wrappers of the decoder kernels with an fp32 residual and a paged KV cache
(``csrc/kernels/residual_rows.hip``, ``token_gate.hip``, ``gemm_f32.hip``,
``paged_attention.hip``, ``qk_norm.hip``, ``latent_attention.hip``, ``poly_norm.hip``).

Operands are bf16 (serving) or fp32 (exact mode: fp32 weights, activations,
cache and MFMA); the residual stream is fp32 in both.  As in
``transformer_ops``, every shape is validated on the host before a launch.
"""
from __future__ import annotations

from typing import Optional

import torch

from . import gemm as G_
from ._lib import check, lib, ptr, stream_ptr

PAGE = 64                      # keys per cache page (paged_attention.hip PG)
HEAD_DIMS = (64, 128, 256)     # head sizes the kernels are built for; others are zero-padded up
TILE_ROWS = 128                # packed (token, head) rows of one prefill workgroup
NO_WINDOW = (1 << 31) - 1
WIDTH_MAX = 16384


def pad_dim(d: int) -> int:
    """Head size a ``d``-wide head is stored at."""
    for p in HEAD_DIMS:
        if d <= p:
            return p
    raise ValueError(f"head size {d} exceeds {HEAD_DIMS[-1]}")


def pad64(n: int) -> int:
    return -(-n // 64) * 64


def _rows(t: Optional[torch.Tensor], M: int, N: int, name: str, dtypes) -> None:
    if t is None:
        return
    if t.dim() != 2 or t.shape[0] < M or t.shape[1] < N or t.stride(1) != 1 or t.dtype not in dtypes:
        raise ValueError(f"{name}: need >= ({M}, {N}) rows of {dtypes}, got {tuple(t.shape)} {t.dtype} "
                         f"strides {t.stride()}")


def _index(t: Optional[torch.Tensor], M: int, name: str) -> None:
    if t is not None and (t.dtype != torch.int32 or t.numel() < M or not t.is_contiguous()):
        raise ValueError(f"{name}: contiguous int32 with >= {M} entries expected")


def _weight(t: Optional[torch.Tensor], N: int, name: str) -> None:
    if t is not None and (t.dtype != torch.float32 or t.numel() < N or not t.is_contiguous()):
        raise ValueError(f"{name}: contiguous fp32 with >= {N} entries expected")


def rows_update(M: int, width: int, *, x_in: Optional[torch.Tensor] = None, xidx: Optional[torch.Tensor] = None,
                y: Optional[torch.Tensor] = None, yidx: Optional[torch.Tensor] = None, mult: float = 1.0,
                y_norm: Optional[torch.Tensor] = None, y2: Optional[torch.Tensor] = None,
                y2_norm: Optional[torch.Tensor] = None, ys: Optional[torch.Tensor] = None,
                ysi: Optional[torch.Tensor] = None, ysw: Optional[torch.Tensor] = None, top: int = 0, y_joined: bool = False,
                x_add: Optional[torch.Tensor] = None, pos: Optional[torch.Tensor] = None,
                freq: Optional[torch.Tensor] = None, x_out: Optional[torch.Tensor] = None,
                copy: Optional[torch.Tensor] = None, norm: Optional[torch.Tensor] = None,
                norm_b: Optional[torch.Tensor] = None, alpha: float = 0.0, h: Optional[torch.Tensor] = None,
                shift=None, eps: float = 1e-5) -> None:
    """``x' = [x_in] [+ x_add] [+ positions] + mult * z`` with ``z = y`` (RMS-
    normalised with weight ``y_norm`` first, if given) ``[+ y2`` normalised with
    ``y2_norm] [+ sum_t ysw[m, t] ys[ysi[m, t]]]`` (``y_joined``: ``y_norm`` norms
    ``y`` with that sum instead), then any of ``x_out = x'``
    (fp32), ``copy = x'`` and ``h = RMSnorm(x') * norm``, or with ``norm_b`` the
    dynamic tanh ``h = tanh(alpha x') * norm + norm_b``.  ``xidx`` / ``yidx``
    gather the rows of ``x_in`` / ``y``; positions: sinusoids of ``pos`` with
    ``freq`` (fp64, turns per position; even columns sine, odd cosine).  Rows are
    zero-padded to a multiple of 4; means are over ``width``.  ``shift``
    (``TokenShift``, RMS norm only): ``h + (h of the sequence's token before - h) *
    mu`` instead of ``h``; ``x_out`` must not be ``x_in`` then."""
    f32, bf = torch.float32, torch.bfloat16
    out = copy if copy is not None else h
    yt = next((t for t in (y, y2, ys) if t is not None), None)
    od = out.dtype if out is not None else (yt.dtype if yt is not None else f32)
    NP = next(t.shape[1] for t in (x_out, x_in, y) if t is not None)
    _rows(x_in, 1 if xidx is not None else M, NP, "rows_update x_in", (f32,))
    _rows(x_out, M, NP, "rows_update x_out", (f32,))
    _rows(x_add, M, NP, "rows_update x_add", (f32,))
    _rows(y, 1 if yidx is not None else M, NP, "rows_update y", (f32, bf))
    _rows(y2, M, NP, "rows_update y2", () if yt is None else (yt.dtype,))
    _rows(ys, 1, NP, "rows_update ys", () if yt is None else (yt.dtype,))
    _rows(copy, M, NP, "rows_update copy", (od,))
    _rows(h, M, NP, "rows_update h", (od,))
    _index(xidx, M, "rows_update xidx")
    _index(yidx, M, "rows_update yidx")
    _index(ysi, M * top, "rows_update ysi")
    _index(pos, M, "rows_update pos")
    _weight(ysw, M * top, "rows_update ysw")
    for t, n in ((y_norm, "y_norm"), (y2_norm, "y2_norm"), (norm, "norm"), (norm_b, "norm_b")):
        _weight(t, NP, "rows_update " + n)
    if y_joined and (ys is None or y_norm is None):
        raise ValueError("rows_update: y_joined norms the sum with ys")
    if x_in is None and yt is None or (norm is None) != (h is None) or width > NP or NP % 4 or NP > WIDTH_MAX \
            or (norm_b is not None and norm is None) or (ys is not None and (ysi is None or ysw is None or top < 1)) \
            or (y2 is not None and (y is None or y_norm is None or y2_norm is None)):
        raise ValueError(f"rows_update: unsupported call (width {width} of {NP})")
    if freq is not None and (pos is None or freq.dtype != torch.float64 or freq.numel() < -(-width // 2)
                             or not freq.is_contiguous()):
        raise ValueError("rows_update: freq needs pos and fp64 entries for half the width")
    if x_in is not None and x_out is not None and x_in.stride(0) != x_out.stride(0):
        raise ValueError("rows_update: x_in and x_out must share a row stride")
    a = lib().RowsArgs()
    a.M, a.N, a.NP, a.mult, a.eps = M, width, NP, float(mult), float(eps)
    if x_in is not None:
        a.x_in, a.xidx, a.xrows, a.ldx = ptr(x_in), ptr(xidx), x_in.shape[0], x_in.stride(0)
    elif x_out is not None:
        a.ldx = x_out.stride(0)
    if y is not None:
        a.y, a.yidx, a.yrows, a.ldy = ptr(y), ptr(yidx), y.shape[0], y.stride(0)
    a.y_w, a.y_joined = ptr(y_norm), int(y_joined)
    if y2 is not None:
        a.y2, a.y2_w, a.ldy2 = ptr(y2), ptr(y2_norm), y2.stride(0)
    if ys is not None:
        a.ys, a.ysi, a.ysw, a.top, a.ldys, a.ysrows = ptr(ys), ptr(ysi), ptr(ysw), top, ys.stride(0), ys.shape[0]
    if x_add is not None:
        a.x_add, a.ldadd = ptr(x_add), x_add.stride(0)
    if freq is not None:
        a.pos, a.freq = ptr(pos), ptr(freq)
    a.x_out = ptr(x_out)
    if copy is not None:
        a.copy, a.ldcopy = ptr(copy), copy.stride(0)
    if h is not None:
        a.n_w, a.n_b, a.n_alpha, a.h, a.ldh = ptr(norm), ptr(norm_b), float(alpha), ptr(h), h.stride(0)
    if shift is not None:
        if norm is None or norm_b is not None or NP != shift.mu.numel() \
                or (x_in is not None and x_out is not None and x_in.data_ptr() == x_out.data_ptr()):
            raise ValueError("rows_update: a token shift needs a norm of the same rows, and x_out apart from x_in")
        shift.fill(a, M)
    y32 = yt is None and od == f32 or yt is not None and yt.dtype == f32
    check(lib().rows_update(a, int(y32), int(od == f32), stream_ptr()), "rows_update")


class TokenShift:
    """Mix of every normed row with that of the token before (``rows_update``).
    ``mu`` (NP,); ``state`` (slots, NP) fp32 keeps every sequence's last row;
    the rows' portions as ``start`` / ``last`` / ``slots`` / ``pos`` (``StepBatch``)."""

    __slots__ = ("mu", "state", "rows")

    def __init__(self, mu: torch.Tensor, state: torch.Tensor, start: torch.Tensor, last: torch.Tensor, slots: torch.Tensor,
                 pos: torch.Tensor):
        _weight(mu, 1, "token shift mu")
        if state.dtype != torch.float32 or state.dim() != 2 or state.shape[1] != mu.numel() or not state.is_contiguous():
            raise ValueError(f"token shift: state {tuple(state.shape)} {state.dtype} of rows of {mu.numel()}")
        self.mu, self.state, self.rows = mu, state, (start, last, slots, pos)

    def fill(self, a, M: int) -> None:
        for t in self.rows:
            _index(t, M, "token shift index")
        a.sh_mu, a.sh_state, a.sh_nslots = ptr(self.mu), ptr(self.state), self.state.shape[0]
        a.sh_start, a.sh_last, a.sh_slots, a.sh_pos = (ptr(t) for t in self.rows)
        # neighbouring rows of a group of threads (a workgroup's; a wave's where rows
        # are short): more of them form fewer rows twice, but the rows of a group are a
        # chain, so only what four workgroups a CU leave over.  4096 wide: 640 rows
        # 11 us (8 at a time 29), 2048 24 (37), 4096 38 (41), 8192 92 (one at a time 124).  Up to 2048 bf16 rows of 1024,
        # 2048 and 4096 columns have a kernel of their own (rows_shift_kernel), which does not ask.
        short = self.mu.numel() <= 1024
        a.sh_rows = min(4 if short else 8, -(-M // (4096 if short and M > 256 else 1024)))


def linear_f32(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor], out: torch.Tensor) -> torch.Tensor:
    """``x @ w.T + bias`` on the fp32 MFMA (K a multiple of 16)."""
    M, K = x.shape
    N = w.shape[0]
    f = (torch.float32,)
    _rows(x, M, K, "linear_f32 x", f)
    _rows(w, N, K, "linear_f32 w", f)
    _rows(out, M, N, "linear_f32 out", f)
    _weight(bias, N, "linear_f32 bias")
    check(lib().gemm_f32(ptr(x), x.stride(0), ptr(w), w.stride(0), ptr(out), out.stride(0), ptr(bias), M, N, K,
                         stream_ptr()), "gemm_f32")
    return out


class Linear:
    """A projection of the decoder layers: bf16 weights on the framework's MFMA
    GEMMs (with the decode copy in fragment order, ``gemm.shuffle_weight``), or
    fp32 weights on ``linear_f32``.  K (weight columns) is zero-padded to a
    multiple of 64 by the caller."""

    __slots__ = ("w", "bias", "ws", "act")

    def __init__(self, w: torch.Tensor, bias: Optional[torch.Tensor], dtype: torch.dtype, device,
                 act: int = G_.ACT_NONE, decode_copy: bool = True, consts: Optional[torch.Tensor] = None):
        """``act``: none, a gated activation of a packed weight (``gemm.pack_gate_up``),
        or xIELU, whose two constants are ``consts``."""
        if (consts is not None) != (act == G_.ACT_XIELU):
            raise ValueError("Linear: xIELU and its constants go together")
        if consts is not None:
            z = torch.zeros(w.shape[0]) if bias is None else bias
            bias = torch.cat([z.to(device=device, dtype=torch.float32), consts.to(device=device, dtype=torch.float32)])
        self.w = w.to(device=device, dtype=dtype).contiguous()
        self.bias = None if bias is None else bias.to(device=device, dtype=torch.float32).contiguous()
        self.act = act
        self.ws = G_.shuffle_weight(self.w) if dtype == torch.bfloat16 and decode_copy else None

    def __call__(self, x: torch.Tensor, out: torch.Tensor, gws: Optional[torch.Tensor] = None,
                 scratch: Optional[torch.Tensor] = None) -> torch.Tensor:
        """``scratch`` (fp32 gated projections): (M, weight rows) before the activation."""
        if self.w.dtype == torch.bfloat16:  # ``out`` may be fp32
            return G_.linear(x, self.w, self.bias, self.act, out=out, w_shuf=self.ws, ws=gws)
        if self.act == G_.ACT_NONE:
            return linear_f32(x, self.w, self.bias, out)
        if self.act == G_.ACT_XIELU:
            linear_f32(x, self.w, self.bias, out)
            M, N = x.shape[0], self.w.shape[0]
            check(lib().xielu_f32(ptr(out), out.stride(0), M, N, ptr(self.bias) + 4 * N, stream_ptr()), "xielu_f32")
            return out
        M, F = x.shape[0], self.w.shape[0] // 2
        gu = linear_f32(x, self.w, self.bias, scratch[:M])
        _rows(out, M, F, "gated linear out", (torch.float32,))
        check(lib().glu_f32(ptr(gu), gu.stride(0), ptr(out), out.stride(0), M, F, self.act, stream_ptr()), "glu_f32")
        return out


def token_gate(x: torch.Tensor, lin: Linear, table: torch.Tensor, off: int, ids: torch.Tensor, out: torch.Tensor,
               n: int, scratch: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``out[m, c] = gelu_tanh((x W^T)[m, c]) * table[ids[m], off + c]`` for c < n,
    0 in the padding columns; ``lin``: W (rows padded to a multiple of 64).
    ``scratch`` (fp32): (M, weight rows) for the projection."""
    M, K = x.shape
    dt, np_ = lin.w.dtype, lin.w.shape[0]
    _rows(x, M, K, "token_gate x", (dt,))
    _rows(table, 1, off + n, "token_gate table", (dt,))
    _rows(out, M, np_, "token_gate out", (dt,))
    _index(ids, M, "token_gate ids")
    if lin.w.shape[1] != K or lin.bias is not None or np_ % 64 or not 0 < n <= np_:
        raise ValueError(f"token_gate: x {tuple(x.shape)} vs w {tuple(lin.w.shape)}, {n} columns")
    if dt == torch.float32:
        z = linear_f32(x, lin.w, None, scratch[:M])
        check(lib().token_gate_f32(ptr(z), z.stride(0), ptr(table), table.stride(0), off, ptr(ids), table.shape[0],
                                   ptr(out), out.stride(0), M, n, np_, stream_ptr()), "token_gate_f32")
        return out
    if lin.ws is None or lin.ws.numel() != np_ * K * 2:
        raise ValueError("token_gate: the weight needs its fragment-order copy")
    check(lib().token_gate(ptr(x), x.stride(0), ptr(lin.w), lin.w.stride(0), ptr(lin.ws), K, ptr(table),
                           table.stride(0), off, ptr(ids), table.shape[0], ptr(out), out.stride(0), M, n, np_,
                           stream_ptr()), "token_gate")
    return out


def paged_args(qkv: torch.Tensor, kp: torch.Tensor, vp: torch.Tensor, table: torch.Tensor, slots: torch.Tensor,
               pos: torch.Tensor, out: torch.Tensor, M: int, H: int, scale: float, window: Optional[int], keep: int,
               gate: int = -1, gate_el: bool = False, kscale: Optional[torch.Tensor] = None,
               slopes: Optional[torch.Tensor] = None, sinks: Optional[torch.Tensor] = None, written: bool = False):
    """Validated arguments of the paged-attention launches.

    qkv rows ``[q H*DK | k G*DK | v G*DV | ...]``; ``kp`` (pages, G, 64, DK),
    ``vp`` (pages, G, 64, DV); ``table`` (slots, pages per sequence) int32;
    ``slots`` / ``pos`` per row; ``out`` rows ``[H*DV]``; ``gate``: first qkv
    column of the output gate, one per head or (``gate_el``) per head and value
    (-1: none); ``kscale`` (pages, 64): a factor of every key's scores;
    ``slopes`` (H,): slope * distance is taken off the scaled scores; ``sinks``
    (H,): scores that join the softmax without a value; ``written``: the rows'
    keys and values are in the cache already.  ``vp is
    kp``: the values are the keys, rows have no v columns, and the rows' keys
    are in the cache already (``mixer_ops.qk_norm``).  Every slot is the
    caller's: ``0 <= slots[m] < table.shape[0]``."""
    dt, shared = qkv.dtype, vp is kp
    if kp.dim() != 4 or vp.dim() != 4 or kp.shape[:3] != vp.shape[:3] or kp.shape[2] != PAGE:
        raise ValueError(f"paged attention: pages {tuple(kp.shape)} / {tuple(vp.shape)}")
    if kp.dtype != dt or vp.dtype != dt or out.dtype != dt or not (kp.is_contiguous() and vp.is_contiguous()):
        raise ValueError("paged attention: the cache and output share the projection's dtype, pages contiguous")
    P, G, _, DK = kp.shape
    DV = vp.shape[3]
    if DK not in HEAD_DIMS or DV not in HEAD_DIMS or H % G:
        raise ValueError(f"paged attention: {H} heads over {G}, sizes {DK} / {DV}")
    need = max((H + G) * DK + (0 if shared else G * DV), gate + H * (DV if gate_el else 1) if gate >= 0 else 0)
    _rows(qkv, M, need, "paged attention qkv", (torch.float32, torch.bfloat16))
    _rows(out, M, H * DV, "paged attention out", (dt,))
    _index(slots, M, "paged attention slots")
    _index(pos, M, "paged attention pos")
    if table.dtype != torch.int32 or table.dim() != 2 or not table.is_contiguous():
        raise ValueError("paged attention: block table must be contiguous int32 (slots, pages)")
    if not scale > 0:
        raise ValueError("paged attention: the score scale must be positive")
    if kscale is not None and (kscale.dtype != torch.float32 or tuple(kscale.shape) != (P, PAGE)
                               or not kscale.is_contiguous()):
        raise ValueError("paged attention: kscale must be contiguous fp32 (pages, 64)")
    _weight(slopes, H, "paged attention slopes")
    _weight(sinks, H, "paged attention sinks")
    keep = min(int(keep), 1 << 30)
    a = lib().PagedAttnArgs(ptr(qkv), qkv.stride(0), ptr(kp), ptr(vp), ptr(table), table.shape[1], P, ptr(slots),
                            ptr(pos), ptr(out), out.stride(0), M, H, G, DK, DV, gate,
                            NO_WINDOW if window is None else int(window), keep, float(scale))
    a.kscale, a.slopes, a.gate_el, a.shared, a.written = ptr(kscale), ptr(slopes), int(gate_el), int(shared), int(shared or written)
    a.sinks = ptr(sinks)
    return a


def paged_write(args, f32: bool) -> None:
    """Store the k / v columns of every row in its sequence's pages."""
    check(lib().paged_write(args, int(f32), stream_ptr()), "paged_write")


def _tiles(tiles: torch.Tensor, what: str) -> None:
    if tiles.dtype != torch.int32 or tiles.dim() != 2 or tiles.shape[1] != 4 or not tiles.is_contiguous():
        raise ValueError(f"{what}: tiles must be contiguous int32 (n, 4)")


def paged_prefill(args, tiles: torch.Tensor) -> None:
    """Attention of chunks of tokens already written to the cache.  ``tiles``
    (n, 4) int32: {first row, tokens, slot, first packed row} (``chunk_tiles``)."""
    _tiles(tiles, "paged_prefill")
    n = tiles.shape[0]
    for i in range(0, n, 65535):
        part = tiles[i:i + 65535]
        check(lib().paged_prefill(args, ptr(part), part.shape[0], stream_ptr()), "paged_prefill")


def chunk_tiles(row0: int, tokens: int, slot: int, group: int, rows: int = TILE_ROWS) -> list:
    """Prefill workgroups of one chunk: ``tokens * group`` packed rows (group =
    query heads per KV head) in groups of ``rows``, the last (longest) ones first."""
    return [(row0, tokens, slot, r) for r in range(0, tokens * group, rows)][::-1]


def paged_splits(n_seq: int, H: int, G: int, keys: int, window: Optional[int], keep: int) -> int:
    """Workgroups per (sequence, KV head) of a decode launch: enough for two per
    CU, with at least eight 32-key units each."""
    if window is not None:
        keys = min(keys, window + keep + 2 * PAGE)
    units = -(-max(keys, 1) // 32)
    wgs = n_seq * G * -(-(H // G) // 32)
    return max(1, min(-(-512 // wgs), units // 8, 64))


def _decode_parts(rows: torch.Tensor, n: int, splits: int, ws: Optional[torch.Tensor], what: str) -> None:
    _index(rows, n, f"{what} rows")
    if splits > 1 and (ws is None or ws.dtype != torch.float32 or not ws.is_contiguous()):
        raise ValueError(f"{what}: splits > 1 needs an fp32 workspace")


def paged_mixed(args, tiles: torch.Tensor, rows: torch.Tensor, n: int, splits: int, ws: Optional[torch.Tensor]) -> None:
    """``paged_prefill`` of ``tiles`` and ``paged_decode`` of ``n`` sequences in one launch; every row's k / v is in the
    cache already."""
    _tiles(tiles, "paged_mixed")
    _decode_parts(rows, n, splits, ws, "paged_mixed")
    check(lib().paged_mixed(args, ptr(tiles), tiles.shape[0], ptr(rows), n, splits, ptr(ws), 0 if ws is None else ws.numel(),
                            stream_ptr()), "paged_mixed")


def paged_decode(args, rows: torch.Tensor, n: int, splits: int, ws: Optional[torch.Tensor]) -> None:
    """One token of each of ``n`` sequences (``rows``: their batch rows); also
    stores the tokens' k / v.  ``ws``: fp32, n * H * splits * (DV + 2) for splits > 1."""
    _decode_parts(rows, n, splits, ws, "paged_decode")
    check(lib().paged_decode(args, ptr(rows), n, splits, ptr(ws), 0 if ws is None else ws.numel(), stream_ptr()),
          "paged_decode")


def paged_attn_f32(args) -> None:
    """fp32 attention of every row (cache already written)."""
    check(lib().paged_attn_f32(args, stream_ptr()), "paged_attn_f32")


def poly_norm(z: torch.Tensor, w: torch.Tensor, M: int, n: int, eps: float) -> None:
    """``z <- a N(z) + b N(z^2) + c N(z^3) + e`` in place over the first n columns,
    ``w`` = (a, b, c, e), ``N(y) = y / sqrt(mean(y^2) + eps)``."""
    f32 = z.dtype == torch.float32
    _rows(z, M, -(-n // 8) * 8, "poly_norm z", (torch.float32, torch.bfloat16))
    _weight(w, 4, "poly_norm weight")
    a = lib().PolyNormArgs()
    a.z, a.w, a.ld, a.M, a.n, a.eps = ptr(z), ptr(w), z.stride(0), M, n, eps
    check(lib().poly_norm(a, int(f32), stream_ptr()), "poly_norm")


# ---------------------------------------------------------------------- attention over a latent cache
LATENT_DIMS, LATENT_ROT = (128, 256, 512), (64, 128)  # latent columns and key-part columns the kernels are built for
LATENT_ROWS = (32, 64)                                # packed (token, head) rows of one workgroup
LATENT_KEYS = (64, 128)                               # head sizes of keys and values for scores over keys


def pad_to(n: int, sizes, what: str) -> int:
    for p in sizes:
        if n <= p:
            return p
    raise ValueError(f"{what} {n} exceeds {sizes[-1]}")


class Rope:
    """Rotation of pairs: radians per position of every pair, and the factor of
    cos and sin."""

    def __init__(self, freqs, mag: float, device):
        import math
        self.freq = torch.tensor(freqs, dtype=torch.float64, device=device) / (2.0 * math.pi)
        self.pairs, self.mag = len(freqs), float(mag)

    def table(self):
        return lib().RopeTable(ptr(self.freq), self.pairs, self.mag)


QK_PAIRS = 128  # pairs of a head that ``qk_heads`` turns at most


def qk_heads(rows: torch.Tensor, kp: torch.Tensor, vp: torch.Tensor, rope: Rope, table: torch.Tensor, slots: torch.Tensor,
             pos: torch.Tensor, M: int, H: int, dim: int, eps: float) -> None:
    """Rows ``[q H*DK | k G*DK | v G*DV | ...]``: every head of q and k rotated
    (value i of a head with value i + pairs) and divided by its root mean square
    over ``dim`` values; q in place, k and v into the pages ``kp`` / ``vp``."""
    if kp.dim() != 4 or vp.dim() != 4 or kp.shape[:3] != vp.shape[:3] or kp.shape[2] != PAGE or kp.dtype != rows.dtype \
            or vp.dtype != rows.dtype or not (kp.is_contiguous() and vp.is_contiguous()):
        raise ValueError(f"qk_heads: pages {tuple(kp.shape)} / {tuple(vp.shape)} of {kp.dtype} / {vp.dtype}")
    P, G, _, DK = kp.shape
    DV = vp.shape[3]
    _rows(rows, M, (H + G) * DK + G * DV, "qk_heads rows", (torch.float32, torch.bfloat16))
    _index(slots, M, "qk_heads slots")
    _index(pos, M, "qk_heads pos")
    if table.dtype != torch.int32 or table.dim() != 2 or not table.is_contiguous() or not 0 < dim <= DK \
            or 2 * rope.pairs > dim or rope.pairs > QK_PAIRS:
        raise ValueError(f"qk_heads: {rope.pairs} pairs in heads of {dim}, or a bad block table")
    a = lib().QkHeadsArgs()
    a.qkv, a.kp, a.vp, a.table, a.slots, a.pos = (ptr(t) for t in (rows, kp, vp, table, slots, pos))
    a.rope, a.ldq, a.ldt, a.npages, a.M = rope.table(), rows.stride(0), table.shape[1], P, M
    a.H, a.G, a.DK, a.DV, a.dim, a.eps = H, G, DK, DV, dim, eps
    check(lib().qk_heads(a, int(rows.dtype == torch.float32), stream_ptr()), "qk_heads")


def rope_rows(x: torch.Tensor, M: int, H: int, hs: int, col: int, RP: int, pos: torch.Tensor, rope: Rope) -> None:
    """Rotate columns ``h * hs + col ..`` of every row and head in place."""
    _rows(x, M, (H - 1) * hs + col + RP, "rope rows", (torch.float32, torch.bfloat16))
    _index(pos, M, "rope pos")
    es = x.element_size()
    if col * es % 16 or 2 * rope.pairs > RP or hs < RP:
        raise ValueError(f"rope_rows: {rope.pairs} pairs in {RP} columns at {col}")
    check(lib().rope_rows(ptr(x) + col * es, x.stride(0), hs, M, H, RP, ptr(pos), rope.table(),
                          int(x.dtype == torch.float32), stream_ptr()), "rope_rows")


def _latent_pool(kp: torch.Tensor, dtype) -> None:
    if kp.dim() != 3 or kp.shape[1] != PAGE or kp.dtype != dtype or not kp.is_contiguous():
        raise ValueError(f"latent cache: contiguous (pages, {PAGE}, columns) of {dtype} expected, got {tuple(kp.shape)}")


def latent_prep(rows: torch.Tensor, kp: torch.Tensor, qw: torch.Tensor, cw: torch.Tensor, rope: Rope, table: torch.Tensor,
                slots: torch.Tensor, pos: torch.Tensor, M: int, QN: int, CN: int, CP: int, eps: float) -> None:
    """Rows ``[query latent | latent CP | key part]`` in place: RMS norms of the
    latents (true widths QN, CN; weights ``qw``, ``cw`` padded with zeros),
    rotation of the key part; latent and key part into the cache ``kp``."""
    _latent_pool(kp, rows.dtype)
    QP, RP = qw.numel(), kp.shape[2] - CP
    _rows(rows, M, QP + kp.shape[2], "latent rows", (rows.dtype,))
    _weight(qw, QP, "latent query norm")
    _weight(cw, CP, "latent norm")
    _index(slots, M, "latent slots")
    _index(pos, M, "latent pos")
    if table.dtype != torch.int32 or table.dim() != 2 or not table.is_contiguous() or RP < 2 * rope.pairs:
        raise ValueError("latent_prep: bad block table or key part")
    a = lib().LatentPrepArgs()
    a.rows, a.kp, a.qw, a.cw, a.table, a.slots, a.pos = (ptr(t) for t in (rows, kp, qw, cw, table, slots, pos))
    a.rope, a.ld, a.ldt, a.npages, a.M = rope.table(), rows.stride(0), table.shape[1], kp.shape[0], M
    a.QN, a.QP, a.CN, a.CP, a.RP, a.eps = QN, QP, CN, CP, RP, eps
    check(lib().latent_prep(a, int(rows.dtype == torch.float32), stream_ptr()), "latent_prep")


def latent_args(qlat: torch.Tensor, q: torch.Tensor, rot_col: int, hs: int, kp: torch.Tensor, table: torch.Tensor,
                slots: torch.Tensor, pos: torch.Tensor, out: torch.Tensor, M: int, H: int, CP: int, scale: float,
                gate: Optional[torch.Tensor] = None):
    """Validated arguments of the latent-attention launches: ``qlat`` rows
    [H][CP], the rotated query parts at columns ``h * hs + rot_col`` of ``q``,
    ``out`` rows [H][CP], ``gate`` rows of one logit per head."""
    dt = qlat.dtype
    _latent_pool(kp, dt)
    RP = kp.shape[2] - CP
    if CP not in LATENT_DIMS or RP not in LATENT_ROT:
        raise ValueError(f"latent attention: {CP} + {RP} columns")
    _rows(qlat, M, H * CP, "latent qlat", (torch.float32, torch.bfloat16))
    _rows(q, M, (H - 1) * hs + rot_col + RP, "latent q", (dt,))
    _rows(out, M, H * CP, "latent out", (dt,))
    if gate is not None:
        _rows(gate, M, H, "latent gate", (dt,))
    _index(slots, M, "latent slots")
    _index(pos, M, "latent pos")
    if table.dtype != torch.int32 or table.dim() != 2 or not table.is_contiguous() or not scale > 0:
        raise ValueError("latent attention: bad block table or score scale")
    a = lib().LatentAttnArgs()
    a.qlat, a.qrot, a.kp, a.table = ptr(qlat), ptr(q) + rot_col * q.element_size(), ptr(kp), ptr(table)
    a.slots, a.pos, a.out, a.gate = ptr(slots), ptr(pos), ptr(out), ptr(gate)
    a.ldql, a.ldqr, a.hs, a.ldo, a.ldg = qlat.stride(0), q.stride(0), hs, out.stride(0), gate.stride(0) if gate is not None else 0
    a.ldt, a.npages, a.M, a.H, a.CP, a.RP, a.scale = table.shape[1], kp.shape[0], M, H, CP, RP, scale
    return a


def latent_splits(n_seq: int, tiles: int, keys: int) -> int:
    """Workgroups per tile of a decoded token (``tiles`` a token): one per CU, two pages each."""
    pages = -(-max(keys, 1) // PAGE)
    return max(1, min(-(-256 // (n_seq * tiles)), pages // 2, 64))


def latent_ws(n_seq: int, H: int, splits: int, CP: int) -> int:
    """fp32 partials of ``n_seq`` decoded tokens."""
    return n_seq * H * splits * (CP + 4) if splits > 1 else 0


def latent_attn(args, tiles: torch.Tensor, rows: int, splits: int = 1, per_token: int = 1,
                ws: Optional[torch.Tensor] = None) -> None:
    """``tiles`` (n, 4) int32: {first row, tokens, slot, first packed row of ``rows``}
    (``chunk_tiles``).  ``splits`` > 1: single tokens, ``per_token`` tiles each;
    ``ws``: fp32, ``latent_ws``."""
    _tiles(tiles, "latent_attn")
    if splits > 1 and (ws is None or ws.dtype != torch.float32 or not ws.is_contiguous()):
        raise ValueError("latent_attn: splits > 1 needs an fp32 workspace")
    check(lib().latent_attn(args, ptr(tiles), tiles.shape[0], rows, splits, per_token, ptr(ws), 0 if ws is None else ws.numel(),
                            stream_ptr()), "latent_attn")


def _tiles(t: torch.Tensor, what: str) -> None:
    if t.dtype != torch.int32 or t.dim() != 2 or t.shape[1] != 4 or not t.is_contiguous():
        raise ValueError(f"{what}: tiles must be contiguous int32 (n, 4)")


def latent_gather(kp: torch.Tensor, table: torch.Tensor, ent: torch.Tensor, out: torch.Tensor) -> None:
    """Cache pages to rows: ``ent`` (n, 4) int32 {first row of the page's 64, slot,
    block, 0}; ``out`` (rows, CP + RP)."""
    _latent_pool(kp, torch.bfloat16)
    _tiles(ent, "latent_gather")
    if out.dtype != kp.dtype or out.dim() != 2 or out.shape[1] != kp.shape[2] or not out.is_contiguous() \
            or table.dtype != torch.int32 or table.dim() != 2 or not table.is_contiguous():
        raise ValueError(f"latent_gather: rows {tuple(out.shape)} {out.dtype} of pages {tuple(kp.shape)}")
    check(lib().latent_gather(ptr(kp), kp.shape[2], ptr(table), table.shape[1], kp.shape[0], ptr(ent), ent.shape[0], ptr(out),
                              out.shape[0], stream_ptr()), "latent_gather")


def latent_prefill(q: torch.Tensor, kv: torch.Tensor, krot: torch.Tensor, pos: torch.Tensor, out: torch.Tensor, M: int, H: int,
                   DP: int, VP: int, scale: float, tiles: torch.Tensor, gate: Optional[torch.Tensor] = None) -> None:
    """Causal attention over gathered keys: ``q`` rows [H][DP + RP], ``kv`` key rows
    [H][DP | VP], ``krot`` key rows [RP], ``out`` rows [H][VP]; ``tiles`` (n, 4)
    int32 {first row, tokens, first key row, first token of 128}."""
    keys, RP = krot.shape
    dt = torch.bfloat16
    if DP not in LATENT_KEYS or VP not in LATENT_KEYS or RP not in LATENT_ROT or not scale > 0:
        raise ValueError(f"latent_prefill: {DP} + {RP} key and {VP} value columns")
    _rows(q, M, H * (DP + RP), "latent q", (dt,))
    _rows(kv, keys, H * (DP + VP), "latent keys", (dt,))
    _rows(krot, keys, RP, "latent key part", (dt,))
    _rows(out, M, H * VP, "latent out", (dt,))
    if gate is not None:
        _rows(gate, M, H, "latent gate", (dt,))
    _index(pos, M, "latent pos")
    _tiles(tiles, "latent_prefill")
    a = lib().LatentKeysArgs()
    a.q, a.kv, a.krot, a.pos, a.out, a.gate = ptr(q), ptr(kv), ptr(krot), ptr(pos), ptr(out), ptr(gate)
    a.ldq, a.ldkv, a.ldr, a.ldo, a.ldg = (t.stride(0) if t is not None else 0 for t in (q, kv, krot, out, gate))
    a.M, a.H, a.DP, a.RP, a.VP, a.keys, a.scale = M, H, DP, RP, VP, keys, scale
    check(lib().latent_prefill(a, ptr(tiles), tiles.shape[0], stream_ptr()), "latent_prefill")


def latent_attn_f32(args) -> None:
    """fp32 attention of every row (cache already written)."""
    check(lib().latent_attn_f32(args, stream_ptr()), "latent_attn_f32")
