"""CIFAR-10 ConvNet on the fused gfx950 kernels.

Two precisions, packed once at load (reference ``node.py:305-306`` only moves
fp32 modules to the device):

* ``fp32`` (the reference's precision, default): ``csrc/kernels/cifar_x3.hip``.
  Every fp32 operand is split into bf16 hi + lo and each product is three bf16
  MFMAs (hi*hi + hi*lo + lo*hi) accumulated in fp32; from three images a workgroup on conv2 is
  Winograd's F(2 x 2, 3 x 3) on two fp16 terms (``cifar_wino.hip``).  Stage boundary tensor
  ``(B,4096)`` fp32 exactly as the reference ships it (``node.py:45-48``).
  fc1 at large batch is ``cifar_fc1_x3``: the fp32 boundary rows come to LDS as they
  are and are split in registers on their way to the MFMAs (no split copy), K in ranges over
  the workgroups where its 256-row tiles would not fill the chip; a typed output, a strided one
  of fewer rows, or rows off 16 bytes are ONE bf16 GEMM over K' = 3*4096 on ``[A_hi | A_hi | A_lo]``
  x ``[W_hi | W_lo | W_hi]``.
  Optional boundary encoding ``boundary="split"`` (fp32 only, both ends of
  the hop must be these kernels): the same 16 KiB/img, each row as 32-k blocks
  of 32 bf16 hi then 32 bf16 lo — the very hi/lo operands the x3 MFMAs consume
  (hi + lo = the fp32 value to ~2^-17) — written by the stage-0 epilogue and
  read as they lie in fc1: 0.624 -> 0.549 ms at B=65536 with bit-identical
  outputs, but the split stores cost the stage-0 epilogue as much, so the 2-stage
  step is unchanged (2.41 vs 2.43 ms) and the pipelines keep plain fp32 (also the wire format a reference peer expects).
  ``decode_boundary`` / ``encode_boundary`` convert.
* ``bf16``: ``csrc/kernels/cifar_fused.hip`` (v4 persistent kernel), bf16
  boundary, an explicitly reduced-precision mode.

Weight layouts:

* conv1 ``(32,3,3,3)`` -> ``[32][48]`` with ``k = ky*16 + kx*4 + c`` (kx<3, c<3 real);
* conv2 ``(64,32,3,3)`` -> ``[64][288]`` with ``k = (ky*3+kx)*32 + c`` (HWC activation image);
* fc1 ``[512][4096]`` (K-contiguous for the GEMM), fc2 ``(10,512)`` -> ``[16][512]``
  zero-padded to one MFMA N-tile.  Biases are fp32.
The flatten order is the reference's NCHW ``c*64 + h*8 + w`` (``cifar_model_parts.py:41``).
"""
from __future__ import annotations

import functools
import math
from dataclasses import dataclass
from typing import Dict, Optional, Tuple

import torch

from ._lib import check, lib, ptr, stream_ptr
from .gemm import ACT_RELU, linear

PRECISIONS = ("fp32", "bf16")


def split_bf16(w: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """fp32 -> (hi, lo) bf16 with hi + lo == w to ~2^-17 relative."""
    w = w.float()
    hi = w.to(torch.bfloat16)
    lo = (w - hi.float()).to(torch.bfloat16)
    return hi, lo


def _conv1_k48(sd) -> torch.Tensor:
    w = torch.zeros(32, 3, 4, 4)  # (oc, ky, kx, c) zero-padded kx=3, c=3
    w[:, :, :3, :3] = sd["conv1.weight"].float().permute(0, 2, 3, 1)
    return w.reshape(32, 48)


def _conv2_k288(sd) -> torch.Tensor:
    return sd["conv2.weight"].float().permute(0, 2, 3, 1).reshape(64, 288)  # (oc, ky, kx, c)


def _conv2_winograd(sd) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
    """U = G g G^T of every conv2 filter, times a power of two per output channel that brings its largest
    number into [2^9, 2^10), as two fp16 terms [4 i + j][oc][c]; the inverse scales; the largest number of a filter (oc, c)."""
    G = torch.tensor([[1, 0, 0], [.5, .5, .5], [.5, -.5, .5], [0, 0, 1]], dtype=torch.float64)
    u = G @ sd["conv2.weight"].detach().cpu().double() @ G.t()  # (oc, c, i, j)
    u_top = torch.nan_to_num(u.abs(), nan=0.0, posinf=0.0).amax((2, 3))
    top = u_top.amax(1)
    k = torch.where(top > 0, 10 - torch.frexp(top).exponent, 0).clamp(-110, 110)
    u = (u * 2.0 ** k.double()[:, None, None, None]).permute(2, 3, 0, 1).reshape(16, 64, 32)
    hi = u.half()
    return hi, (u - hi.double()).half(), (2.0 ** -k.double()).float(), u_top


def _winograd_range(sd, u_top: torch.Tensor) -> Optional[torch.Tensor]:
    """(l1, b, most): conv1 of an image of magnitudes up to m stays within l1 m + b; up to ``most`` that is at most
    ``WINO_RANGE`` times what conv1's biases bring to every conv2 channel: their mean by the magnitudes of its
    weights, each up to 4 times the median bias (one large bias lifts the scale of all channels, and may never pass
    the ReLU).  None where one scale an image or an output channel would cost precision: ``most`` is
    below ``WINO_IMAGES``; or a filter's numbers in U (``u_top``: the largest, (oc, c)), which keep 2^-34 of the
    channel's largest, lie below 2^-16 of it, so that they keep fewer bits than a pair of bf16.
    What is not finite does not count: its channel is lost whatever the scale."""
    w1, b1, w2 = (torch.nan_to_num(sd[k].detach().cpu().double().abs(), nan=0.0, posinf=0.0)
                  for k in ("conv1.weight", "conv1.bias", "conv2.weight"))
    by = w2.sum((2, 3))
    by = by[by.sum(1) > 0]
    typical = b1.clamp(max=4 * b1.median())
    floor = (by @ typical / by.sum(1)).min() if len(by) else b1.median()
    l1, b = w1.sum((1, 2, 3)).max() * (1 + 2.0 ** -12), b1.max()
    most = (WINO_RANGE * floor - b) / l1 if l1 > 0 else torch.tensor(math.inf, dtype=torch.float64)
    if not most >= WINO_IMAGES or bool(((u_top > 0) & (u_top < u_top.amax(1, keepdim=True) * 2.0 ** -16)).any()):
        return None
    return torch.stack([l1, b, most]).float()


def _fc2_pad(sd) -> torch.Tensor:
    w = torch.zeros(16, 512)
    w[:10] = sd["fc2.weight"].float()
    return w


@dataclass
class CifarStage0Weights:
    precision: str
    b1: torch.Tensor
    b2: torch.Tensor
    w1: torch.Tensor = None    # bf16: [32][48]
    w2: torch.Tensor = None    # bf16: [64][288]
    w1h: torch.Tensor = None   # fp32 path: split conv weights
    w1l: torch.Tensor = None
    w2h: torch.Tensor = None
    w2l: torch.Tensor = None
    u2h: torch.Tensor = None   # fp32 path, Winograd's conv2: [16][64][32] fp16, two terms
    u2l: torch.Tensor = None
    sc: torch.Tensor = None    # its scales: _winograd_range, 64 inverse scales of u2


@dataclass
class CifarHeadWeights:
    precision: str
    w_fc1: torch.Tensor = None   # bf16: [512][4096]; fp32: [512][3*4096] = [hi | lo | hi] (typed, strided outputs)
    w_fc1h: torch.Tensor = None  # fp32 path: W hi / lo [512][4096] each (cifar_fc1_x3)
    w_fc1l: torch.Tensor = None
    b_fc1: torch.Tensor = None
    w_fc2: torch.Tensor = None   # bf16: [16][512]
    w_fc2h: torch.Tensor = None  # fp32 path: split fc2
    w_fc2l: torch.Tensor = None
    b_fc2: torch.Tensor = None


def _check_precision(p: str) -> str:
    if p not in PRECISIONS:
        raise ValueError(f"CIFAR precision must be one of {PRECISIONS}, got {p!r}")
    return p


def pack_stage0(sd: Dict[str, torch.Tensor], device, precision: str = "fp32") -> CifarStage0Weights:
    _check_precision(precision)
    b1 = sd["conv1.bias"].float().to(device).contiguous()
    b2 = sd["conv2.bias"].float().to(device).contiguous()
    w1, w2 = _conv1_k48(sd), _conv2_k288(sd)
    if precision == "bf16":
        return CifarStage0Weights("bf16", b1, b2,
                                  w1=w1.to(device=device, dtype=torch.bfloat16).contiguous(),
                                  w2=w2.to(device=device, dtype=torch.bfloat16).contiguous())
    (w1h, w1l), (w2h, w2l) = split_bf16(w1), split_bf16(w2)
    dv = lambda t: t.to(device).contiguous()  # noqa: E731
    w = CifarStage0Weights("fp32", b1, b2, w1h=dv(w1h), w1l=dv(w1l), w2h=dv(w2h), w2l=dv(w2l))
    u2h, u2l, inv, u_top = _conv2_winograd(sd)
    if (rng := _winograd_range(sd, u_top)) is not None:
        w.u2h, w.u2l, w.sc = dv(u2h), dv(u2l), dv(torch.cat([rng, inv]))
    return w


def pack_head(sd: Dict[str, torch.Tensor], device, fc1: bool = True, fc2: bool = True,
              precision: str = "fp32") -> CifarHeadWeights:
    _check_precision(precision)
    w = CifarHeadWeights(precision)
    if fc1:
        f = sd["fc1.weight"].float()
        if precision == "bf16":
            w.w_fc1 = f.to(device=device, dtype=torch.bfloat16).contiguous()
        else:
            hi, lo = split_bf16(f)
            w.w_fc1 = torch.cat([hi, lo, hi], dim=1).to(device).contiguous()
            w.w_fc1h, w.w_fc1l = hi.to(device).contiguous(), lo.to(device).contiguous()
        w.b_fc1 = sd["fc1.bias"].float().to(device).contiguous()
    if fc2:
        f2 = _fc2_pad(sd)
        if precision == "bf16":
            w.w_fc2 = f2.to(device=device, dtype=torch.bfloat16).contiguous()
        else:
            hi, lo = split_bf16(f2)
            w.w_fc2h, w.w_fc2l = hi.to(device).contiguous(), lo.to(device).contiguous()
        w.b_fc2 = sd["fc2.bias"].float().to(device).contiguous()
    return w


def act_dtype(precision: str) -> torch.dtype:
    """dtype of the stage-boundary activations (flattened conv map, fc1 hidden)."""
    return torch.float32 if _check_precision(precision) == "fp32" else torch.bfloat16


STAGE0_GRID = 0  # persistent stage-0 workgroups; 0 = one per CU (256)
# conv2 by Winograd (cifar_wino.hip) beyond this many images a workgroup (us, direct : this: 256 images 12.9 :
# 13.6, 512 19.2 : 18.1, 600 23.9 : 22.2, 1000 32.5 : 28.3, 8192 228 : 192, 65536 1796 : 1475).  Up to two images a
# workgroup the results are those of the bands of few images, bit by bit; beyond, of another rounding: the rows of a batch
# and of its parts of up to 512 images (256 CUs) differ by 3.5e-6 (2-norm; the distances to 64 bits are 3.0e-6 and 4.8e-6).
WINO_ROUNDS = 2
WINO_RANGE = 65536  # its fp16 terms hold a range of this much beside conv1's biases; wider images go the direct way there
WINO_IMAGES = 256  # magnitudes that have to be in range, raw pixels among them, for weights to take it
# strided fp32 rows below this batch are written by the GEMM over [hi | hi | lo] rows; from it
# on the fused fc1, without a split of K, is the faster one (us, GEMM : fused: 8192 rows 197 :
# 237, 9216 251 : 230, 16384 324 : 235).  Outputs of another type or layout are the GEMM's.
FC1_X3_MIN_ROWS = 8704
# fp32 head up to this batch: fc1 in slices of K and a finish of one workgroup a row
# (pipeline pass, us, with and without: 1 row 27.7 / 44.3, 64 29.7 / 57.4, 256 50.6 /
# 84.9, 512 79.1 / 88.3, 768 104.4 / 96.2: each 32 rows are a round of every workgroup)
FC1_FEW_ROWS = 512


def set_stage0_grid(grid: int = 0) -> None:
    """Persistent stage-0 grid size (0 = one workgroup per CU).  With fewer
    workgroups than CUs the spare CUs stay free for concurrent kernels (an RCCL
    hop kernel cannot start a workgroup on a CU the stage-0 kernel holds)."""
    global STAGE0_GRID
    STAGE0_GRID = int(grid)


def _check_act(t: torch.Tensor, shape, dtype, what: str) -> None:
    if t.dtype != dtype or tuple(t.shape[1:]) != tuple(shape) or not t.is_contiguous():
        raise ValueError(f"{what}: expected contiguous {dtype} (B,{','.join(map(str, shape))}), "
                         f"got {t.dtype} {tuple(t.shape)}")


BOUNDARIES = ("fp32", "split")


def _split_boundary(boundary: str, precision: str) -> int:
    if boundary not in BOUNDARIES:
        raise ValueError(f"boundary must be one of {BOUNDARIES}, got {boundary!r}")
    if boundary == "split" and precision != "fp32":
        raise ValueError("the split boundary encoding exists for the fp32 precision only")
    return int(boundary == "split")


def encode_boundary(h: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """fp32 (B,K) -> the blocked hi/lo boundary encoding (same shape and dtype)."""
    out = torch.empty_like(h) if out is None else out
    check(lib().cifar_split_blocked(ptr(h), ptr(out), h.shape[0], h.shape[1], 0, stream_ptr()), "encode_boundary")
    return out


def decode_boundary(h: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Blocked hi/lo boundary encoding -> fp32 values (hi + lo)."""
    out = torch.empty_like(h) if out is None else out
    check(lib().cifar_split_blocked(ptr(h), ptr(out), h.shape[0], h.shape[1], 1, stream_ptr()), "decode_boundary")
    return out


def stage0_forward(x: torch.Tensor, w: CifarStage0Weights, out: Optional[torch.Tensor] = None,
                   grid: int = 0, boundary: str = "fp32", keep: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Units 0-1: x (B,3,32,32) fp32 contiguous -> (B,4096) fp32 (or bf16 in bf16 mode;
    ``boundary="split"``: the blocked hi/lo encoding in the fp32 tensor).  ``keep``
    (fp32 precision; apart from x): receives a copy of x in the same launch."""
    split = _split_boundary(boundary, w.precision)
    grid = grid or STAGE0_GRID
    _check_act(x, (3, 32, 32), torch.float32, "stage0 input")
    B = x.shape[0]
    dt = act_dtype(w.precision)
    if out is None:
        out = torch.empty((B, 4096), dtype=dt, device=x.device)
    if tuple(out.shape) != (B, 4096) or out.dtype != dt or not out.is_contiguous():
        raise ValueError("stage0: bad output buffer")
    if keep is not None:
        if w.precision != "fp32":
            raise ValueError("stage0: keep exists for the fp32 precision only")
        _check_act(keep, (3, 32, 32), torch.float32, "stage0 keep")
        if keep.shape[0] != B or abs(ptr(keep) - ptr(x)) < x.nbytes:
            raise ValueError("stage0: keep must be as large as x and apart from it")
    if w.precision == "fp32":
        if not stage0_direct(B, w, grid):
            check(lib().cifar_stage0_wino(ptr(x), ptr(out), ptr(w.w1h), ptr(w.w1l), ptr(w.b1), ptr(w.w2h), ptr(w.w2l),
                                          ptr(w.u2h), ptr(w.u2l), ptr(w.b2), ptr(w.sc), B, grid, stream_ptr(), split,
                                          ptr(keep)), "cifar_stage0_wino")
        else:
            check(lib().cifar_stage0_x3(ptr(x), ptr(out), ptr(w.w1h), ptr(w.w1l), ptr(w.b1), ptr(w.w2h), ptr(w.w2l),
                                        ptr(w.b2), B, grid, stream_ptr(), split, ptr(keep)), "cifar_stage0_x3")
    else:
        check(lib().cifar_stage0_v4(ptr(x), ptr(out), ptr(w.w1), ptr(w.b1), ptr(w.w2), ptr(w.b2), B, grid,
                                    stream_ptr()), "cifar_stage0_v4")
    return out


def stage0_direct(B: int, w: CifarStage0Weights, grid: int = 0) -> bool:
    """fp32: conv2 as it is, not by Winograd."""
    return B <= WINO_ROUNDS * (grid or STAGE0_GRID or 256) or w.u2h is None


def plain(t: torch.Tensor, shape: tuple) -> bool:
    return t.shape == shape and t.dtype == torch.float32 and t.is_contiguous()


def pass_few(x: torch.Tensor, w0: CifarStage0Weights, h: torch.Tensor, keep: torch.Tensor, wh: CifarHeadWeights,
             scratch: torch.Tensor, hid: torch.Tensor, probs: torch.Tensor, pred: torch.Tensor, boundary: str) -> None:
    """``stage0_forward`` (``keep``) and ``head_forward`` of up to ``FC1_FEW_ROWS`` images, fp32, into plain buffers that are
    as large as those take, by one native call."""
    args = [0 if t is None else t.data_ptr() for t in (x, h, w0.w1h, w0.w1l, w0.b1, w0.w2h, w0.w2l, w0.b2, keep, wh.w_fc1h,
                                                       wh.w_fc1l, wh.b_fc1, scratch, hid, wh.w_fc2h, wh.w_fc2l, wh.b_fc2,
                                                       probs, pred)]
    check(lib().cifar_pass_few(args, x.shape[0], STAGE0_GRID, int(boundary == "split"), stream_ptr()), "cifar_pass_few")


def _head_few(h: torch.Tensor, w: CifarHeadWeights, hid: Optional[torch.Tensor], probs: Optional[torch.Tensor],
              pred: Optional[torch.Tensor], scratch: Optional[torch.Tensor], split: int) -> None:
    B = h.shape[0]
    part = _fc1_scratch(scratch, B, h.device)  # 8 x B x 512 floats of the 12288 bf16 a row
    check(lib().cifar_head_few(ptr(h), split, ptr(w.w_fc1h), ptr(w.w_fc1l), ptr(w.b_fc1), ptr(part), ptr(hid),
                               ptr(w.w_fc2h), ptr(w.w_fc2l), ptr(w.b_fc2), ptr(probs), ptr(pred), B, stream_ptr()),
          "cifar_head_few")


def _fc1_scratch(scratch: Optional[torch.Tensor], B: int, device) -> torch.Tensor:
    """``scratch`` where its first ``B`` rows are 24 KB each, one behind the other."""
    if scratch is not None and scratch.dtype != torch.bfloat16:
        raise TypeError(f"fc1 scratch: bf16 rows expected, got {scratch.dtype}")
    if (scratch is None or scratch.shape[0] < B or tuple(scratch.shape[1:]) != (3 * 4096,)
            or not scratch[:B].is_contiguous()):
        scratch = torch.empty((B, 3 * 4096), dtype=torch.bfloat16, device=device)
    return scratch


@functools.lru_cache(maxsize=256)
def _fc1_splits(B: int) -> int:
    """Ranges of K of the fused fc1, so that its tiles fill one round of 256 CUs: a k-step
    takes 1.75 us, a workgroup 5 around its steps, the sum of the parts a launch and their way
    out and in at 4 TB/s.  us, GEMM over [hi | hi | lo] rows : this (whole): 520 rows 46.8 : 38.2
    (226), 2000 57.4 : 52.7 (228), 4000 92.6 : 66.2 (230), 8192 195 : 97.5 (231), 12288 291 : 149
    (232), 16384 328 : 176 (252)."""
    tiles, best, splits = -(-B // 256) * 2, math.inf, 1
    for s in range(1, 13):  # 12: the parts of a row in the 24 KB of its scratch
        if s > 1 and tiles * s > 256:
            break
        us = -(-tiles * s // 256) * (5 + 1.75 * -(-128 // s)) + (4 + s * B * 4096 / 4e6 if s > 1 else 0)
        if us < best:
            best, splits = us, s
    return splits


def fc1_scratch_rows(B: int) -> int:
    """Rows of 24 KB that ``fc1_forward`` of a batch into a plain output takes as ``scratch`` (0:
    none); into another one it takes ``B``, and brings its own where it is given fewer."""
    if B <= FC1_FEW_ROWS:
        return B
    s = _fc1_splits(B)
    return -(-B * s // 12) if s > 1 else 0


def _plain(hid: Optional[torch.Tensor], B: int) -> bool:
    return hid is None or (tuple(hid.shape) == (B, 512) and hid.dtype == torch.float32 and hid.is_contiguous())


def _fp32_rows(out: torch.Tensor, B: int) -> bool:
    """Can the fused fc1 write these rows, at a distance of their own?"""
    return (tuple(out.shape) == (B, 512) and out.dtype == torch.float32 and out.stride(1) == 1
            and out.stride(0) >= 512 and out.stride(0) % 4 == 0)


def _dma_rows(h: torch.Tensor, w: CifarHeadWeights) -> bool:
    """The fused fc1 fetches rows and weights by 16-byte LDS-DMA; split3 and the GEMM take any ``h``."""
    return (ptr(h) | ptr(w.w_fc1h) | ptr(w.w_fc1l)) % 16 == 0


def _few_rows(h: torch.Tensor, w: CifarHeadWeights, hid: Optional[torch.Tensor]) -> bool:
    """One row a workgroup of the finish; a strided or typed ``hid`` is the GEMM's."""
    B = h.shape[0]
    return w.precision == "fp32" and 0 < B <= FC1_FEW_ROWS and _plain(hid, B)


def fc1_forward(h: torch.Tensor, w: CifarHeadWeights, out: Optional[torch.Tensor] = None,
                scratch: Optional[torch.Tensor] = None, boundary: str = "fp32") -> torch.Tensor:
    """Unit 2: (B,4096) -> relu(fc1) (B,512) on the MFMA GEMM (fp32: split operand,
    ``scratch`` = (>= fc1_scratch_rows(B), 12288) bf16 for parts, or (>= B, 12288) for [hi | hi | lo]
    rows; ``boundary``: the encoding of ``h``)."""
    split = _split_boundary(boundary, w.precision)
    dt = act_dtype(w.precision)
    _check_act(h, (4096,), dt, "fc1 input")
    B = h.shape[0]
    if w.precision == "bf16":
        return linear(h, w.w_fc1, w.b_fc1, act=ACT_RELU, out=out)
    if _few_rows(h, w, out):
        out = torch.empty((B, 512), dtype=torch.float32, device=h.device) if out is None else out
        _head_few(h, w, out, None, None, scratch, split)
        return out
    plain = _plain(out, B)
    if ((plain and B > FC1_FEW_ROWS) or (B >= FC1_X3_MIN_ROWS and _fp32_rows(out, B))) and _dma_rows(h, w):
        if out is None:
            out = torch.empty((B, 512), dtype=torch.float32, device=h.device)
        s = _fc1_splits(B) if plain else 1
        part = _fc1_scratch(scratch, -(-B * s // 12), h.device) if s > 1 else None
        check(lib().cifar_fc1_x3(ptr(h), 4096, ptr(w.w_fc1h), ptr(w.w_fc1l), 4096, ptr(w.b_fc1), ptr(out),
                                 512 if plain else out.stride(0), B, 512, 4096, stream_ptr(), split, s, ptr(part)),
              "cifar_fc1_x3")
        return out
    a3 = _fc1_scratch(scratch, B, h.device)[:B]
    check(lib().cifar_split3(ptr(h), 4096, ptr(a3), 3 * 4096, B, 4096, stream_ptr(), split), "cifar_split3")
    if out is None:
        out = torch.empty((B, 512), dtype=torch.float32, device=h.device)
    return linear(a3, w.w_fc1, w.b_fc1, act=ACT_RELU, out=out)


def head_tail(hid: torch.Tensor, w: CifarHeadWeights, probs: Optional[torch.Tensor] = None,
              pred: Optional[torch.Tensor] = None) -> Tuple[torch.Tensor, torch.Tensor]:
    """Unit 3: (B,512) -> fc2 + softmax (B,10) fp32 + per-row argmax (B,) int32."""
    _check_act(hid, (512,), act_dtype(w.precision), "head_tail input")
    B = hid.shape[0]
    probs = probs if probs is not None else torch.empty((B, 10), dtype=torch.float32, device=hid.device)
    pred = pred if pred is not None else torch.empty((B,), dtype=torch.int32, device=hid.device)
    if w.precision == "fp32":
        check(lib().cifar_head_tail_x3(ptr(hid), ptr(w.w_fc2h), ptr(w.w_fc2l), ptr(w.b_fc2), ptr(probs), ptr(pred),
                                       B, stream_ptr()), "cifar_head_tail_x3")
    else:
        check(lib().cifar_head_tail(ptr(hid), ptr(w.w_fc2), ptr(w.b_fc2), ptr(probs), ptr(pred), B, stream_ptr()),
              "cifar_head_tail")
    return probs, pred


def head_forward(h: torch.Tensor, w: CifarHeadWeights, hid: Optional[torch.Tensor] = None,
                 probs: Optional[torch.Tensor] = None, pred: Optional[torch.Tensor] = None,
                 boundary: str = "fp32", scratch: Optional[torch.Tensor] = None) -> Tuple[torch.Tensor, torch.Tensor]:
    """Units 2-3: h (B,4096) -> (probs (B,10) fp32, pred (B,) int32); ``hid`` (if given) holds
    relu(fc1) afterwards, ``scratch`` as in ``fc1_forward``."""
    if _few_rows(h, w, hid):
        split = _split_boundary(boundary, w.precision)
        _check_act(h, (4096,), torch.float32, "fc1 input")
        probs = probs if probs is not None else torch.empty((h.shape[0], 10), dtype=torch.float32, device=h.device)
        pred = pred if pred is not None else torch.empty((h.shape[0],), dtype=torch.int32, device=h.device)
        _head_few(h, w, hid, probs, pred, scratch, split)
        return probs, pred
    hid = fc1_forward(h, w, out=hid, scratch=scratch, boundary=boundary)
    return head_tail(hid, w, probs, pred)
