"""Colocated pipeline: every stage on one GPU (the 1-GPU measurement point).

Stage forwards are chained on one stream over preallocated buffers.  A step on
the images in ``ColocatedPipeline.x`` can be captured into one HIP graph (``capture``);
a step on images that the first stage reads where they lie is launched, captured
or not.  The multi-rank schedules (GPipe
stream, CLI request stream, decode ring) live in ``runtime/scheduler.py``.
"""
from __future__ import annotations

from typing import List, Optional, Sequence

import torch

from ..utils import trace
from .graph import GraphedStep
from .stages import StageCompute, StageOutput


class ColocatedPipeline:
    def __init__(self, stages: Sequence[StageCompute], batch: int):
        self.stages = list(stages)
        self.batch = batch
        dev = self.stages[0].device
        shp, dt = self.stages[0].in_spec(batch)
        self.x = torch.zeros(shp, dtype=dt, device=dev)
        self.bufs: List[torch.Tensor] = []
        for s in self.stages:
            oshp, odt = s.out_spec(batch)
            self.bufs.append(torch.empty(oshp, dtype=odt, device=dev))
        self._in = (self.x.get_device(), dt, self.x.shape)
        self._writes = [(b.data_ptr(), b.nbytes) for b in (self.x, *self.bufs)]
        self._graph: Optional[GraphedStep] = None

    def _step(self, x: Optional[torch.Tensor] = None):
        h = self.x
        for i, (s, b) in enumerate(zip(self.stages, self.bufs)):
            h = s.forward(x, b, keep=self.x) if i == 0 and x is not None else s.forward(h, b)
        return h

    def capture(self) -> None:
        self._graph = GraphedStep(self._step, self.stages[0].device)

    def _reads(self, x: torch.Tensor) -> bool:
        """Can the first stage read ``x`` where it lies?  Its launch then leaves the
        copy in ``self.x`` that a later call without an input runs on.  Not what shares
        memory with a buffer the pass writes, nor a tensor whose values are not the
        bytes at its address (negated views, zeros without memory)."""
        return (type(x) is torch.Tensor and x.is_cuda and getattr(self.stages[0], "keeps_input", False)
                and x.get_device() == self._in[0] == torch.cuda.current_device() and x.dtype == self._in[1]
                and x.shape == self._in[2] and x.is_contiguous() and not x.requires_grad
                and not x.is_neg() and not x._is_zerotensor() and self._apart(x.data_ptr()))

    def _apart(self, at: int) -> bool:
        """Does an input at this address share no byte with a buffer the pass writes?"""
        n = self._writes[0][1]
        for start, size in self._writes:
            if -n < at - start < size:
                return False
        return True

    def __call__(self, x: Optional[torch.Tensor] = None) -> StageOutput:
        # an input read in place: no copy kernel in front (301 of 2718 us at 65536 images),
        # and the few launches of a pass go out before the device has run the first
        direct = x is not None and self._reads(x)
        if x is not None and not direct:
            self.x.copy_(x, non_blocking=True)
        few = getattr(self.stages[0], "pass_few", None) if direct and len(self.stages) == 2 and not trace.enabled() else None
        if few is not None:
            out = few(self.stages[1], x, self.bufs[0], self.bufs[1], self.x)
            if out is not None:
                return out
        with trace.span("pipeline_step", "compute", device=self.x.device, batch=self.batch):
            if direct:
                return self._step(x)
            if self._graph is not None:
                return self._graph()
            return self._step()
