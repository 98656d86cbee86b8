"""A whole forward or backward in one library call (`moba_forward_step`,
`moba_backward_step`): the stages of `pooling`, `gating`, `routing`, `moba_fwd`
and `moba_bwd` in order, without their per-stage allocations and calls."""

import ctypes
from dataclasses import dataclass

import torch

from moba import _lib
from moba.config import MoBAConfig
from moba.kernels.routing import MAX_SEGMENTS, segment_entries

_POINTERS = _lib.Step.q.offset  # the device addresses end the struct


@dataclass(frozen=True)
class SavedStep:
    """What a forward keeps for its backward: the call's shape and one buffer
    holding the CSC index, the (m, l) pairs and lse."""

    shape: _lib.Step  # without addresses: the backward fills in its own
    saved: torch.Tensor
    cu_seqlens: torch.Tensor | None


def forward(q, k, v, cfg: MoBAConfig, causal: bool, cu_seqlens, max_seqlen, keep: bool):
    """out [B, S, H_q, D], and with `keep` a `SavedStep` (else None). q, k, v
    validated and contiguous, routing by the exact gate, partials in q's
    dtype."""
    dev = _lib.require_gpu(q, k, v, cu_seqlens)
    q, k, v = (_lib.aligned_contiguous(t) for t in (q, k, v))
    b, s, h_q, d = q.shape
    packed = cu_seqlens is not None
    rows, rps = (cu_seqlens.numel() - 1, max_seqlen) if packed else (b, s)
    slots = cfg.slots()
    dtype = _lib.DTYPE_CODE[q.dtype]
    step = _lib.Step(rows, s, rps, h_q, k.shape[2], d, cfg.block_size, slots,
                     cfg.past_blocks_selected(cfg.num_blocks(rps)), bool(cfg.always_select_current),
                     bool(causal), dtype, dtype, keep, packed,
                     max(0, segment_entries(rows * h_q * rps * slots)), MAX_SEGMENTS)
    _lib.run_step("moba_step_layout", step)
    out = torch.empty_like(q)
    saved = torch.empty(step.saved_bytes, device=dev, dtype=torch.uint8)
    temp = torch.empty(step.forward_temp, device=dev, dtype=torch.uint8)
    step.q, step.k, step.v = q.data_ptr(), k.data_ptr(), v.data_ptr()
    step.cu_seqlens = cu_seqlens.data_ptr() if packed else None
    step.out, step.saved, step.temp = out.data_ptr(), saved.data_ptr(), temp.data_ptr()
    _lib.run_step("moba_forward_step", step, _lib.stream_handle(dev))
    if not keep:
        return out, None
    ctypes.memset(ctypes.byref(step, _POINTERS), 0, ctypes.sizeof(step) - _POINTERS)
    return out, SavedStep(step, saved, cu_seqlens)


def backward(dout, q, k, v, out, kept: SavedStep, dkv_dtype=None):
    """(dq, dk, dv) of a `forward` with `keep`; dk / dv in `dkv_dtype`
    (None: q's dtype, or torch.float32 for sums the caller adds to others)."""
    dev = _lib.require_gpu(dout, q, k, v, out)
    q, k, v = (_lib.aligned_contiguous(t) for t in (q, k, v))
    dout, out = _lib.aligned_contiguous(dout.to(q.dtype)), _lib.aligned_contiguous(out)
    step = _lib.Step.from_buffer_copy(kept.shape)
    dq = torch.empty_like(q)
    dk, dv = torch.empty_like(k, dtype=dkv_dtype), torch.empty_like(v, dtype=dkv_dtype)
    temp = torch.empty(step.backward_temp, device=dev, dtype=torch.uint8)
    step.dkv_dtype = _lib.DTYPE_CODE[dk.dtype]
    step.q, step.k, step.v = q.data_ptr(), k.data_ptr(), v.data_ptr()
    step.cu_seqlens = None if kept.cu_seqlens is None else kept.cu_seqlens.data_ptr()
    step.out, step.saved, step.temp = out.data_ptr(), kept.saved.data_ptr(), temp.data_ptr()
    step.dout, step.dq, step.dk, step.dv = (dout.data_ptr(), dq.data_ptr(), dk.data_ptr(),
                                            dv.data_ptr())
    _lib.run_step("moba_backward_step", step, _lib.stream_handle(dev))
    return dq, dk, dv
