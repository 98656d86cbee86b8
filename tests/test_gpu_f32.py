"""The float32 matrix kernels (csrc/attn_f32.hip) at every head_dim and block
size they take: ragged lengths, grouped query heads, packed sequences shorter
than a block, columns cut into segments and whole, against float64 autograd
of the oracle with the routing held fixed. Bar: the float32 path's 1e-5
(tolerance.py), scaled where gradients exceed 1 as the other tests scale it.
"""

import pytest
import torch

from conftest import make_qkv, oracle_cfg
from moba import _lib
from moba.config import MoBAConfig
from moba.kernels.attention import moba_attention
from moba.kernels.moba_bwd import bwd_kernel, compute_delta
from moba.kernels.moba_fwd import attend_partials, combine_partials, empty_partials
from moba.kernels.routing import build_csc_fused, csc_to_mask, index_stride
from oracle import naive as O
from tolerance import FP32_MAX_ABS

pytestmark = pytest.mark.gpu

# (S or packed lengths, query heads, kv heads, head_dim, block, top_k)
CASES = [(513, 4, 2, 64, 32, 5), (1000, 4, 4, 64, 64, 4), (777, 8, 2, 64, 128, 3),
         (300, 4, 1, 128, 32, 6), (449, 4, 2, 128, 64, 2), (900, 2, 2, 128, 128, 8),
         ([200, 1, 33, 391], 4, 2, 64, 32, 3), ([64, 500, 129], 4, 4, 128, 128, 2),
         # more than 256 columns: one program past every segment list
         (2200, 2, 2, 64, 32, 3)]


def _inputs(case, device):
    s, hq, hk, d, bs, k = case
    lens = s if isinstance(s, list) else None
    t = sum(lens) if lens else s
    b = 1 if lens else 2
    q, do = make_qkv((b, t, hq, d), torch.float32, seed=d + bs, n=2)
    kk, v = make_qkv((b, t, hk, d), torch.float32, seed=d + bs + 1, n=2)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32) if lens else None
    kw = {"cu_seqlens": cu.to(device), "max_seqlen": max(lens)} if lens else {}
    return MoBAConfig(block_size=bs, top_k=k, dtype=torch.float32), q, kk, v, do, cu, kw


@pytest.mark.parametrize("entries", ["0", "48", None])
@pytest.mark.parametrize("case", CASES)
def test_f32_forward_and_backward_match_oracle(device, monkeypatch, case, entries):
    if entries is not None:
        monkeypatch.setenv("MOBA_SEGMENT_ENTRIES", entries)
    cfg, q, k, v, do, cu, kw = _inputs(case, device)
    qd, kd, vd = (t.to(device).requires_grad_(True) for t in (q, k, v))
    out = moba_attention(qd, kd, vd, cfg, **kw)
    out.backward(do.to(device))
    sel = csc_to_mask(build_csc_fused(qd.detach(), kd.detach(), cfg, **kw), q.shape[1]).cpu()
    qr, kr, vr = (t.double().requires_grad_(True) for t in (q, k, v))
    ref = O.moba_attention(qr, kr, vr, oracle_cfg(cfg), selected=sel, query_chunk=256, cu_seqlens=cu)
    ref.backward(do.double())
    for name, got, want in (("out", out, ref), ("dq", qd.grad, qr.grad), ("dk", kd.grad, kr.grad),
                            ("dv", vd.grad, vr.grad)):
        err = (got.detach().cpu().double() - want.detach()).abs().max().item()
        assert err <= FP32_MAX_ABS * max(1.0, want.detach().abs().max().item()), (name, err)


@pytest.mark.parametrize("case", [CASES[2], CASES[4]])
def test_f32_kernels_agree_with_the_fma_kernels(device, monkeypatch, case):
    """Inputs off a 16-byte boundary run the FMA kernels: the same slots are
    written, with every m, l and partial row, and every gradient, within 1e-5
    of the matrix kernels' (scaled where values exceed 1)."""
    monkeypatch.setenv("MOBA_SEGMENT_ENTRIES", "0")
    cfg, q, k, v, do, _, _ = _inputs(case, device)
    q, k, v, do = (t.to(device) for t in (q, k, v, do))
    index = build_csc_fused(q, k, cfg)

    def shifted(t):  # the same values 4 bytes off
        buf = torch.empty(t.numel() + 1, device=t.device, dtype=t.dtype)
        buf[1:] = t.reshape(-1)
        return buf[1:].view(t.shape)

    def attend(q_):  # as attend_partials, which would realign q
        part = empty_partials(q.shape, index.max_slots, q.device, q.dtype)
        _lib.call("moba_attend", *(_lib.ptr(t) for t in (
            q_, k, v, index.col_nnz, index.col_offsets, index.row_indices, index.head_indices,
            index.slot_of_pair, index.order, part[0], part[2])), None, 2, q.shape[1], q.shape[1],
            q.shape[2], k.shape[2], q.shape[3], index.num_blocks, cfg.block_size, index.max_slots,
            index.row_indices.shape[-1], index_stride(index), None, None, None, 0, 1, 2, 2,
            _lib.stream_handle(q.device))
        return part

    def close(a, b):
        return (a - b).abs().max().item() <= FP32_MAX_ABS * max(1.0, b.abs().max().item())

    fast, slow = attend(q), attend(shifted(q))
    wrote = fast[0] > -float("inf")
    assert bool(wrote.any()) and bool((~wrote).any())
    assert torch.equal(wrote, slow[0] > -float("inf"))
    assert bool(torch.isneginf(fast[0][~wrote]).all()) and bool(torch.isneginf(slow[0][~wrote]).all())
    for a, b in zip(fast, slow):
        assert close(a[wrote], b[wrote])
    assert not torch.equal(fast[2][wrote], slow[2][wrote]), "one kernel ran both times"
    out, lse = combine_partials(*fast, q.dtype, return_lse=True)
    ld = compute_delta(out, do, lse)

    def backward(q_):
        dk, dv = torch.empty_like(k), torch.empty_like(v)
        dq = torch.zeros((*q.shape[:1], q.shape[2], q.shape[1], index.max_slots, q.shape[3]),
                         device=device)
        bwd_kernel(do, q_, k, v, ld, cfg, index, dk, dv, dq)
        return dq[wrote], dk, dv

    for a, b in zip(backward(q), backward(shifted(q))):
        assert close(a, b)


def test_f32_backward_with_float32_sized_scratch_runs_whole_columns(device, monkeypatch):
    """A caller whose segment scratch holds float32 sums only (scratch_cap 2 *
    (seg_cap - nb)) gets whole columns: dK / dV those of an uncut index."""
    cfg, q, k, v, do, _, _ = _inputs(CASES[1], device)
    q, k, v, do = (t.to(device) for t in (q, k, v, do))
    monkeypatch.setenv("MOBA_SEGMENT_ENTRIES", "48")
    index = build_csc_fused(q, k, cfg)
    assert int(index.seg_counts[..., 1].sum()) > 0, "no column was cut"
    out, lse = combine_partials(*attend_partials(q, k, v, cfg, index), q.dtype, return_lse=True)
    ld = compute_delta(out, do, lse)
    cap = 2 * (index.seg_cap - index.num_blocks)
    res = {}
    for name, times in (("float32", 1), ("float64", 2)):
        scratch = torch.full((2 * k.shape[2] * cap * times * 2 * cfg.block_size * q.shape[3] + 64,),
                             7.0, device=device)
        dk, dv = torch.empty_like(k), torch.empty_like(v)
        dq = torch.zeros((2, q.shape[2], q.shape[1], index.max_slots, q.shape[3]), device=device)
        _lib.call("moba_bwd", *(_lib.ptr(t) for t in (
            q, k, v, do, ld, index.col_nnz, index.col_offsets, index.row_indices,
            index.head_indices, index.slot_of_pair, index.order, dk, dv, dq)), None, 2, q.shape[1],
            q.shape[1], q.shape[2], k.shape[2], q.shape[3], index.num_blocks, cfg.block_size,
            index.max_slots, index.row_indices.shape[-1], index_stride(index),
            _lib.ptr(index.segments), _lib.ptr(index.seg_split), _lib.ptr(index.seg_counts),
            index.seg_cap, _lib.ptr(scratch), cap * times, 1, 2, 2, 2, _lib.stream_handle(q.device))
        assert bool((scratch[-64:] == 7.0).all()), "wrote past the scratch"
        if times == 1:
            assert bool((scratch == 7.0).all()), "whole columns need no scratch"
        res[name] = (dq, dk, dv)
    assert torch.equal(res["float32"][0], res["float64"][0])
    for a, b in zip(res["float32"][1:], res["float64"][1:]):
        assert (a - b).abs().max().item() <= 2.0 ** -22 * b.abs().max().item()  # float64 sums, rounded once
