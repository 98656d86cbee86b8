"""The head_dim 128 backward kernel (bwd_wide_kernel in csrc/attn_mfma.hip)
where its work split can go wrong: columns of 1, 63, 64, 65 and 129 entries
(steps of 64), blocks that end inside a 32-key group, two waves a group at
every block size, grouped heads, cut and whole columns, both partial types.
Yardstick: float64 autograd of the oracle with the routing held fixed, bar
twice the oracle's own error in the input type (tolerance.py)."""

import pytest
import torch

from conftest import make_qkv, oracle_cfg
from moba.config import MoBAConfig
from moba.kernels.attention import moba_attention
from moba.kernels.moba_bwd import bwd_kernel, compute_delta
from moba.kernels.moba_fwd import attend_partials, combine_partials
from moba.kernels.routing import ENV_SEGMENT, build_csc_fused, csc_to_mask
from oracle import naive as O
from tolerance import assert_within_tolerance, max_abs_error

pytestmark = pytest.mark.gpu

# (S or packed lengths, query heads, kv heads, block, top_k)
CASES = [([63, 64, 65, 1, 129, 300], 1, 1, 32, 3), ([63, 64, 65, 1, 129, 300], 1, 1, 64, 2),
         ([63, 64, 65, 1, 129, 300], 1, 1, 128, 2), (513, 8, 2, 32, 5), (1000, 4, 1, 64, 4),
         (777, 4, 4, 128, 3),
         # more than 256 columns: one program past every segment list
         (2200, 2, 2, 32, 3)]


def _inputs(case, dtype, device):
    s, hq, hk, bs, k = case
    lens = s if isinstance(s, list) else None
    b, t = (1, sum(lens)) if lens else (2, s)
    q, do = make_qkv((b, t, hq, 128), dtype, seed=bs, n=2)
    kk, v = make_qkv((b, t, hk, 128), dtype, seed=bs + 1, n=2)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32) if lens else None
    kw = {"cu_seqlens": cu.to(device), "max_seqlen": max(lens)} if lens else {}
    return MoBAConfig(block_size=bs, top_k=k, dtype=dtype), q, kk, v, do, cu, kw


@pytest.mark.parametrize("entries", ["0", "96"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES)
def test_gradients_match_oracle(device, monkeypatch, case, dtype, entries):
    monkeypatch.setenv(ENV_SEGMENT, entries)
    cfg, q, k, v, do, cu, kw = _inputs(case, dtype, device)
    qd, kd, vd = (t.to(device).requires_grad_(True) for t in (q, k, v))
    moba_attention(qd, kd, vd, cfg, **kw).backward(do.to(device))
    sel = csc_to_mask(build_csc_fused(qd.detach(), kd.detach(), cfg, **kw), q.shape[1]).cpu()

    def grads(to):
        leaves = [t.detach().to(to, copy=True).requires_grad_(True) for t in (q, k, v)]
        O.moba_attention(*leaves, oracle_cfg(cfg), selected=sel, query_chunk=256,
                         cu_seqlens=cu).backward(do.to(to))
        return [t.grad for t in leaves]

    for name, got, low, want in zip(("dq", "dk", "dv"), (qd.grad, kd.grad, vd.grad),
                                    grads(dtype), grads(torch.float64)):
        assert_within_tolerance(got, want, max_abs_error(low, want), name)


@pytest.mark.parametrize("case", CASES[2:5])
def test_float32_partials_round_to_the_16_bit_ones(device, case):
    """One program for both partial types: dK / dV are the same bits, and the
    float32 dQ partials round to the 16-bit ones."""
    cfg, q, k, v, do, _, kw = _inputs(case, torch.bfloat16, device)
    q, k, v, do = (t.to(device) for t in (q, k, v, do))
    index = build_csc_fused(q, k, cfg, **kw)
    out, lse = combine_partials(*attend_partials(q, k, v, cfg, index), q.dtype, return_lse=True)
    ld = compute_delta(out, do, lse)

    def backward(dtype):
        dk, dv = torch.empty_like(k), torch.empty_like(v)
        dq = torch.zeros((q.shape[0], q.shape[2], q.shape[1], index.max_slots, 128),
                         device=device, dtype=dtype)
        bwd_kernel(do, q, k, v, ld, cfg, index, dk, dv, dq)
        return dq, dk, dv

    wide, narrow = backward(torch.float32), backward(torch.bfloat16)
    assert torch.equal(wide[0].bfloat16(), narrow[0])
    assert torch.equal(wide[1], narrow[1]) and torch.equal(wide[2], narrow[2])
