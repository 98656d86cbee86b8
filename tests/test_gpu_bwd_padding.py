"""The backward kernels pad a column's last step with dead entries: whatever
statistics the call's first row has (the one a dead entry's reads fall on),
they add nothing to dK / dV of other rows. The first row's lse is its own
single score, its delta that of whatever output it has: NaN where it selects
nothing, or where its query holds NaN. Yardstick: dense float64 attention over
the selected keys.
"""

import pytest
import torch

from conftest import make_qkv
from moba.config import MoBAConfig
from moba.kernels.attention import moba_attention
from moba.kernels.routing import build_csc_fused, csc_to_mask
from tolerance import FP32_MAX_ABS, assert_within_tolerance, max_abs_error

pytestmark = pytest.mark.gpu

SHAPES = [(d, bs) for d in (64, 128) for bs in (32, 64, 128)]


def _dense_grads(q, k, v, do, sel, bs, dtype):
    """(dq, dk, dv) of dense attention in `dtype`; a query that sees no key
    has output 0 and no gradient."""
    q, k, v = (t.detach().cpu().to(dtype).requires_grad_(True) for t in (q, k, v))
    s, group = q.shape[1], q.shape[2] // k.shape[2]
    seen = sel.repeat_interleave(bs, -1)[..., :s] & torch.ones(s, s, dtype=torch.bool).tril()
    kk, vv = (t.repeat_interleave(group, 2).transpose(1, 2).contiguous() for t in (k, v))
    score = torch.matmul(q.transpose(1, 2), kk.transpose(2, 3).contiguous()) * q.shape[3] ** -0.5
    some = seen.any(-1, keepdim=True)
    p = torch.softmax(torch.where(some, score.masked_fill(~seen, -float("inf")), 0.0), -1) * some
    torch.matmul(p, vv).transpose(1, 2).backward(do.cpu().to(dtype))
    return q.grad, k.grad, v.grad


def _inputs(d, bs, dtype, device):
    """Two rows of grouped heads, a length that ends inside a block."""
    q, do = make_qkv((2, 7 * bs - 5, 4, d), dtype, seed=d + bs, n=2)
    k, v = make_qkv((2, 7 * bs - 5, 2, d), dtype, seed=d + bs + 1, n=2)
    return [t.to(device) for t in (q, k, v, do)]


def _ours(q, k, v, do, cfg):
    """Gradients and the selection, on the CPU."""
    index = build_csc_fused(q, k, cfg)
    assert bool((index.col_nnz % 32 != 0).any()), "no step is padded"
    sel = csc_to_mask(index, q.shape[1]).cpu()
    q, k, v = (t.clone().requires_grad_(True) for t in (q, k, v))
    # nan_to_num: queries with no selection produce NaN by design
    torch.nan_to_num(moba_attention(q, k, v, cfg)).backward(do)
    return [t.grad.cpu() for t in (q, k, v)], sel


def _check(got, q, k, v, do, sel, bs, dtype, keep=None):
    """Float32: the float32 path's bar; 16-bit types: twice the error of the
    dense attention in that type. `keep`: masks of what to compare."""
    want = _dense_grads(q, k, v, do, sel, bs, torch.float64)
    low = None if dtype == torch.float32 else _dense_grads(q, k, v, do, sel, bs, dtype)
    for i, name in enumerate(("dq", "dk", "dv")):
        m = keep[i] if keep else torch.ones(got[i].shape[:3], dtype=torch.bool)
        assert bool(torch.isfinite(got[i][m]).all()), name
        if low is not None:
            assert_within_tolerance(got[i][m], want[i][m], max_abs_error(low[i][m], want[i][m]), name)
            continue
        bar = FP32_MAX_ABS * max(1.0, want[i][m].abs().max().item())
        assert max_abs_error(got[i][m], want[i][m]) <= bar, name


DTYPES = [torch.float32, torch.float16, torch.bfloat16]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("d,bs", SHAPES)
def test_first_rows_without_selection(device, d, bs, dtype):
    """Without the own block the first block's queries select nothing, so the
    first row's output and delta are NaN."""
    cfg = MoBAConfig(block_size=bs, top_k=2, dtype=dtype, always_select_current=False)
    q, k, v, do = _inputs(d, bs, dtype, device)
    got, sel = _ours(q, k, v, do, cfg)
    assert not bool(sel[:, :, 0].any())
    _check(got, q, k, v, do, sel, bs, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("d,bs", SHAPES)
def test_nan_in_the_first_row_stays_there(device, d, bs, dtype):
    """NaN in the first query of batch row 0, head 0: its own block's keys of
    its kv head may have NaN gradients, nothing else."""
    cfg = MoBAConfig(block_size=bs, top_k=3, dtype=dtype)
    q, k, v, do = _inputs(d, bs, dtype, device)
    q[0, 0, 0] = float("nan")
    got, sel = _ours(q, k, v, do, cfg)
    q[0, 0, 0] = 0.0
    keep = [torch.ones(t.shape[:3], dtype=torch.bool) for t in got]
    keep[0][0, 0, 0] = False
    keep[1][0, :bs, 0] = keep[2][0, :bs, 0] = False
    _check(got, q, k, v, do, sel, bs, dtype, keep)


@pytest.mark.parametrize("dtype,score", [(torch.float32, -200.0), (torch.float16, -20.0),
                                         (torch.bfloat16, -100.0)])
@pytest.mark.parametrize("d,bs", SHAPES)
def test_low_score_of_the_first_row(device, d, bs, dtype, score):
    """The first row's lse, its one score, so low that exp2(0 - lse) overflows
    the type the weights are held in."""
    cfg = MoBAConfig(block_size=bs, top_k=3, dtype=dtype)
    q, k, v, do = _inputs(d, bs, dtype, device)
    key = k[0, 0, 0].float()
    q[0, 0, 0] = (key * (score * d ** 0.5 / key.square().sum())).to(dtype)
    got, sel = _ours(q, k, v, do, cfg)
    _check(got, q, k, v, do, sel, bs, dtype)
