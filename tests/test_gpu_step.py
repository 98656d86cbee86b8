"""The whole-step entry points (csrc/step.cpp) against the stages called one by
one: with the same index, output and gradients are the same bits.
"""

import pytest
import torch

from conftest import make_qkv
from moba import _lib
from moba.config import MoBAConfig
from moba.kernels.attention import moba_attention
from moba.kernels.moba_fwd import moba_forward
from moba.kernels.routing import build_csc_fused

pytestmark = pytest.mark.gpu

# (S or packed lengths, batch, query heads, kv heads, head_dim, block, top_k, dtype)
CASES = [(515, 2, 4, 2, 64, 64, 4, torch.bfloat16), (1, 1, 2, 2, 64, 32, 8, torch.float16),
         ([130, 1, 700], 1, 8, 2, 128, 64, 3, torch.bfloat16), (400, 1, 4, 1, 64, 32, 1, torch.float32),
         ([64, 900], 1, 4, 4, 64, 128, 6, torch.float32), (300, 1, 2, 1, 256, 32, 3, torch.bfloat16)]


@pytest.mark.parametrize("entries", ["0", "64", None])
@pytest.mark.parametrize("case", CASES)
def test_step_equals_stages(device, monkeypatch, case, entries):
    """No segment list, cut columns, the default; a backward run twice."""
    if entries is not None:
        monkeypatch.setenv("MOBA_SEGMENT_ENTRIES", entries)
    s, b, hq, hk, d, bs, k, dtype = case
    lens = s if isinstance(s, list) else None
    t = sum(lens) if lens else s
    cfg = MoBAConfig(block_size=bs, top_k=k, dtype=dtype)
    q, do = make_qkv((b, t, hq, d), dtype, seed=1, device=device, n=2)
    kk, v = make_qkv((b, t, hk, d), dtype, seed=2, device=device, n=2)
    kw = {}
    if lens:
        kw = {"cu_seqlens": torch.tensor([0] + lens).cumsum(0).to(torch.int32).to(device),
              "max_seqlen": max(lens)}
    index = build_csc_fused(q, kk, cfg, **kw)
    results = []
    for given in (index, None):
        x = [z.clone().requires_grad_(True) for z in (q, kk, v)]
        out = moba_attention(*x, cfg, index=given, **({} if given is not None else kw))
        grads = torch.autograd.grad(out, x, do, retain_graph=True)
        again = torch.autograd.grad(out, x, do)
        assert all(torch.equal(a, c) for a, c in zip(grads, again))
        results.append((out.detach(), *grads))
    assert all(torch.equal(a, c) for a, c in zip(*results))
    assert torch.equal(moba_forward(q, kk, v, cfg, **kw), results[0][0])
    assert torch.equal(moba_forward(q, kk, v, cfg, index=index), results[0][0])


def test_step_errors_name_the_stage(device):
    """A shape a stage refuses (the gate takes at most 128 past blocks) fails
    with that stage's message, as the stage called alone."""
    cfg = MoBAConfig(block_size=16, top_k=200, dtype=torch.float32)
    q, k, v = make_qkv((1, 4096, 1, 64), torch.float32, device=device)
    for call in (lambda: build_csc_fused(q, k, cfg), lambda: moba_forward(q, k, v, cfg)):
        with pytest.raises(ValueError, match="moba_gate: gate supports at most 128"):
            call()


# Where the (m, l) pairs are cleared: beside the one-launch middle of the index
# build on short calls, by the attention stage on others (few and many columns,
# one and several rows).
@pytest.mark.parametrize("s,b,hq,hk,bs,k", [(515, 2, 4, 2, 64, 4), (20011, 1, 4, 2, 64, 5),
                                            (9000, 3, 8, 1, 128, 3), (32 * 4099 + 3, 1, 1, 1, 32, 2)])
def test_step_clears_unwritten_slots(device, s, b, hq, hk, bs, k):
    """Memory that held finite values before: slots without a block are still
    left out of the merge."""
    cfg = MoBAConfig(block_size=bs, top_k=k, dtype=torch.bfloat16)
    q, do = make_qkv((b, s, hq, 64), torch.bfloat16, seed=3, device=device, n=2)
    kk, v = make_qkv((b, s, hk, 64), torch.bfloat16, seed=4, device=device, n=2)
    index = build_csc_fused(q, kk, cfg)
    results = []
    for given in (index, None):
        x = [z.clone().requires_grad_(True) for z in (q, kk, v)]
        torch.cuda.empty_cache()
        old = torch.full((b * s * hq * k * 80,), 3.0, device=device)
        del old  # its block serves the next allocations
        out = moba_attention(*x, cfg, index=given)
        results.append((out.detach(), *torch.autograd.grad(out, x, do)))
    assert all(torch.equal(a, c) for a, c in zip(*results))


@pytest.mark.parametrize("d,bs,cuts", [(64, 64, True), (32, 64, False), (64, 16, False)])
def test_segment_scratch_only_where_columns_are_cut(device, monkeypatch, d, bs, cuts):
    """The stages called one by one: no scratch for segments at shapes whose
    kernels run whole columns, and the same gradients as the step's."""
    monkeypatch.setenv("MOBA_SEGMENT_ENTRIES", "64")
    cfg = MoBAConfig(block_size=bs, top_k=3, dtype=torch.float32)
    q, do = make_qkv((1, 700, 4, d), torch.float32, seed=5, device=device, n=2)
    k, v = make_qkv((1, 700, 2, d), torch.float32, seed=6, device=device, n=2)
    scratch, call = [], _lib.call

    def spy(name, *args):
        if name == "moba_bwd":
            scratch.append(args[-7])  # scratch, scratch_cap, causal, three dtypes, stream
        return call(name, *args)

    monkeypatch.setattr(_lib, "call", spy)
    grads = []
    for index in (build_csc_fused(q, k, cfg), None):
        x = [t.clone().requires_grad_(True) for t in (q, k, v)]
        grads.append(torch.autograd.grad(moba_attention(*x, cfg, index=index), x, do))
    assert [s is not None for s in scratch] == [cuts]
    assert all(torch.equal(a, b) for a, b in zip(*grads))
