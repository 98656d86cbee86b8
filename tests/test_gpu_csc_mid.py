"""The CSC build's three-launch form (csrc/csc.hip:csc_mid_kernel) against the
general one. Both place a column's entries in (query head, row) order, so
every array is the same; a call with more columns than the short form takes
(the further ones empty) runs the general one.
"""

import pytest
import torch

from moba.config import MoBAConfig
from moba.kernels.routing import build_csc_from_indices

pytestmark = pytest.mark.gpu

# (lengths or S, batch, query heads, kv heads, columns, slots): one entry per
# query (rows of ids in halves), queries that straddle rows of ids, one tile
# and one column, far more columns than it takes (the general build on both
# sides), the last unit count taken with 64-query units and one more, packed
# sequences down to one token, the last column count taken, with the last unit
# count and two more, and one more column.
CASES = [(1000, 2, 4, 2, 16, 1), (777, 1, 6, 2, 7, 3), (9, 1, 1, 1, 1, 5), (2048, 1, 1, 1, 1024, 8),
         (64 * 32, 1, 4, 1, 256, 4), (64 * 32 + 1, 1, 4, 1, 256, 4), (600, 3, 3, 3, 33, 17),
         ([300, 1, 64, 555, 2], 1, 4, 2, 20, 4), ([5, 40], 1, 8, 1, 3, 64),
         (48 * 64, 1, 2, 1, 320, 8), (48 * 64 + 1, 1, 2, 1, 320, 8), (3210, 1, 1, 1, 321, 8)]


@pytest.mark.parametrize("entries", ["0", "24"])
@pytest.mark.parametrize("case", CASES)
def test_short_form_equals_general_build(device, monkeypatch, case, entries):
    monkeypatch.setenv("MOBA_SEGMENT_ENTRIES", entries)
    s, b, hq, hk, nb, slots = case
    lens = s if isinstance(s, list) else None
    t, longest = (sum(lens), max(lens)) if lens else (s, s)
    bs = -(-longest // nb)
    cfg = MoBAConfig(block_size=bs, top_k=slots)
    g = torch.Generator().manual_seed(t + slots)
    pos = torch.cat([torch.arange(n) for n in lens]) if lens else torch.arange(s)
    own = (pos // bs)[None, None, :, None]
    # Ids a query may hold, each at most once, ascending, -1 padded.
    ids = torch.rand((b, hq, t, nb), generator=g).masked_fill(torch.arange(nb) > own, 2.0)
    val, at = ids.topk(min(slots, nb), dim=-1, largest=False)
    at = torch.where((val < 2.0) & (torch.rand(val.shape, generator=g) < 0.9), at, nb).sort(-1).values
    ids = torch.full((b, hq, t, slots), -1, dtype=torch.int32)
    ids[..., :at.shape[-1]] = torch.where(at < nb, at, -1).to(torch.int32)
    ids = ids.to(device)
    kw = {}
    if lens:
        kw = {"cu_seqlens": torch.tensor([0] + lens).cumsum(0).to(torch.int32).to(device),
              "max_seqlen": longest}
    small = build_csc_from_indices(ids, nb, cfg, num_kv_heads=hk, **kw)
    wide = build_csc_from_indices(ids, 1100, cfg, num_kv_heads=hk, **kw)
    assert torch.equal(small.col_nnz, wide.col_nnz[..., :nb])
    assert int(wide.col_nnz[..., nb:].sum()) == 0
    assert torch.equal(small.col_offsets, wide.col_offsets[..., :nb + 1])
    total = small.col_offsets[..., nb]
    live = torch.arange(small.row_indices.shape[-1], device=device) < total[..., None]
    for name in ("row_indices", "head_indices", "slot_of_pair"):
        assert torch.equal(getattr(small, name)[live], getattr(wide, name)[live]), name
    for i in range(small.col_nnz.shape[0]):
        for h in range(hk):
            want = [c for c in wide.order[i, h].tolist() if c < nb]
            assert small.order[i, h].tolist() == want
            if small.segments is None:
                continue
            n, cut = small.seg_counts[i, h].tolist()
            assert cut == int(wide.seg_counts[i, h, 1])
            rows = [x for x in wide.segments[i, h, :int(wide.seg_counts[i, h, 0])].tolist() if x[0] < nb]
            assert small.segments[i, h, :n].tolist() == rows
            assert torch.equal(small.seg_split[i, h, :cut], wide.seg_split[i, h, :cut])
