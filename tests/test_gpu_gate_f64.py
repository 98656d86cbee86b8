"""The float64 matrix gate (csrc/gate_f64.hip) at the edges of what it takes.

Calls with few blocks per row (and every float32 call at head_dim 64 / 128)
run it; the same queries against a kbar padded with further rows (ids no
query may rank) have more blocks per row and run the approximate kernels
(16-bit types). Both must give the same ids, and the oracle's.
"""

import pytest
import torch

from conftest import oracle_cfg
from moba import _lib
from moba.config import MoBAConfig
from moba.kernels.pooling import pool_blocks
from oracle import c_oracle

pytestmark = pytest.mark.gpu


def _gate(q, kbar, cfg, rows, take, cu=None):
    b, s, h, d = q.shape
    seqs = b if cu is None else cu.numel() - 1
    out = torch.full((b, h, s, cfg.slots()), -7, dtype=torch.int32, device=q.device)
    ws = torch.zeros(int(_lib.load().moba_gate_workspace_size(seqs, rows, h)), dtype=torch.uint8,
                     device=q.device)
    _lib.call("moba_gate", _lib.ptr(q), _lib.ptr(kbar), _lib.ptr(out), _lib.ptr(cu), seqs, s, rows,
              h, kbar.shape[1], d, kbar.shape[2], cfg.block_size, cfg.slots(), take,
              int(cfg.always_select_current), _lib.DTYPE_CODE[q.dtype], _lib.ptr(ws), ws.numel(),
              _lib.stream_handle(q.device))
    return out


def _padded(kbar, n):
    pad = torch.full(kbar.shape[:2] + (n - kbar.shape[2], kbar.shape[3]), 9.0, dtype=kbar.dtype,
                     device=kbar.device)
    return torch.cat((kbar, pad), 2).contiguous()


def _shifted(t):
    """The same values off a 16-byte boundary: the approximate kernels."""
    buf = torch.empty(t.numel() + 4, device=t.device, dtype=t.dtype)
    buf[4:] = t.reshape(-1)
    return buf[4:].view(t.shape)


# (S, query heads, kv heads, head_dim, block, top_k): one query, one block,
# a tile of 16 blocks or queries less / exactly / plus one, the last block
# counts of the rule, list lengths 1, 4, 5, 8, 9 and 16 and slots left over.
CASES = [(1, 1, 1, 64, 16, 4), (15, 2, 1, 64, 16, 1), (16 * 16 + 1, 2, 2, 64, 16, 2),
         (17 * 16 - 3, 2, 1, 128, 16, 5), (96 * 16, 2, 2, 64, 16, 6), (64 * 32 - 1, 4, 2, 128, 32, 9),
         (255 * 16 + 16, 1, 1, 64, 16, 10), (255 * 16 - 5, 2, 1, 128, 16, 17), (3 * 128, 2, 2, 64, 128, 16)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("case", CASES)
def test_gate_f64_matches_oracle_and_general_path(device, case, dtype):
    s, hq, hk, d, bs, k = case
    cfg = MoBAConfig(block_size=bs, top_k=k, dtype=dtype)
    g = torch.Generator().manual_seed(s + d)
    q = torch.randn((2, s, hq, d), generator=g).to(dtype).to(device)
    kk = torch.randn((2, s, hk, d), generator=g) + 3.0 * torch.randn((1, 1, hk, d), generator=g)
    kbar = pool_blocks(kk.to(dtype).to(device), cfg)
    n = kbar.shape[2]
    take = cfg.past_blocks_selected(n)
    got = _gate(q, kbar, cfg, s, take)
    ref = c_oracle.gate_select(q.cpu(), kbar.cpu(), oracle_cfg(cfg))
    assert torch.equal(got.cpu(), ref)
    if dtype != torch.float32:
        assert torch.equal(got, _gate(q, _padded(kbar, 300), cfg, s, take))
        assert torch.equal(got, _gate(_shifted(q), kbar, cfg, s, take))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", ["ties", "inf_nan", "tiny", "huge"])
def test_gate_f64_special_values_match_general_path(device, kind, dtype):
    """Ties in every place, inf and NaN (which never rank), scores that
    round to 0 or overflow: the ids of the approximate kernels, whose
    unsettled queries are rescored one by one. Without the own block too."""
    cfg = MoBAConfig(block_size=16, top_k=5, dtype=dtype, always_select_current=kind != "ties")
    lens = [700, 33, 1, 417]
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).to(device)
    g = torch.Generator().manual_seed(5)
    q = torch.randn((1, sum(lens), 4, 64), generator=g)
    kbar = torch.randn((len(lens), 2, 44, 64), generator=g)
    if kind == "ties":
        q, kbar = q.sign(), (kbar * 0.4).round()
    elif kind == "inf_nan":
        kbar[0, 0, 3, 5], kbar[0, 1, 7, 0], kbar[0, 0, 20, 1] = float("inf"), float("nan"), -float("inf")
        q[0, 300, 1, 2], q[0, 500:, 2, 3] = float("nan"), -float("inf")
    elif kind == "tiny":
        q, kbar = q * 1e-5, kbar * 1e-3
    else:
        q, kbar = q * 2e3, kbar * 10.0
    q, kbar = q.to(dtype).to(device), kbar.to(dtype).to(device)
    take = cfg.past_blocks_selected(44)
    got = _gate(q, kbar, cfg, max(lens), take, cu)
    assert torch.equal(got, _gate(q, _padded(kbar, 300), cfg, max(lens), take, cu))


# With lists over 8 and 256 blocks or more, the first 240 (head_dim 64) or 128
# blocks' queries, to a whole 128-query tile, go to these kernels and the rest
# to the approximate ones, if they are 65536 or more. (lengths, query heads,
# kv heads, head_dim, block, blocks per row, top_k): lines on a tile and inside
# one, sequences that end before, on, one past and far past the line, exactly
# 65536 queries and fewer.
SPLITS = [([255 * 16 + 1], 18, 1, 64, 16, 256, 17), ([256 * 17], 17, 1, 64, 17, 256, 10),
          ([3840], 18, 2, 64, 16, 300, 13), ([3841, 100, 3839, 3900, 1], 4, 2, 64, 16, 300, 13),
          ([2048, 2049, 4096, 700], 8, 2, 128, 16, 256, 10), ([257 * 20], 26, 2, 128, 20, 257, 17),
          ([3841, 3900], 2, 2, 64, 16, 256, 12)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("offset", [0.0, 3.0])
@pytest.mark.parametrize("case", SPLITS)
def test_gate_split_by_position_matches_oracle_and_general_path(device, case, offset, dtype):
    lens, hq, hk, d, bs, n, k = case
    cfg = MoBAConfig(block_size=bs, top_k=k, dtype=dtype)
    g = torch.Generator().manual_seed(len(lens) + d)
    q = torch.randn((1, sum(lens), hq, d), generator=g).to(dtype)
    kbar = torch.randn((len(lens), hk, n, d), generator=g) * bs ** -0.5 + offset * torch.randn(
        (1, hk, 1, d), generator=g)
    kbar = kbar.to(dtype)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    take, qd, kd, cud = k - 1, q.to(device), kbar.to(device), cu.to(device)
    got = _gate(qd, kd, cfg, max(lens), take, cud)
    assert torch.equal(got, _gate(_shifted(qd), kd, cfg, max(lens), take, cud))
    need = -(-max(lens) // bs)  # the oracle's rows: what the longest sequence has
    ref = c_oracle.gate_select(q, kbar[:, :, :need].contiguous(), oracle_cfg(cfg), cu, max(lens))
    assert torch.equal(got.cpu(), ref)


def _off_by_one(t):
    """The same float32 values 4 bytes off a 16-byte boundary: gate_exact_kernel."""
    buf = torch.empty(t.numel() + 1, device=t.device, dtype=t.dtype)
    buf[1:] = t.reshape(-1)
    return buf[1:].view(t.shape)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("kind", ["ties", "inf_nan", "tiny", "huge"])
def test_gate_f64_float32_special_values_match_exact_path(device, kind, d):
    """As above in float32: inf and NaN never rank, scores that round to 0 or
    overflow tie. The ids of the exact kernel and of the oracle."""
    cfg = MoBAConfig(block_size=16, top_k=5, dtype=torch.float32, always_select_current=kind != "ties")
    lens = [700, 33, 1, 417]
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    g = torch.Generator().manual_seed(6)
    q = torch.randn((1, sum(lens), 4, d), generator=g)
    kbar = torch.randn((len(lens), 2, 44, d), generator=g)
    if kind == "ties":
        q, kbar = q.sign(), (kbar * 0.4).round()
    elif kind == "inf_nan":
        kbar[0, 0, 3, 5], kbar[0, 1, 7, 0], kbar[0, 0, 20, 1] = float("inf"), float("nan"), -float("inf")
        q[0, 300, 1, 2], q[0, 500:, 2, 3] = float("nan"), -float("inf")
    elif kind == "tiny":  # products of 1e-46 and below: most scores round to 0
        q, kbar = q * 1e-23, kbar * 1e-23
    else:  # of 1e40: most scores overflow
        q, kbar = q * 1e20, kbar * 1e20
    take, cud = cfg.past_blocks_selected(44), cu.to(device)
    qd, kd = q.to(device), kbar.to(device)
    got = _gate(qd, kd, cfg, max(lens), take, cud)
    assert torch.equal(got, _gate(_off_by_one(qd), kd, cfg, max(lens), take, cud))
    assert torch.equal(got.cpu(), c_oracle.gate_select(q, kbar, oracle_cfg(cfg), cu, max(lens)))
