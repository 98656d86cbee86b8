"""Workloads of MoBA attention whose times and results are tracked.

A case is one call that a program makes through the public entry points: a
training step of the attention layer (`moba_attention` and its backward), a
forward for inference (`moba_forward`), the packed [T, H, D] signature
(`moba_attn_varlen_triton`), or the routing stage alone (`pool_blocks`,
`gate_select`). Sizes are those of this repository's benchmark, tests and
baseline configurations, and of the ranges around them.

The ranges (`draw`): 256 to 512K tokens; one to sixteen batch rows or two to
64 packed sequences, lengths mostly no multiple of the block; 1 to 32 query
heads over 1 to 8 kv heads; head_dim 64 and 128; block size 32, 64 and 128;
top_k 2 to 16; bfloat16, float16 and (at lengths where full precision is
asked for: reference runs, gradient checks) float32; keys i.i.d., with a
per-channel offset shared by every token as trained keys have, or drifting
along the sequence.
"""

import math
import sys
from pathlib import Path

import torch

# The package folder's name is no module name: its modules are found there.
_PKG = str(Path.cwd() / "moba-triton_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

from implementations.triton_moba import moba_attn_varlen_triton  # noqa: E402
from moba.config import MoBAConfig  # noqa: E402
from moba.kernels.attention import moba_attention  # noqa: E402
from moba.kernels.gating import gate_select  # noqa: E402
from moba.kernels.moba_fwd import moba_forward  # noqa: E402
from moba.kernels.pooling import pool_blocks  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _case(name, mode, dtype, batch, seq, heads, kv_heads, head_dim, block, top_k,
          keys="iid", packed=0, shortest=0):
    """batch x seq tokens; `packed` > 0 instead packs that many sequences of
    lengths between `shortest` and `seq` (drawn from the sizes alone)."""
    return {"name": name, "mode": mode, "dtype": dtype, "batch": batch, "seq": seq,
            "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim, "block": block,
            "top_k": top_k, "keys": keys, "packed": packed, "shortest": shortest}


def listed():
    return [
        # The smallest training step: a short sequence, where launches and
        # host work are most of the time.
        _case("train_2k", "train", "bf16", 1, 2048, 4, 4, 64, 128, 8),
        # A small inference batch of grouped-query layers, ragged length.
        _case("prefill_4x1000_gqa", "infer", "bf16", 4, 1000, 16, 4, 128, 64, 4),
        # Inference over a long prompt.
        _case("prefill_64k", "infer", "bf16", 1, 65536, 4, 4, 64, 128, 8),
        # Training steps on long sequences: the length most runs use, and the
        # longest (the benchmark's workload).
        _case("train_128k", "train", "bf16", 1, 131072, 4, 4, 64, 128, 8),
        _case("train_512k", "train", "bf16", 1, 524288, 4, 4, 64, 128, 8),
        # A grouped-query layer of a large model, head_dim 128.
        _case("train_gqa_32k_d128", "train", "bf16", 1, 32768, 32, 8, 128, 128, 8),
        # Documents packed into one row: a few long ones, and many short ones.
        _case("train_varlen_long", "train", "bf16", 1, 131072, 4, 4, 64, 128, 8,
              packed=8, shortest=2048),
        _case("train_varlen_short", "varlen", "bf16", 1, 4096, 16, 4, 128, 64, 4,
              packed=24, shortest=200),
        # Half precision, small blocks and many of them per query, trained
        # keys, a length that is no multiple of the block.
        _case("train_fp16_ragged", "train", "fp16", 2, 20011, 8, 2, 64, 64, 12, keys="offset"),
        # Full precision: a forward at the size of the fp32 configuration and
        # a training step of grouped-query heads.
        _case("fp32_fwd_4k", "infer", "fp32", 1, 4096, 4, 4, 64, 128, 8),
        _case("fp32_train_8k_gqa", "train", "fp32", 1, 8192, 8, 2, 64, 64, 8),
        # Routing alone, as a program does that keeps the routing of one
        # layer for others; keys drift along the sequence.
        _case("route_256k_d128", "route", "bf16", 1, 262144, 4, 2, 128, 128, 8, keys="walk"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    # Cost limits: the longest listed step for 16-bit types, and for float32
    # a sixteenth of that (the products of its steps run at full precision).
    top = listed()[4]
    top_flops, top_pairs = work(top)["flops"], 524288 * 4 * 64 * 8
    while True:
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
        mode = rng.choice(["train", "train", "infer", "varlen", "route"])
        kv_heads = rng.choice([1, 2, 4, 4, 8])
        heads = kv_heads * rng.choice([1, 1, 2, 4])
        head_dim = rng.choice([64, 64, 128])
        block = rng.choice([32, 64, 128, 128])
        top_k = rng.choice([2, 3, 4, 6, 8, 8, 12, 16])
        packed, shortest, batch = 0, 0, 1
        if mode == "varlen" or (mode != "route" and rng.random() < 0.2):
            packed = _log_int(rng, 2, 64)
            longest = _log_int(rng, 256, 131072)
            shortest = max(1, longest // rng.choice([2, 8, 64]))
            seq = longest
        else:
            batch = rng.choice([1, 1, 1, 2, 3, 4, 16])
            seq = _log_int(rng, 256, 524288)
        if seq > 1024 and rng.random() < 0.4:
            seq -= seq % 128
        case = _case("", mode, dtype, batch, seq, heads, kv_heads, head_dim, block, top_k,
                     rng.choice(["iid", "iid", "offset", "walk"]), packed, shortest)
        share = 1 / 16 if dtype == "fp32" else 1
        pairs = sum(_lengths(case)) * heads * head_dim * top_k
        if 256 <= sum(_lengths(case)) <= 1 << 20 and pairs <= share * top_pairs and \
                work(case)["flops"] <= share * top_flops:
            del case["name"]
            return case


def _lengths(case):
    """Sequence lengths: batch rows, or the packed documents'."""
    if not case["packed"]:
        return [case["seq"]] * case["batch"]
    n, lo, hi = case["packed"], case["shortest"], case["seq"]
    # Spread over [lo, hi] by the golden ratio's multiples: uneven, the same
    # for a case whatever the seed, the longest one first reached by hi.
    frac = [(i * 0.6180339887498949) % 1.0 for i in range(n)]
    return [hi] + [lo + int((hi - lo) * f) for f in frac[1:]]


def _config(case):
    return MoBAConfig(block_size=case["block"], top_k=case["top_k"], dtype=DTYPES[case["dtype"]])


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    lens = _lengths(case)
    b = 1 if case["packed"] else case["batch"]
    s = sum(lens) // b
    hq, hkv, d = case["heads"], case["kv_heads"], case["head_dim"]

    def normal(h):
        return torch.randn((b, s, h, d), generator=g, device=dev, dtype=torch.float32)

    q, k, v = normal(hq), normal(hkv), normal(hkv)
    if case["keys"] == "offset":
        k = k + 3.0 * torch.randn((1, 1, hkv, d), generator=g, device=dev)
    elif case["keys"] == "walk":
        step = torch.randn((b, s, hkv, d), generator=g, device=dev) * (3.0 / math.sqrt(s))
        k = k + step.cumsum(1)
    q, k, v = q.to(dt), k.to(dt), v.to(dt)
    state = {"case": case, "cfg": _config(case), "q": q, "k": k, "v": v, "kw": {}}
    if case["packed"]:
        cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).to(dev)
        state["kw"] = {"cu_seqlens": cu, "max_seqlen": max(lens)}
    if case["mode"] == "varlen":
        state.update(q=q[0], k=k[0], v=v[0])
    if case["mode"] in ("train", "varlen"):
        do = normal(hq).to(dt)
        state["do"] = do[0] if case["mode"] == "varlen" else do
        for n in ("q", "k", "v"):
            state[n].requires_grad_(True)
    return state


def run(state):
    mode, cfg, kw = state["case"]["mode"], state["cfg"], state["kw"]
    q, k, v = state["q"], state["k"], state["v"]
    if mode == "route":
        kbar = pool_blocks(k, cfg, **kw)
        return {"kbar": kbar, "ids": gate_select(q, kbar, cfg, **kw)}
    if mode == "infer":
        return {"out": moba_forward(q, k, v, cfg, **kw)}
    if mode == "varlen":
        out = moba_attn_varlen_triton(q, k, v, kw["cu_seqlens"], kw["max_seqlen"],
                                      cfg.block_size, cfg.top_k)
    else:
        out = moba_attention(q, k, v, cfg, **kw)
    dq, dk, dv = torch.autograd.grad(out, (q, k, v), state["do"])
    return {"out": out.detach(), "dq": dq, "dk": dk, "dv": dv}


def work(case):
    """Inputs read once and outputs written once; the scores of every
    strictly-past block (the gate) and, on the selected blocks' visible
    keys, the products of the forward (2) and the backward (5 with the
    scores again)."""
    e = torch.empty((), dtype=DTYPES[case["dtype"]]).element_size()
    d, bs = case["head_dim"], case["block"]
    past_budget = case["top_k"] - 1
    gate = pairs = 0
    for n in _lengths(case):
        for j in range(-(-n // bs)):
            rows = min(bs, n - j * bs)
            gate += rows * j
            pairs += rows * (rows + 1) // 2 + rows * bs * min(past_budget, j)
    tokens = sum(_lengths(case))
    nq, nkv = tokens * case["heads"] * d, tokens * case["kv_heads"] * d
    flops = 2 * d * gate * case["heads"]
    if case["mode"] == "route":
        nb = sum(-(-n // bs) for n in _lengths(case))
        return {"bytes": e * (nq + nkv + nb * case["kv_heads"] * d) +
                4 * tokens * case["heads"] * case["top_k"], "flops": flops}
    flops += 4 * d * pairs * case["heads"]
    bytes_ = e * (2 * nq + 2 * nkv)
    if case["mode"] != "infer":
        flops += 10 * d * pairs * case["heads"]
        bytes_ += e * (2 * nq + 2 * nkv)  # dO and dQ; dK and dV
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """Routing is exact in every type. The rest is about four times the
    distance from the 64-bit values that the types give: probabilities,
    their gradients and the per-block partial rows are rounded to 16 bits
    before they are summed in 32. dQ sums dS K with sum dS = 0, so a part
    shared by all keys cancels in the exact result and its rounding stays."""
    if case["mode"] == "route":
        return "exact"
    rel = {"bf16": {"iid": 1.2e-2, "walk": 2.2e-2, "offset": 4.6e-2},
           "fp16": {"iid": 1.5e-3, "walk": 2.8e-3, "offset": 6e-3},
           "fp32": {"iid": 5e-6, "walk": 5e-6, "offset": 5e-6}}
    return {"rel": rel[case["dtype"]][case["keys"]]}


# ---------------------------------------------------------------------------
# The same results in 64 bits.
# ---------------------------------------------------------------------------
def _exact_means(k, bs, dt):
    """Block representatives [nb, D] of k [n, D] float64: the sum rounded to
    the dtype, divided by the keys in the block and rounded again."""
    n = k.shape[0]
    nb = -(-n // bs)
    pad = torch.zeros((nb * bs, k.shape[1]), dtype=torch.float64, device=k.device)
    pad[:n] = k
    total = pad.view(nb, bs, -1).sum(1).to(torch.float32).to(dt)
    count = torch.full((nb, 1), bs, device=k.device)
    count[-1] = n - (nb - 1) * bs
    return (total.float() / count.float()).to(dt)


def _exact_select(q, kbar, bs, take, dt):
    """Past blocks [n, take] of q [n, D] float64 (-1 where there are fewer):
    score exact, rounded to float32 and to the dtype; ties to the lower id."""
    n, nb = q.shape[0], kbar.shape[0]
    take = min(take, nb)
    out = torch.full((n, take), -1, dtype=torch.int64, device=q.device)
    kb = kbar.double().t().contiguous()
    rows = max(bs, (1 << 25) // max(nb, 1) // bs * bs)
    lowest = torch.iinfo(torch.int64).min
    for t0 in range(0, n, rows):
        t1 = min(n, t0 + rows)
        hz = (t1 - 1) // bs
        if hz == 0 or take == 0:
            continue
        x = (q[t0:t1] @ kb[:, :hz]).float().to(dt).float() + 0.0
        i = x.view(torch.int32)
        i = torch.where(i < 0, i ^ 0x7FFFFFFF, i).long()
        ids = torch.arange(hz, device=q.device)
        key = i * (1 << 24) + ((1 << 24) - 1 - ids)
        own = torch.arange(t0, t1, device=q.device)[:, None] // bs
        key = torch.where(ids[None] < own, key, lowest)
        best, at = key.topk(min(take, hz), dim=1)
        out[t0:t1, :at.shape[1]] = torch.where(best > lowest, at, -1)
    return out


def _exact_head(q, k, v, do, ids, bs, dk, dv):
    """One query head of one sequence, float64: (out, dq); adds its dK and
    dV. ids [n, slots] are the selected blocks, -1 for none."""
    n, d = q.shape
    nb = -(-n // bs)
    scale = d ** -0.5
    flat = torch.where(ids >= 0, ids, nb).flatten()
    order = flat.sort(stable=True).indices
    row_of = order // ids.shape[1]
    counts = torch.bincount(flat, minlength=nb + 1)[:nb].tolist()
    pos = torch.arange(n, device=q.device)
    m = torch.full((n,), -math.inf, dtype=torch.float64, device=q.device)
    l = torch.zeros_like(m)
    out = torch.zeros_like(q)

    def blocks():
        at = 0
        for j, c in enumerate(counts):
            rows, at = row_of[at:at + c], at + c
            if c:
                lo, hi = j * bs, min(n, j * bs + bs)
                qr = q[rows]
                s = qr @ k[lo:hi].t() * scale
                s = s.masked_fill(pos[lo:hi][None] > rows[:, None], -math.inf)
                yield rows, lo, hi, qr, s

    for rows, lo, hi, _, s in blocks():
        m[rows] = torch.maximum(m[rows], s.max(1).values)
    for rows, lo, hi, _, s in blocks():
        p = (s - m[rows][:, None]).exp()
        l[rows] += p.sum(1)
        out[rows] += p @ v[lo:hi]
    out /= l[:, None]
    if do is None:
        return out, None
    dq = torch.zeros_like(q)
    delta = (out * do).sum(1)
    for rows, lo, hi, qr, s in blocks():
        p = (s - m[rows][:, None]).exp() / l[rows][:, None]
        dor = do[rows]
        dv[lo:hi] += p.t() @ dor
        ds = p * (dor @ v[lo:hi].t() - delta[rows][:, None]) * scale
        dk[lo:hi] += ds.t() @ qr
        dq[rows] += ds @ k[lo:hi]
    return out, dq


def exact(case, seed):
    # A few launches per (block, query head) and pass.
    if sum(-(-n // case["block"]) for n in _lengths(case)) * case["heads"] > 40000:
        return None
    st = prepare(case, seed)
    dt, bs, mode = DTYPES[case["dtype"]], case["block"], case["mode"]
    lens = _lengths(case)
    hq, hkv, d = case["heads"], case["kv_heads"], case["head_dim"]
    # One token axis: batch rows and packed sequences alike follow each other.
    q, k, v = (st[n].detach().reshape(-1, h, d).double()
               for n, h in (("q", hq), ("k", hkv), ("v", hkv)))
    do = st["do"].reshape(-1, hq, d).double() if "do" in st else None
    take = case["top_k"] - 1
    if mode == "route":
        nb = -(-max(lens) // bs)
        means = torch.zeros((len(lens), hkv, nb, d), dtype=torch.float64, device=q.device)
        ids = torch.full((len(lens), hq, max(lens), case["top_k"]), -1, dtype=torch.int64,
                         device=q.device)
    out = torch.empty_like(q)
    dq, dk, dv = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
    t0 = 0
    for r, n in enumerate(lens):
        own = (torch.arange(n, device=q.device) // bs)[:, None]
        for h in range(hq):
            hk = h // (hq // hkv)
            at = (slice(t0, t0 + n), h)
            kh = k[t0:t0 + n, hk].contiguous()
            kbar = _exact_means(kh, bs, dt)
            qh = q[at].contiguous()
            sel = torch.cat((_exact_select(qh, kbar, bs, take, dt), own), 1)
            if mode == "route":
                means[r, hk] = kbar.double()
                big = torch.where(sel >= 0, sel, 1 << 40).sort(1).values
                ids[r, h, :, :sel.shape[1]] = torch.where(big < 1 << 40, big, -1)
                continue
            out[at], g = _exact_head(
                qh, kh, v[t0:t0 + n, hk].contiguous(),
                None if do is None else do[at].contiguous(), sel, bs,
                dk[t0:t0 + n, hk], dv[t0:t0 + n, hk])
            if g is not None:
                dq[at] = g
        t0 += n
    if mode == "route":
        return {"kbar": means, "ids": ids}
    shape_q, shape_k = st["q"].shape, st["k"].shape
    if mode == "infer":
        return {"out": out.view(shape_q)}
    return {"out": out.view(shape_q), "dq": dq.view(shape_q), "dk": dk.view(shape_k),
            "dv": dv.view(shape_k)}
