"""moba_step on the host: the binding's struct is the header's, sizes follow
the shapes, bad shapes are refused before any launch."""

import ctypes
import re
from pathlib import Path

import pytest

from moba import _lib

HEADER = Path(__file__).resolve().parents[1] / "include" / "moba_hip.h"


def _step(**kw):
    base = dict(batch=1, seq_len=2048, max_seqlen=2048, h_q=4, h_kv=2, head_dim=64, block_size=128,
                slots=8, take=7, always_current=1, causal=1, dtype=0, dkv_dtype=0, keep=1, packed=0,
                seg_len=512, max_seg=8)
    return _lib.Step(**{**base, **kw})


def test_struct_matches_header():
    body = re.search(r"typedef struct moba_step \{(.*?)\} moba_step;", HEADER.read_text(), re.S).group(1)
    body = re.sub(r"/\*.*?\*/", "", body, flags=re.S)
    names = [n.strip().lstrip("*").split()[-1].lstrip("*") for decl in body.split(";") if decl.strip()
             for n in decl.split(",")]
    assert names == [f[0] for f in _lib.Step._fields_]
    assert ctypes.sizeof(_lib.Step) == 8 * len(names)


def test_layout_sizes():
    a = _step()
    _lib.run_step("moba_step_layout", a)
    assert a.n_blocks == 16
    partials = 4 * 2048 * 8
    assert a.saved_bytes >= 12 * partials + 8 * partials + 4 * 4 * 2048
    assert a.forward_temp == a.backward_temp >= partials * 64 * 2 + 8 * 4 * 2048
    infer = _step(keep=0)
    _lib.run_step("moba_step_layout", infer)
    assert infer.saved_bytes < a.saved_bytes and infer.forward_temp < a.forward_temp
    packed = _step(packed=1, batch=3, seq_len=3000)  # 3 sequences of up to 2048 tokens
    _lib.run_step("moba_step_layout", packed)
    assert packed.n_blocks == 16 and packed.saved_bytes > 12 * 3 * partials


@pytest.mark.parametrize("bad", [dict(seq_len=0), dict(h_q=3), dict(slots=0), dict(head_dim=0),
                                 dict(packed=1, max_seqlen=0), dict(dtype=7), dict(seg_len=-1)])
def test_bad_shapes_are_refused(bad):
    for name, stream in (("moba_step_layout", ()), ("moba_forward_step", (None,)),
                         ("moba_backward_step", (None,))):
        with pytest.raises(ValueError, match=name):
            _lib.run_step(name, _step(**bad), *stream)


def test_null_buffers_are_refused():
    with pytest.raises(ValueError, match="null pointer"):
        _lib.run_step("moba_forward_step", _step(), None)
    with pytest.raises(ValueError, match="kept nothing"):
        _lib.run_step("moba_backward_step", _step(keep=0), None)


@pytest.mark.parametrize("dtype", [0, 2])
@pytest.mark.parametrize("d,bs,cuts", [(64, 128, True), (128, 32, True), (256, 128, False), (64, 256, False)])
def test_segment_scratch_only_where_columns_are_cut(d, bs, cuts, dtype):
    """Scratch for the sums of cut columns' segments (2 block sums of dK and
    dV per segment, float64 for float32 inputs) only at shapes whose kernels
    cut columns."""
    sizes = []
    for seg_len in (0, 512):
        a = _step(head_dim=d, block_size=bs, dtype=dtype, seg_len=seg_len)
        _lib.run_step("moba_step_layout", a)
        sizes.append(a.backward_temp)
    if not cuts:
        assert sizes[1] == sizes[0]
        return
    extra = 2 * 2048 * 8 // 512  # of each of 2 (row, kv head) pairs
    scratch = 2 * 2 * extra * 2 * bs * d * (8 if dtype == 2 else 4)
    assert sizes[0] < sizes[1]
    assert sizes[1] >= 4 * 2048 * 8 * d * (4 if dtype == 2 else 2) + scratch
