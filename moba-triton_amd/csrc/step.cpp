// A whole forward or backward per call: the stages of moba_hip.h in order on
// one stream, their buffers carved from two allocations of the caller's.
//
// What it saves is host time. A caller that runs the stages one by one makes
// about twenty allocations and eight calls per training step; on short
// sequences the GPU waits for that. [1, 2048, 4, 64], 128-key blocks, top_k 8,
// bf16: forward and backward through autograd 322 us a pass stage by stage,
// 188 us here; the forward alone 119 and 57 us.
#include <hip/hip_runtime.h>

#include "common.h"

namespace moba {
namespace {

// Carves consecutive pieces from a buffer; with a null base it only adds up
// sizes. A piece starts on 256 bytes, a large one on a power of two up to
// 2 MiB and a sixteenth of its size, as allocations of their own would: with
// every piece on 256 bytes the (m, l) records of [1, 524288, 4, 64] lay off
// the pages, and the dQ reduce that reads them took 462 us instead of 441,
// the merge 455 instead of 449.
struct Carve {
  char* base;
  size_t at = 0;
  template <typename T>
  T* take(int64_t n) {
    const size_t bytes = (sizeof(T) * static_cast<size_t>(n) + 255) & ~size_t(255);
    size_t align = 256;
    while (align < (size_t(2) << 20) && align * 16 <= bytes) align *= 2;
    at = (at + align - 1) & ~(align - 1);
    T* p = base ? reinterpret_cast<T*>(base + at) : nullptr;
    at += bytes;
    return p;
  }
};

struct Shape {
  int64_t rps, cap, pairs, cols, rows, seg_cap, extra, esize, n;
  size_t gate_ws, csc_ws;
};

// What the backward reads.
struct Saved {
  int32_t *nnz, *offsets, *order, *entries, *seg, *split, *counts;
  float *ml, *lse;
  size_t bytes;
};

// The forward's own buffers. The partial rows take the place of everything
// that is dead once the index exists.
struct Temp {
  void *kbar, *gate_ws, *csc_ws, *acc;
  int32_t* ids;
  size_t bytes;
};

struct BackTemp {
  float *lse_delta, *scratch;
  void* dq_part;
  int64_t scratch_cap;
  size_t bytes;
};

Shape shape_of(const moba_step& s) {
  Shape h;
  h.rps = s.packed ? s.max_seqlen : s.seq_len;
  h.pairs = s.batch * s.h_kv;
  h.cap = s.h_q / s.h_kv * h.rps * s.slots;
  h.cols = h.pairs * s.n_blocks;
  h.rows = (s.packed ? 1 : s.batch) * s.h_q * s.seq_len;  // query rows of the partials
  h.n = h.rows * s.slots;
  h.extra = s.seg_len > 0 ? cdiv(h.cap, s.seg_len) : 0;
  h.seg_cap = s.n_blocks + h.extra;
  h.esize = s.dtype == MOBA_FP32 ? 4 : 2;
  h.gate_ws = moba_gate_workspace_size(s.batch, h.rps, s.h_q);
  h.csc_ws = moba_csc_workspace_size(s.batch, h.rps, s.h_q, s.h_kv, s.n_blocks, s.slots);
  return h;
}

Saved saved_of(const moba_step& s, const Shape& h) {
  Carve c{static_cast<char*>(s.saved)};
  Saved v;
  v.nnz = c.take<int32_t>(h.cols);
  v.offsets = c.take<int32_t>(h.cols + h.pairs);
  v.order = c.take<int32_t>(h.cols);
  v.entries = c.take<int32_t>(3 * h.pairs * h.cap);
  const bool list = s.seg_len > 0;
  v.seg = list ? c.take<int32_t>(4 * h.pairs * h.seg_cap) : nullptr;
  v.split = list ? c.take<int32_t>(h.pairs * h.extra) : nullptr;
  v.counts = list ? c.take<int32_t>(2 * h.pairs) : nullptr;
  v.ml = c.take<float>(2 * h.n);
  v.lse = s.keep ? c.take<float>(h.rows) : nullptr;
  v.bytes = c.at;
  return v;
}

Temp temp_of(const moba_step& s, const Shape& h) {
  Carve c{static_cast<char*>(s.temp)};
  Temp t;
  t.kbar = c.take<char>(h.cols * s.head_dim * h.esize);
  t.ids = c.take<int32_t>(h.n);
  t.gate_ws = c.take<char>(static_cast<int64_t>(h.gate_ws));
  t.csc_ws = c.take<char>(static_cast<int64_t>(h.csc_ws));
  Carve d{static_cast<char*>(s.temp)};
  t.acc = d.take<char>(h.n * s.head_dim * h.esize);
  t.bytes = c.at > d.at ? c.at : d.at;
  return t;
}

BackTemp back_temp_of(const moba_step& s, const Shape& h) {
  Carve c{static_cast<char*>(s.temp)};
  BackTemp t;
  t.lse_delta = c.take<float>(2 * h.rows);
  t.dq_part = c.take<char>(h.n * s.head_dim * h.esize);
  // Sums of cut columns' segments: float32, for float32 inputs float64 (two
  // slots each); none where the kernels run whole columns.
  t.scratch_cap = matrix_shape(s.head_dim, s.block_size) ? 2 * h.extra * (h.esize / 2) : 0;
  t.scratch = t.scratch_cap
                  ? c.take<float>(h.pairs * t.scratch_cap * 2 * s.block_size * s.head_dim)
                  : nullptr;
  t.bytes = c.at;
  return t;
}

int check(moba_step* s) {
  s->failed_stage = 0;
  if (s->batch <= 0 || s->seq_len <= 0 || s->h_q <= 0 || s->h_kv <= 0 || s->head_dim <= 0 ||
      s->block_size <= 0 || s->slots <= 0 || (s->packed && s->max_seqlen <= 0) || s->seg_len < 0)
    return fail(MOBA_ERR_INVALID, "non-positive shape argument");
  if (s->h_q % s->h_kv != 0)
    return fail(MOBA_ERR_INVALID, "query heads " + std::to_string(s->h_q) + " not divisible by kv heads " +
                                      std::to_string(s->h_kv));
  if (s->dtype < MOBA_BF16 || s->dtype > MOBA_FP32)
    return fail(MOBA_ERR_UNSUPPORTED, "unknown dtype code");
  return MOBA_OK;
}

}  // namespace
}  // namespace moba

extern "C" int moba_step_layout(moba_step* step) {
  using namespace moba;
  const int st = check(step);
  if (st) return st;
  step->n_blocks = cdiv(step->packed ? step->max_seqlen : step->seq_len, step->block_size);
  moba_step s = *step;
  s.saved = s.temp = nullptr;
  const Shape h = shape_of(s);
  step->saved_bytes = static_cast<int64_t>(saved_of(s, h).bytes);
  step->forward_temp = static_cast<int64_t>(temp_of(s, h).bytes);
  step->backward_temp = static_cast<int64_t>(back_temp_of(s, h).bytes);
  // One size for both: a caching allocator then hands the backward the block
  // the forward gave back.
  if (s.keep)
    step->forward_temp = step->backward_temp = step->forward_temp > step->backward_temp
                                                   ? step->forward_temp : step->backward_temp;
  return MOBA_OK;
}

extern "C" int moba_forward_step(moba_step* step, void* stream) {
  using namespace moba;
  int st = check(step);
  if (st) return st;
  const moba_step& s = *step;
  if (!s.saved || !s.temp || !s.out || (s.packed && !s.cu_seqlens))
    return fail(MOBA_ERR_INVALID, "null pointer");
  const Shape h = shape_of(s);
  const Saved v = saved_of(s, h);
  const Temp t = temp_of(s, h);
  const int32_t* cu = s.packed ? s.cu_seqlens : nullptr;
  const int dt = static_cast<int>(s.dtype);
  auto stage = [&](int n, int rc) {
    if (rc) step->failed_stage = n;
    return rc;
  };
  st = stage(1, moba_pool(s.k, t.kbar, cu, s.batch, s.seq_len, s.max_seqlen, s.h_kv, s.head_dim,
                          s.n_blocks, s.block_size, dt, stream));
  if (st) return st;
  st = stage(2, moba_gate(s.q, t.kbar, t.ids, cu, s.batch, s.seq_len, s.max_seqlen, s.h_q, s.h_kv,
                          s.head_dim, s.n_blocks, s.block_size, s.slots, s.take,
                          static_cast<int>(s.always_current), dt, t.gate_ws, h.gate_ws, stream));
  if (st) return st;
  bool cleared = false;
  st = stage(3, csc_build(t.ids, v.nnz, v.offsets, v.entries, v.entries + 1, v.entries + 2, v.order,
                          cu, s.batch, s.seq_len, h.rps, s.h_q, s.h_kv, s.n_blocks, s.slots, 3,
                          v.seg, v.split, v.counts, v.seg ? h.seg_cap : 0,
                          s.seg_len > 0 ? s.seg_len : 1, s.max_seg, t.csc_ws, h.csc_ws, stream,
                          v.ml, 2 * h.n, &cleared));
  if (st) return st;
  st = stage(4, attend(s.q, s.k, s.v, v.nnz, v.offsets, v.entries, v.entries + 1, v.entries + 2,
                       v.order, v.ml, t.acc, cu, s.batch, s.seq_len, s.max_seqlen, s.h_q, s.h_kv,
                       s.head_dim, s.n_blocks, s.block_size, s.slots, h.cap, 3, v.seg, v.split,
                       v.counts, v.seg ? h.seg_cap : 0, static_cast<int>(s.causal), dt, dt, stream,
                       cleared));
  if (st) return st;
  return stage(5, moba_combine(v.ml, t.acc, s.out, v.lse, s.packed ? 1 : s.batch, s.seq_len, s.h_q,
                               s.head_dim, s.slots, dt, dt, stream));
}

extern "C" int moba_backward_step(moba_step* step, void* stream) {
  using namespace moba;
  int st = check(step);
  if (st) return st;
  const moba_step& s = *step;
  if (!s.keep) return fail(MOBA_ERR_INVALID, "the forward kept nothing for a backward");
  if (!s.saved || !s.temp || !s.out || !s.dout || !s.dq || !s.dk || !s.dv || (s.packed && !s.cu_seqlens))
    return fail(MOBA_ERR_INVALID, "null pointer");
  const Shape h = shape_of(s);
  const Saved v = saved_of(s, h);
  const BackTemp t = back_temp_of(s, h);
  const int32_t* cu = s.packed ? s.cu_seqlens : nullptr;
  const int dt = static_cast<int>(s.dtype);
  const int64_t b = s.packed ? 1 : s.batch;
  auto stage = [&](int n, int rc) {
    if (rc) step->failed_stage = n;
    return rc;
  };
  st = stage(6, moba_bwd_delta(s.out, s.dout, v.lse, t.lse_delta, b, s.seq_len, s.h_q, s.head_dim, dt, stream));
  if (st) return st;
  // Segments need scratch; a list that cuts nothing has none.
  const bool list = v.seg && t.scratch;
  st = stage(7, moba_bwd(s.q, s.k, s.v, s.dout, t.lse_delta, v.nnz, v.offsets, v.entries, v.entries + 1,
                         v.entries + 2, v.order, s.dk, s.dv, t.dq_part, cu, s.batch, s.seq_len,
                         s.max_seqlen, s.h_q, s.h_kv, s.head_dim, s.n_blocks, s.block_size, s.slots,
                         h.cap, 3, list ? v.seg : nullptr, v.split, v.counts, list ? h.seg_cap : 0,
                         t.scratch, t.scratch_cap, static_cast<int>(s.causal), dt, dt,
                         static_cast<int>(s.dkv_dtype), stream));
  if (st) return st;
  return stage(8, moba_dq_reduce(t.dq_part, v.ml, 2, s.dq, b, s.seq_len, s.h_q, s.head_dim, s.slots, dt,
                                 dt, stream));
}
