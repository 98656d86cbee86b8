// The gate by float64 matrix products: every (query, past block) score exact,
// no candidate lists, no second look.
//
// Semantics: src/moba/naive.py:64-146, as gate.hip: the exact dot product
// rounded once to float32 and once to the dtype, the top `take` strictly-past
// blocks by (score desc, id asc), ids ascending, the own block last, -1
// padding.
//
// A wave owns 16 consecutive queries of one (row, query head), four lanes
// per query. v_mfma_f64_16x16x4 forms 16 blocks x 16 queries of scores; a
// product of two 24-bit significands is exact in float64 and so is the sum
// for any realistic 16-bit input. The query sits in registers as the B
// operand (D / 4 doubles per lane), the blocks' rows come straight from kbar
// (a wave reads each row once, the workgroup's waves share them in L1) one
// tile ahead, and nothing goes through LDS, so there are no barriers.
// Lane group g = lane / 16 takes features g D/4 .. of both operands (the
// contraction's order is free) and holds the scores of blocks 4v + g,
// v = 0..3, of its query.
//
// Each lane keeps the best T scores of its blocks and the four lists meet in
// two butterfly steps. For 16-bit types a score is one 32-bit word, its
// rounded value as an ordered integer above the complemented block id, so
// the order of the words is (score desc, id asc) and an insertion is one
// v_med3_u32 per entry; float32 scores travel with their ids.
//
// Bound: the float64 matrix rate (71 TFLOP/s measured, 4 or 8 cycles per
// score and SIMD at head_dim 64 / 128), several times the cost per score of
// the approximate kernel of gate.hip, against that kernel's cost per query
// (lists, classification and rescoring of candidates, six launches).
// gate_f64_rows() below draws the line.
#include "common.h"

namespace moba {

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Element e of a 16-byte piece as float64.
template <typename T> __device__ inline double widen(u32x4 w, int e);
template <> __device__ inline double widen<bf16_t>(u32x4 w, int e) {
  const uint32_t u = w[e >> 1];
  return static_cast<double>(u2f(e & 1 ? u & 0xffff0000u : u << 16));
}
template <> __device__ inline double widen<f16_t>(u32x4 w, int e) {
  const uint32_t u = w[e >> 1];
  return static_cast<double>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(e & 1 ? u >> 16 : u)));
}
template <> __device__ inline double widen<float>(u32x4 w, int e) {
  return static_cast<double>(u2f(w[e]));
}

// The score rounded to T, as the bits of T in the upper half of a word, -0
// as +0. `s` is the score rounded to float32, opaque to the compiler, which
// would otherwise round the double to the 16-bit type in one step.
__device__ inline uint32_t rounded_bits(float s, bf16_t) {
  const float r = static_cast<float>(static_cast<__bf16>(s)) + 0.0f;
  return f2u(r);
}
__device__ inline uint32_t rounded_bits(float s, f16_t) {
  const _Float16 r = static_cast<_Float16>(s) + static_cast<_Float16>(0);
  return static_cast<uint32_t>(__builtin_bit_cast(uint16_t, r)) << 16;
}

__device__ inline uint32_t med3(uint32_t a, uint32_t b, uint32_t c) {
  return max(min(a, b), min(max(a, b), c));
}

// The best T entries of one lane, best first.
template <typename T, int TM> struct Top {  // 16-bit types: (score, id) in one word, 0 for none
  uint32_t key[TM];
  __device__ void clear() {
#pragma unroll
    for (int p = 0; p < TM; ++p) key[p] = 0;
  }
  __device__ void insert(double acc, int j, bool past) {
    float s = static_cast<float>(acc);
    asm volatile("" : "+v"(s));
    const uint32_t u = rounded_bits(s, T{});
    // Ordered integers: sign bit flipped, negative values complemented.
    // -inf and NaN (either sign) never rank.
    const uint32_t up = u ^ (static_cast<uint32_t>(static_cast<int32_t>(u) >> 31) | 0x80000000u);
    const bool ok = past && kLowest < up && up < kNan;
    const uint32_t x = ok ? (up & 0xffff0000u) | (0xffffu - static_cast<uint32_t>(j)) : 0u;
#pragma unroll
    for (int p = TM - 1; p > 0; --p) key[p] = med3(key[p - 1], key[p], x);
    key[0] = max(key[0], x);
  }
  // The best of this list and lane ^ off's: the better of entry p and the
  // other's entry TM - 1 - p, an order that log2 TM exchange stages sort.
  __device__ void merge(int off) {
    uint32_t o[TM];
#pragma unroll
    for (int p = 0; p < TM; ++p) o[p] = static_cast<uint32_t>(__shfl_xor(static_cast<int>(key[p]), off));
#pragma unroll
    for (int p = 0; p < TM; ++p) key[p] = max(key[p], o[TM - 1 - p]);
#pragma unroll
    for (int st = TM / 2; st > 0; st >>= 1)
#pragma unroll
      for (int p = 0; p < TM; ++p)
        if ((p & st) == 0) {
          const uint32_t a = key[p], b = key[p + st];
          key[p] = max(a, b);
          key[p + st] = min(a, b);
        }
  }
  __device__ uint32_t id(int p) const { return key[p] ? 0xffffu - (key[p] & 0xffffu) : 0x7fffffffu; }
  // Bounds of the ordered word (its lower half 0 or, below zero, all ones).
  static constexpr uint32_t kInfBits = sizeof(T) == 2 && Elem<T>::kCode == MOBA_BF16 ? 0x7f80u : 0x7c00u;
  static constexpr uint32_t kLowest = (~((kInfBits | 0x8000u) << 16)) | 0xffffu;
  static constexpr uint32_t kNan = ((kInfBits | 0x8000u) + 1u) << 16;
};
template <int TM> struct Top<float, TM> {  // score and id; a lane's ids come in rising order
  float val[TM];
  int idx[TM];
  __device__ void clear() {
#pragma unroll
    for (int p = 0; p < TM; ++p) { val[p] = -INFINITY; idx[p] = 0x7fffffff; }
  }
  __device__ void insert(double acc, int j, bool past) {
    const float s = static_cast<float>(acc);
    const float x = past ? s : -INFINITY;  // -inf and NaN compare greater than nothing
#pragma unroll
    for (int p = TM - 1; p >= 0; --p) {
      const bool here = x > val[p];
      const bool above = p > 0 && x > val[p > 0 ? p - 1 : 0];
      idx[p] = above ? idx[p > 0 ? p - 1 : 0] : (here ? j : idx[p]);
      val[p] = above ? val[p > 0 ? p - 1 : 0] : (here ? x : val[p]);
    }
  }
  __device__ static bool before(float a, int i, float b, int j) { return a > b || (a == b && i < j); }
  __device__ void merge(int off) {
    float ov[TM];
    int oi[TM];
#pragma unroll
    for (int p = 0; p < TM; ++p) { ov[p] = __shfl_xor(val[p], off); oi[p] = __shfl_xor(idx[p], off); }
#pragma unroll
    for (int p = 0; p < TM; ++p) {
      const bool other = before(ov[TM - 1 - p], oi[TM - 1 - p], val[p], idx[p]);
      val[p] = other ? ov[TM - 1 - p] : val[p];
      idx[p] = other ? oi[TM - 1 - p] : idx[p];
    }
#pragma unroll
    for (int st = TM / 2; st > 0; st >>= 1)
#pragma unroll
      for (int p = 0; p < TM; ++p)
        if ((p & st) == 0) {
          const bool sw = before(val[p + st], idx[p + st], val[p], idx[p]);
          const float a = val[p], b = val[p + st];
          const int ia = idx[p], ib = idx[p + st];
          val[p] = sw ? b : a;
          val[p + st] = sw ? a : b;
          idx[p] = sw ? ib : ia;
          idx[p + st] = sw ? ia : ib;
        }
  }
  __device__ uint32_t id(int p) const { return val[p] > -INFINITY ? static_cast<uint32_t>(idx[p]) : 0x7fffffffu; }
};

constexpr int kWaves = 4;

template <typename T, int D, int TM>
__global__ void __launch_bounds__(64 * kWaves)
gate_f64_kernel(const T* __restrict__ q, const T* __restrict__ kbar, int32_t* __restrict__ out,
                const int32_t* __restrict__ cu, int64_t S, int64_t h_q, int64_t h_kv,
                int64_t n_blocks, int bs, int take, int cur, int slots) {
  constexpr int E = D / 4;                                  // features per lane
  constexpr int C = E * static_cast<int>(sizeof(T)) / 16;   // 16-byte pieces of them
  constexpr int PE = 16 / static_cast<int>(sizeof(T));      // elements per piece
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4;
  const int64_t rh = blockIdx.y;
  const int64_t r = rh / h_q, hq = rh % h_q;
  const SeqSpan sp = seq_span(cu, r, S);
  // The last queries, with the most blocks, start first.
  const int64_t t0 = (static_cast<int64_t>(gridDim.x - 1 - blockIdx.x) * kWaves + (threadIdx.x >> 6)) * 16;
  if (t0 >= sp.len) return;  // wave-uniform; no barriers below
  const int64_t t = t0 + (lane & 15);
  const int64_t last = sp.len - 1;
  const int64_t tc = t < sp.len ? t : last;  // lanes past the end compute on a valid row
  const int own = static_cast<int>(tc / bs);
  const int64_t t_end = t0 + 15 < last ? t0 + 15 : last;
  const int horizon = take > 0 ? static_cast<int>(t_end / bs) : 0;  // blocks any query of the wave ranks

  double qv[E];
  {
    const T* qrow = q + ((sp.bos + tc) * h_q + hq) * D + g * E;
    u32x4 w[C];
#pragma unroll
    for (int c = 0; c < C; ++c) w[c] = *reinterpret_cast<const u32x4*>(qrow + c * PE);
#pragma unroll
    for (int e = 0; e < E; ++e) qv[e] = widen<T>(w[e / PE], e % PE);
  }
  const T* kb = kbar + (r * h_kv + hq / (h_q / h_kv)) * n_blocks * D + g * E;
  // Rows past the last block read the last one; their scores are not past.
  auto load = [&](int j0, u32x4 (&w)[C]) {
    const int64_t j = j0 + (lane & 15) < n_blocks ? j0 + (lane & 15) : n_blocks - 1;
#pragma unroll
    for (int c = 0; c < C; ++c) w[c] = *reinterpret_cast<const u32x4*>(kb + j * D + c * PE);
  };
  Top<T, TM> top;
  top.clear();
  u32x4 cw[C];
  if (horizon > 0) load(0, cw);
  for (int j0 = 0; j0 < horizon; j0 += 16) {
    u32x4 nw[C];
    load(j0 + 16, nw);
    f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int e = 0; e < E; ++e)
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(widen<T>(cw[e / PE], e % PE), qv[e], acc, 0, 0, 0);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int j = j0 + 4 * v + g;
      top.insert(acc[v], j, j < own);
    }
#pragma unroll
    for (int c = 0; c < C; ++c) cw[c] = nw[c];
  }
  top.merge(16);
  top.merge(32);
  if (t >= sp.len) return;

  // The first `take` entries' ids, ascending (empty ones last).
  uint32_t id[TM];
  int n_sel = 0;
#pragma unroll
  for (int p = 0; p < TM; ++p) {
    id[p] = p < take ? top.id(p) : 0x7fffffffu;
    n_sel += id[p] != 0x7fffffffu;
  }
#pragma unroll
  for (int k = 2; k <= TM; k <<= 1)
#pragma unroll
    for (int st = k >> 1; st > 0; st >>= 1)
#pragma unroll
      for (int p = 0; p < TM; ++p)
        if ((p & st) == 0) {
          const uint32_t a = id[p], b = id[p + st];
          const bool up = (p & k) == 0;
          id[p] = up ? min(a, b) : max(a, b);
          id[p + st] = up ? max(a, b) : min(a, b);
        }
  // Slot p of the query: lane group p % 4 writes it, four slots of each of
  // the 16 queries per store.
  int32_t* o = out + (cu ? hq * S + sp.bos + t : (r * h_q + hq) * S + t) * slots;
#pragma unroll
  for (int p = 0; p < TM + 4; p += 4) {
    uint32_t x = 0x7fffffffu;
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (p + u < TM) x = g == u ? id[p + u < TM ? p + u : 0] : x;
    const int at = p + g;
    int32_t y = x != 0x7fffffffu ? static_cast<int32_t>(x) : -1;
    if (at == n_sel && cur) y = own;
    if (at < slots) o[at] = y;
  }
  for (int at = TM + 4 + g; at < slots; at += 4) o[at] = -1;
}

template <typename T, int D>
int launch(const void* q, const void* kbar, int32_t* out, const int32_t* cu, const Geometry& g,
           int64_t rows, int take, int cur, hipStream_t st) {
  const dim3 grid(static_cast<unsigned>(cdiv(rows, 16 * kWaves)),
                  static_cast<unsigned>(g.rows * g.h_q));
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(64 * kWaves), 0, st, static_cast<const T*>(q),
                       static_cast<const T*>(kbar), out, cu, g.seq_len, g.h_q, g.h_kv, g.n_blocks,
                       static_cast<int>(g.block_size), take, cur, static_cast<int>(g.slots));
    return check_launch("moba_gate (float64)");
  };
  if (take <= 4) return go(gate_f64_kernel<T, D, 4>);
  if (take <= 8) return go(gate_f64_kernel<T, D, 8>);
  return go(gate_f64_kernel<T, D, 16>);
}

}  // namespace

// Where the line lies (us, this kernel against gate.hip's, bf16 keys i.i.d. /
// with a shared offset). 512K queries, top_k 8: at 64 blocks 106 against 131 /
// 158 (head_dim 64) and 182 against 217 / 254 (128), at 127 blocks 156
// against 130 / 193 and 266 against 214 / 278; with top_k 4 the two are even
// at 64 blocks (102 against 104 / 112, 171 against 168 / 174). Small calls
// gain from one launch instead of six: 64K queries of 32 blocks 16 against
// 36 / 40. Lists of 9 to 16 cost the approximate kernels far more: 128K
// queries of 255 blocks, head_dim 64: 82 against 128 / 215 (top_k 10), 278 /
// 349 (12), 1464 / 1645 (17, which overflow the buffers and are rescored one
// by one); head_dim 128: 135 against 147 / 179, 164 / 233, 419 / 523.
// float32 has no approximate kernel: 64K queries of 127 blocks take 33 us
// (head_dim 64) and 54 us (128), and took 1330 and 2400 in gate_exact_kernel.
//
// With lists of 9 to 16 and 256 blocks or more, the line is drawn per position
// instead of per call: the cost here grows with a query's past blocks, the
// approximate kernels' hardly does. Against those kernels for the whole call,
// over lists of 9 to 16 and both 16-bit types: 128K queries of 256 blocks 128
// .. 294 us and 116 .. 226 split (head_dim 64 and 128), 156K of 313 blocks 146
// .. 347 and 139 .. 287, 512K of 512 blocks 450 .. 1167 and 380 .. 1019. The
// two parts run one after the other, so a split pays only where the first part
// fills the chip by itself: 61K queries of it (512K of 2048 blocks) are even,
// 41K (125K of 400, head_dim 128) lose 1% on some keys, 7K (8K of 256) 15 us.
// Against this kernel for the whole call, top_k 10 .. 17, i.i.d. / offset
// keys, whole and split: head_dim 128, 224 blocks 111 and 122 .. 140 / 151 ..
// 228, 255 blocks 135 and 125 .. 142 / 152 .. 231; head_dim 64, 255 blocks 80
// and 106 .. 114 / 120 .. 179. So below 256 nothing is split. The whole call
// stays ahead for a while above it too (320 blocks: 190 against 156 .. 181 /
// 241 .. 297 and 116 against 131 .. 146 / 195 .. 231; 512 blocks: 405 against
// 254 .. 304 / 382 .. 488 and 254 against 211 .. 245 / 306 .. 427): the line
// at 256 is on the safe side of where the two meet, about 300 blocks on i.i.d.
// keys at head_dim 128 and 450 at 64.
int64_t gate_f64_rows(const void* q, const void* kbar, const Geometry& g, int take, int dtype) {
  if ((g.head_dim != 64 && g.head_dim != 128) || take > 16 || g.rows * g.h_q > 65535) return 0;
  // Rows are read in 16-byte pieces.
  if ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(kbar)) & 15) return 0;
  if (dtype == MOBA_FP32) return g.rows_per_seq;
  if (take <= 8) return g.n_blocks <= (g.head_dim == 64 ? 96 : 64) ? g.rows_per_seq : 0;
  if (g.n_blocks < 256) return g.rows_per_seq;
  const int64_t rows = (g.head_dim == 64 ? 240 : 128) * g.block_size / kGateTile * kGateTile;
  const int64_t part = rows < g.rows_per_seq ? rows : g.rows_per_seq;
  return g.rows * g.h_q * part >= 65536 ? part : 0;
}

int gate_f64(const void* q, const void* kbar, int32_t* out, const int32_t* cu, const Geometry& g,
             int64_t rows, int take, int cur, int dtype, hipStream_t st) {
  return MOBA_DISPATCH_DTYPE(dtype, T, [&] {
    return g.head_dim == 64 ? launch<T, 64>(q, kbar, out, cu, g, rows, take, cur, st)
                            : launch<T, 128>(q, kbar, out, cu, g, rows, take, cur, st);
  });
}

}  // namespace moba
