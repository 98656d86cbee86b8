// Block mean-pooling of keys: kbar[r, h, n, :].
//
// Restates src/moba/kernels/pooling.py:26-96 (launcher :103-163) with the
// oracle's rounding: the block sum is formed in float64 (exact for any
// realistic input), rounded to float32 and to the storage dtype, divided by
// the real occupancy in float32 and rounded again.
//
// The whole pass reads K once.
#include <type_traits>

#include "common.h"

namespace moba {

// TS threads per (row, kv head, block, 16-byte piece of features). Each walks
// every TS-th token of the block with one 16-byte load per token (8 or 16
// lanes read each key row whole), a fixed number of tokens in flight, and
// accumulates the features in float64; the TS partial sums then meet by
// shuffles. Bound by the latency of those batches of loads on short
// sequences, by HBM on long ones. bf16, 128-key blocks, four heads of 64:
// 5.6 us at 2K tokens (9.1 with loads kept in order by a loop that tests
// every row, four threads per piece), 9.0 at 64K (17.8), 12.5 at 128K
// (21.2), 47 at 512K (52); float32 10.5 at 2K (19.3) and 23 at 128K (47).
// For 16-bit inputs (8- or 11-bit significands, at most 128 terms) every
// partial and total float64 sum is exact whenever the block's values span
// less than 2^38 in magnitude, so the split changes nothing there; float32
// inputs use TS = 1 (token order, like the oracle). The total is rounded
// once to float32 and to the dtype, then divided by the block's real
// occupancy.
template <typename T, int TS>
__global__ void __launch_bounds__(256)
pool_kernel(const T* __restrict__ k, T* __restrict__ kbar,
            const int32_t* __restrict__ cu, int64_t S, int64_t h_kv,
            int64_t D, int64_t n_blocks, int64_t bs, int64_t n_items) {
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  constexpr int F = 16 / static_cast<int>(sizeof(T));  // features per thread: one 16-byte piece
  const int64_t cpr = D / F;                 // pieces per row
  const int ts = static_cast<int>(gid % TS); // token phase (adjacent lanes)
  const int64_t lin = gid / TS;
  const int64_t item = lin / cpr;            // (r * h_kv + h) * n_blocks + blk
  const bool ok = item < n_items;
  const int64_t it = ok ? item : 0;
  const int64_t d0 = (lin % cpr) * F;
  const int64_t blk = it % n_blocks;
  const int64_t rh = it / n_blocks;
  const int64_t r = rh / h_kv, h = rh % h_kv;
  const SeqSpan sp = seq_span(cu, r, S);
  const int64_t lo = blk * bs;
  const int64_t hi = lo + bs < sp.len ? lo + bs : sp.len;
  double acc[F] = {};
  if (ok && lo < sp.len) {
    // R rows in flight at a time (rows past the end read the last one and
    // add 0), in token order; non-temporal, since K is read once here.
    constexpr int R = sizeof(T) == 2 ? 8 : 16;
    typedef unsigned int u32x4_nt __attribute__((ext_vector_type(4)));
    const T* src = k + ((sp.bos + lo) * h_kv + h) * D + d0;
    const int n = static_cast<int>(hi - lo);
    const int64_t step = h_kv * D;
    for (int t0 = ts; t0 < n; t0 += TS * R) {
      u32x4_nt x[R];
#pragma unroll
      for (int u = 0; u < R; ++u) {
        const T* p = src + min(t0 + TS * u, n - 1) * step;
        x[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_nt*>(p));
      }
#pragma unroll
      for (int u = 0; u < R; ++u) {
        const bool in = t0 + TS * u < n;
#pragma unroll
        for (int i = 0; i < F; ++i) {
          const double v = static_cast<double>(Elem<T>::load(reinterpret_cast<const T*>(&x[u]), i));
          acc[i] += in ? v : 0.0;
        }
      }
    }
  }
#pragma unroll
  for (int off = TS / 2; off > 0; off >>= 1)
#pragma unroll
    for (int i = 0; i < F; ++i) acc[i] += __shfl_xor(acc[i], off);
  if (!ok || ts != 0) return;
  T* dst = kbar + item * D + d0;
  if (lo >= sp.len) {  // a padded block slot of a short sequence: zeros
#pragma unroll
    for (int i = 0; i < F; ++i) Elem<T>::store(dst, i, 0.f);
    return;
  }
  const float count = static_cast<float>(hi - lo);
#pragma unroll
  for (int i = 0; i < F; ++i)
    Elem<T>::store(dst, i, Elem<T>::round(static_cast<float>(acc[i])) / count);
}

// Same semantics for head_dim not a multiple of 8: one workgroup per block,
// threads over the features.
template <typename T>
__global__ void __launch_bounds__(256)
pool_any_kernel(const T* __restrict__ k, T* __restrict__ kbar,
                const int32_t* __restrict__ cu, int64_t S, int64_t h_kv,
                int64_t D, int64_t n_blocks, int64_t bs) {
  const int64_t blk = blockIdx.x;
  const int64_t r = blockIdx.y / h_kv;
  const int64_t h = blockIdx.y % h_kv;
  const SeqSpan sp = seq_span(cu, r, S);
  const int64_t lo = blk * bs;
  if (lo >= sp.len) {
    for (int64_t d = threadIdx.x; d < D; d += blockDim.x)
      Elem<T>::store(kbar, ((r * h_kv + h) * n_blocks + blk) * D + d, 0.f);
    return;
  }
  const int64_t hi = lo + bs < sp.len ? lo + bs : sp.len;
  for (int64_t d = threadIdx.x; d < D; d += blockDim.x) {
    double acc = 0.0;
    for (int64_t t = lo; t < hi; ++t)
      acc += static_cast<double>(Elem<T>::load(k, ((sp.bos + t) * h_kv + h) * D + d));
    float sum = Elem<T>::round(static_cast<float>(acc));
    float mean = sum / static_cast<float>(hi - lo);
    Elem<T>::store(kbar, ((r * h_kv + h) * n_blocks + blk) * D + d, mean);
  }
}

}  // namespace moba

extern "C" int moba_pool(const void* k, void* kbar, const int32_t* cu_seqlens,
                         int64_t batch, int64_t seq_len, int64_t max_seqlen,
                         int64_t h_kv, int64_t head_dim, int64_t n_blocks,
                         int64_t block_size, int dtype, void* stream) {
  using namespace moba;
  Geometry g;
  int st = make_geometry(&g, batch, seq_len, max_seqlen, h_kv, h_kv, head_dim,
                         n_blocks, block_size, 0, cu_seqlens);
  if (st) return st;
  if (!k || !kbar) return fail(MOBA_ERR_INVALID, "null pointer");
  return MOBA_DISPATCH_DTYPE(dtype, T, [&] {
    if (head_dim % 8 == 0) {
      const int64_t n_items = g.rows * h_kv * n_blocks;
      auto go = [&](auto ts) {
        constexpr int TS = decltype(ts)::value;
        hipLaunchKernelGGL((pool_kernel<T, TS>),
                           dim3(static_cast<unsigned>(cdiv(n_items * (head_dim * static_cast<int64_t>(sizeof(T)) / 16) * TS, 256))),
                           dim3(256), 0, as_stream(stream), static_cast<const T*>(k),
                           static_cast<T*>(kbar), cu_seqlens, seq_len, h_kv, head_dim, n_blocks,
                           block_size, n_items);
      };
      // Few blocks: more threads per block, so that a block's rows are all
      // in flight at once on an otherwise idle chip. With enough blocks to
      // fill it, four: a wider split's shuffles cost more than they hide.
      if constexpr (sizeof(T) == 2) {
        const int64_t threads4 = n_items * (head_dim / 8) * 4;
        if (threads4 <= 1 << 15) go(std::integral_constant<int, 16>{});
        else if (threads4 <= 1 << 16) go(std::integral_constant<int, 8>{});
        else go(std::integral_constant<int, 4>{});
      } else {
        go(std::integral_constant<int, 1>{});
      }
    } else {
      dim3 grid(static_cast<unsigned>(n_blocks), static_cast<unsigned>(g.rows * h_kv));
      const int threads = head_dim < 256 ? static_cast<int>(head_dim) : 256;
      hipLaunchKernelGGL(pool_any_kernel<T>, grid, dim3(threads), 0, as_stream(stream),
                         static_cast<const T*>(k), static_cast<T*>(kbar), cu_seqlens,
                         seq_len, h_kv, head_dim, n_blocks, block_size);
    }
    return check_launch("moba_pool");
  });
}
