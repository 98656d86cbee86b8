// float32 kernels of the KV-block-major attention on the matrix cores
// (gfx950), head_dim 64 and 128, blocks of 32, 64 and 128 keys. Other float32
// shapes run the FMA kernels of attn_simple.hip.
//
// Every product and sum is at least as wide as there: scores, weights, the
// forward's P.V and dQ in float32 (v_mfma_f32_16x16x4), dK and dV in float64
// over the whole column (v_mfma_f64_16x16x4 on operands widened exactly).
//
// Bound: the float32 / float64 matrix rates (144 / 71 TFLOP/s measured). The
// layouts keep every other pipe below that: operands come from LDS in whole
// 16-byte pieces or conflict-free words, the contraction's order is chosen so
// that a wave's own accumulators feed its next product straight from
// registers, and the rows of the next group are in flight meanwhile.
//
// Semantics as attn_mfma.hip: src/moba/kernels/moba_fwd.py:230-425 and
// moba_bwd.py:216-394.
#include "attn_common.h"

namespace moba {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));

__device__ inline f32x4 ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }

// ---------------------------------------------------------------------------
// Forward. One workgroup per KV block column (segment); a wave takes 32
// entries at a time, as two query tiles of 16. Lane (n = lane % 16, g = lane
// / 16) works for queries n and 16 + n:
//   S^T[key][q] = K . Q^T   16 x 16 tiles; group g contracts features g D/4
//                           .., register v is key 4g + v of the tile
//   O^T[d][q]   = V^T . P^T step v contracts the keys 4g + v, so P^T feeds
//                           it straight from the registers of S^T
// The backward forms S with the same instruction in the same order, so the
// weights it rebuilds agree with the forward's lse to the last bit of S: the
// rounding of S then cancels in sum dS = 0 (with S summed in another order
// than the backward's, dQ was twice as far from float64 on keys that share
// an offset: 2.1e-6 against 1.1e-6 relative).
// Rows of K and V are padded by 4 floats: 16 consecutive rows meet 16
// distinct 4-bank groups, four rows 4 apart the four quarters of the banks.
//
// [1, 4096, 4, 64], 128-key blocks, top_k 8: 155 us, 12900 in the FMA kernel;
// [1, 8192, 8 query / 2 kv, 64], 64-key blocks: 158 us, 20750.
// ---------------------------------------------------------------------------
// S or dP of one 16 x 16 tile: rows of A and B both 16-byte pieces of the
// features this lane contracts. Two chains: half as many roundings in a row.
template <int N, typename A, typename B>
__device__ inline f32x4 dot_tile(A&& pa, B&& pb) {
  f32x4 c[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const f32x4 x = pa(i), y = pb(i);
#pragma unroll
    for (int u = 0; u < 4; ++u) c[i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[u], y[u], c[i & 1], 0, 0, 0);
  }
  f32x4 r;
#pragma unroll
  for (int v = 0; v < 4; ++v) r[v] = c[0][v] + c[1][v];
  return r;
}

constexpr int fwd_waves(int D, int BS) { return D * BS > 8192 ? 8 : 4; }

template <int D, int BS>
__global__ void __launch_bounds__(64 * fwd_waves(D, BS), D * BS > 8192 ? 1 : 2)
attend_f32_kernel(AttnArgs a) {
  constexpr int RS = D + 4;
  constexpr int KT = BS / 16;
  constexpr int DT = D / 16;
  constexpr int NW = fwd_waves(D, BS);
  constexpr int NT = 64 * NW;
  __shared__ __attribute__((aligned(16))) float Ks[BS * RS];
  __shared__ __attribute__((aligned(16))) float Vs[BS * RS];

  const Column c = resolve_column(a, blockIdx.x, blockIdx.y);
  if (c.n == 0) return;
  const float* K = static_cast<const float*>(a.k);
  const float* V = static_cast<const float*>(a.v);
  const float* Q = static_cast<const float*>(a.q);
  float* acc_out = static_cast<float*>(a.part_acc);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int n = lane & 15;
  const int g = lane >> 4;

  // Lane i % 32 holds the entry of query i % 32 of a group; slot < 0 marks a
  // dead one. Loads are clamped, not skipped.
  auto load_idx = [&](int32_t g0, int32_t& r, int32_t& hd, int32_t& sl) {
    const int32_t e = g0 + (lane & 31);
    const int64_t i = c.lo + (e < c.n ? e : c.n - 1);
    r = a.row_indices[i * a.istride];
    hd = a.head_indices[i * a.istride];
    sl = e < c.n ? a.slot_of_pair[i * a.istride] : -1;
  };
  // B operands of S: features g D/4 + [0, D/4) of queries n and 16 + n. A
  // dead entry reads a live one's row; its results are not stored.
  f32x4 bq[2][D / 16];
  auto fetch = [&](int32_t r, int32_t hd) {
    const int64_t off = q_offset(a, c, r, hd);
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      const float* p = Q + __shfl(off, 16 * qt + n) + g * (D / 4);
#pragma unroll
      for (int i = 0; i < D / 16; ++i) bq[qt][i] = ld4(p + 4 * i);
    }
  };
  int32_t cr, chd, csl, nr, nhd, nsl;
  load_idx(wave * 32, cr, chd, csl);
  for (int i = tid; i < BS * D / 4; i += NT) {
    const int key = i / (D / 4), d4 = (i % (D / 4)) * 4;
    const bool in = c.key0 + key < c.key_end;
    const int64_t off = ((c.tok0 + (in ? key : 0)) * a.h_kv + c.hk) * D + d4;
    const f32x4 kv = ld4(K + off), vv = ld4(V + off);
    *reinterpret_cast<f32x4*>(&Ks[key * RS + d4]) = in ? kv : f32x4{0.f, 0.f, 0.f, 0.f};
    *reinterpret_cast<f32x4*>(&Vs[key * RS + d4]) = in ? vv : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  fetch(cr, chd);
  load_idx(wave * 32 + NW * 32, nr, nhd, nsl);
  __syncthreads();

  for (int32_t g0 = wave * 32; g0 < c.n; g0 += NW * 32) {
    f32x4 s[KT][2];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      // Tiles one after the other (the scheduling barrier): all operands
      // read at once would spill.
      f32x4 ka[D / 16];
#pragma unroll
      for (int i = 0; i < D / 16; ++i) ka[i] = ld4(&Ks[(16 * kt + n) * RS + g * (D / 4) + 4 * i]);
#pragma unroll
      for (int qt = 0; qt < 2; ++qt)
        s[kt][qt] = dot_tile<D / 16>([&](int i) { return ka[i]; }, [&](int i) { return bq[qt][i]; });
      if (kt % 2 == 1 || D == 128) __builtin_amdgcn_sched_barrier(0);
    }
    // Last visible key of each query, and where its results go.
    const bool live = csl >= 0;
    const int key_lim = static_cast<int>(c.key_end - c.key0);
    const int64_t rrel = static_cast<int64_t>(cr) - c.key0;
    const int row_lim = !a.causal ? BS : (rrel < 0 ? -1 : (rrel >= BS ? BS : static_cast<int>(rrel)));
    const int my_lim = live ? min(key_lim - 1, row_lim) : -1;
    const int64_t my_dst = live ? part_row(a, c, cr, chd) * a.slots + csl : -1;
    cr = nr;
    chd = nhd;
    csl = nsl;
    // The next group's rows and the entries of the one after, in flight
    // through the softmax and P.V.
    fetch(cr, chd);
    load_idx(g0 + 2 * NW * 32, nr, nhd, nsl);

    int64_t dst[2];
    float m[2], l[2];
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      const int lim = __shfl(my_lim, 16 * qt + n);
      dst[qt] = __shfl(my_dst, 16 * qt + n);
      float mx = -INFINITY, sum = 0.f;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          s[kt][qt][v] = 16 * kt + 4 * g + v <= lim ? s[kt][qt][v] : -INFINITY;
          mx = fmaxf(mx, s[kt][qt][v]);
        }
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32)) * a.scale_log2;
      const float mz = mx > -INFINITY ? mx : 0.f;  // no visible key: every p is 0
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float p = __builtin_amdgcn_exp2f(fmaf(s[kt][qt][v], a.scale_log2, -mz));
          s[kt][qt][v] = p;
          sum += p;
        }
      sum += __shfl_xor(sum, 16);
      l[qt] = sum + __shfl_xor(sum, 32);
      m[qt] = mx;
    }

    f32x4 o[DT][2];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt][0] = o[dt][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    float va[2][4][DT];
    auto load_v = [&](int kt) {  // keys 16 kt + 4g + [0, 4)
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) va[kt & 1][u][dt] = Vs[(16 * kt + 4 * g + u) * RS + 16 * dt + n];
    };
    load_v(0);
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      if (kt + 1 < KT) load_v(kt + 1);
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int qt = 0; qt < 2; ++qt)
            o[dt][qt] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[kt & 1][u][dt], s[kt][qt][u], o[dt][qt], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int qt = 0; qt < 2; ++qt)
      if (dst[qt] >= 0) {
        if (g == 0) *reinterpret_cast<float2*>(a.part_ml + 2 * dst[qt]) = make_float2(m[qt], l[qt]);
        // o[dt][qt][v] is feature 16 dt + 4g + v.
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          *reinterpret_cast<f32x4*>(acc_out + dst[qt] * D + 16 * dt + 4 * g) = o[dt][qt];
      }
  }
}

// ---------------------------------------------------------------------------
// Backward. One workgroup per KV block column (segment), one wave per 16 of
// its keys, steps of 32 entries. Lane (n = lane % 16, g = lane / 16) holds
// key 16 wave + n. Per step:
//   S[q][key] = Q . K^T, dP = dO . V^T   16 x 16 tiles; group g contracts
//                                        features g D/4 .. (V rows of the
//                                        wave's keys in registers for the
//                                        whole column, K rows in LDS);
//                                        register v is query 4g + v
//   dV[key][d] += P^T . dO, dK += dS^T . Q   float64, step v contracts the
//                                        queries 4g + v: P and dS straight
//                                        from registers, widened
//   dQ^T[d][q] = K^T . dS^T              over all keys, dS rows exchanged in
//                                        LDS; one float32 row per (query,
//                                        slot)
// dK / dV sums never leave float64: a cut column's segments hand float64
// sums to the finishing pass. Rows padded by 4 floats keep every LDS read
// free of bank conflicts (16 rows a 16-byte piece each, or 4 rows 4 apart a
// 64-byte run each).
//
// [1, 8192, 8 query / 2 kv, 64], 64-key blocks, top_k 8: 531 us, 62100 in the
// two FMA kernels (which form S and dP twice).
// ---------------------------------------------------------------------------
template <int D, int BS>
__global__ void __launch_bounds__(4 * BS, D == 64 ? 2 : 1)
bwd_f32_kernel(AttnArgs a) {
  constexpr int NQ = 32;
  constexpr int NW = BS / 16;
  constexpr int NT = 64 * NW;
  constexpr int RS = D + 4;
  constexpr int DS = BS + 4;
  constexpr int DT = D / 16;
  constexpr int TPW = DT * (NQ / 16) / NW;  // dQ tiles per wave
  constexpr int CH = NQ * D / 4 / NT;       // 16-byte pieces per thread and tensor
  __shared__ __attribute__((aligned(16))) float Kl[BS * RS];
  __shared__ __attribute__((aligned(16))) float Qs[NQ * RS];
  __shared__ __attribute__((aligned(16))) float Os[NQ * RS];
  __shared__ __attribute__((aligned(16))) float Ds[NQ * DS];
  __shared__ __attribute__((aligned(16))) float s_lse[NQ], s_delta[NQ];
  __shared__ __attribute__((aligned(16))) int s_lim[NQ];
  __shared__ int64_t s_qoff[NQ];     // next step's rows, -1 for a dead entry
  __shared__ int64_t s_dst[2][NQ];   // dQ rows by step parity, -1 for a dead entry

  const Column c = resolve_column(a, blockIdx.x, blockIdx.y);
  if (c.skip) return;  // past the segment list (uniform)
  const int key_lim = static_cast<int>(c.key_end - c.key0);
  if (key_lim <= 0) return;  // a column past its sequence: its rows lie past the tensor
  const float* Kg = static_cast<const float*>(a.k);
  const float* Vg = static_cast<const float*>(a.v);
  const float* Qg = static_cast<const float*>(a.q);
  const float* Og = static_cast<const float*>(a.dout);
  float* dq_out = static_cast<float*>(a.part_acc);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int n = lane & 15;
  const int g = lane >> 4;
  const int mykey = wave * 16 + n;
  const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};

  // Entry pipeline: thread q < NQ tracks entry q of a step. While step s is
  // computed, the rows and (lse, delta) of step s + 1 and the index entries
  // of step s + 2 are in flight.
  int32_t i_row = 0, i_head = 0, i_slot = 0;
  bool i_live = false;
  auto load_idx = [&](int32_t base) {
    if (tid >= NQ) return;
    const int32_t e = base + tid;
    const int64_t i = c.lo + (e < c.n ? e : c.n - 1);
    i_row = a.row_indices[i * a.istride];
    i_head = a.head_indices[i * a.istride];
    i_slot = a.slot_of_pair[i * a.istride];
    i_live = e < c.n;
  };
  int64_t n_pr = 0, n_dst = -1;
  int n_lim = -1;
  auto derive = [&]() {
    if (tid >= NQ) return;
    const int64_t pr = part_row(a, c, i_row, i_head);
    const int64_t rrel = static_cast<int64_t>(i_row) - c.key0;
    const int row_lim = !a.causal ? BS : (rrel < 0 ? -1 : (rrel >= BS ? BS : static_cast<int>(rrel)));
    n_pr = i_live ? pr : 0;
    n_dst = i_live ? pr * a.slots + i_slot : -1;
    n_lim = i_live ? min(key_lim - 1, row_lim) : -1;
    s_qoff[tid] = i_live ? q_offset(a, c, i_row, i_head) : -1;
  };
  f32x4 pq[CH], po[CH];
  float2 ld = make_float2(0.f, 0.f);
  int64_t c_dst = -1;
  int c_lim = -1;
  auto fetch = [&]() {  // the step that s_qoff / n_* describe
    if (tid < NQ) {
      ld = *reinterpret_cast<const float2*>(a.lse_delta + 2 * n_pr);
      c_dst = n_dst;
      c_lim = n_lim;
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int i = tid + u * NT;
      const int64_t o = s_qoff[i / (D / 4)];
      pq[u] = po[u] = zero4;  // a dead entry adds nothing to dK / dV
      if (o >= 0) {
        pq[u] = ld4(Qg + o + (i % (D / 4)) * 4);
        po[u] = ld4(Og + o + (i % (D / 4)) * 4);
      }
    }
  };
  auto stage = [&](int par) {
    if (tid < NQ) {
      s_lim[tid] = c_lim;
      // A dead entry has read the call's first row: with that row's delta
      // NaN or infinite, 0 * (dP - delta) would reach every key's dK.
      s_lse[tid] = c_dst < 0 ? INFINITY : ld.x;
      s_delta[tid] = c_dst < 0 ? 0.f : ld.y;
      s_dst[par][tid] = c_dst;
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int i = tid + u * NT;
      const int at = (i / (D / 4)) * RS + (i % (D / 4)) * 4;
      *reinterpret_cast<f32x4*>(&Qs[at]) = pq[u];
      *reinterpret_cast<f32x4*>(&Os[at]) = po[u];
    }
  };

  // Column start: the block's keys to LDS, this lane's features of its key's
  // V row to registers; keys past the end are zero.
  if (c.n > 0) load_idx(0);
  for (int i = tid; i < BS * D / 4; i += NT) {
    const int key = i / (D / 4), d4 = (i % (D / 4)) * 4;
    const bool in = key < key_lim;
    const f32x4 kv = ld4(Kg + ((c.tok0 + (in ? key : 0)) * a.h_kv + c.hk) * D + d4);
    *reinterpret_cast<f32x4*>(&Kl[key * RS + d4]) = in ? kv : zero4;
  }
  f32x4 vb[D / 16];
  {
    const bool in = mykey < key_lim;
    const int64_t off = ((c.tok0 + (in ? mykey : 0)) * a.h_kv + c.hk) * D + g * (D / 4);
#pragma unroll
    for (int i = 0; i < D / 16; ++i) {
      const f32x4 vv = ld4(Vg + off + 4 * i);
      vb[i] = in ? vv : zero4;
    }
  }
  f64x4 dk[DT], dv[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) dk[dt] = dv[dt] = f64x4{0.0, 0.0, 0.0, 0.0};
  if (c.n > 0) {
    derive();
    __syncthreads();
    fetch();
    load_idx(NQ);
    stage(0);
    __syncthreads();  // every thread has read step 0's s_qoff
    derive();
  }

  // Two barriers per step: the first makes the step's staging visible and
  // orders the previous step's reads of dS before this step's writes, the
  // second makes dS visible and frees Qs / Os.
  int par = 0;
  for (int32_t base = 0; base < c.n; base += NQ, par ^= 1) {
    __syncthreads();
    const bool next = base + NQ < c.n;  // uniform
    if (next) {
      fetch();
      load_idx(base + 2 * NQ);
    }
#pragma unroll
    for (int qt = 0; qt < NQ / 16; ++qt) {
      const int at = (16 * qt + n) * RS + g * (D / 4);
      const f32x4 s = dot_tile<D / 16>([&](int i) { return ld4(&Qs[at + 4 * i]); },
                                       [&](int i) { return ld4(&Kl[mykey * RS + g * (D / 4) + 4 * i]); });
      const f32x4 dp = dot_tile<D / 16>([&](int i) { return ld4(&Os[at + 4 * i]); },
                                        [&](int i) { return vb[i]; });
      if (D == 128) __builtin_amdgcn_sched_barrier(0);
      const int q0 = 16 * qt + 4 * g;  // this lane's queries q0 + v
      const int4 lim4 = *reinterpret_cast<const int4*>(&s_lim[q0]);
      const f32x4 lse = ld4(&s_lse[q0]), dl = ld4(&s_delta[q0]);
      const int lim[4] = {lim4.x, lim4.y, lim4.z, lim4.w};
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float p = mykey <= lim[v]
                            ? __builtin_amdgcn_exp2f(fmaf(s[v], a.scale_log2, -lse[v])) : 0.f;
        const float ds = p * (dp[v] - dl[v]);
        Ds[(q0 + v) * DS + mykey] = ds;
        const double pd = p, dsd = ds;
        const float* orow = &Os[(q0 + v) * RS + n];
        const float* qrow = &Qs[(q0 + v) * RS + n];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          dv[dt] = __builtin_amdgcn_mfma_f64_16x16x4f64(pd, static_cast<double>(orow[16 * dt]), dv[dt], 0, 0, 0);
          dk[dt] = __builtin_amdgcn_mfma_f64_16x16x4f64(dsd, static_cast<double>(qrow[16 * dt]), dk[dt], 0, 0, 0);
          if (dt % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // few widened operands at a time
        }
      }
    }
    __syncthreads();  // dS of every wave visible; Qs / Os free
    const int64_t* dst = s_dst[par];
    if (next) {
      stage(par ^ 1);
      derive();
    }
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      const int tt = wave + t * NW;
      const int dt = tt % DT, qt = tt / DT;
      f32x4 acc2[2] = {zero4, zero4};
#pragma unroll
      for (int i = 0; i < BS / 16; ++i) {
        const f32x4 ds4 = ld4(&Ds[(16 * qt + n) * DS + 16 * i + 4 * g]);
#pragma unroll
        for (int u = 0; u < 4; ++u)
          acc2[i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(
              Kl[(16 * i + 4 * g + u) * RS + 16 * dt + n], ds4[u], acc2[i & 1], 0, 0, 0);
        if (D == 128 && i % 2 == 1) __builtin_amdgcn_sched_barrier(0);
      }
      // acc2[.][v]: feature 16 dt + 4g + v of query 16 qt + n.
      const int64_t row = dst[16 * qt + n];
      f32x4 acc;
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[v] = (acc2[0][v] + acc2[1][v]) * a.scale;
      if (row >= 0) *reinterpret_cast<f32x4*>(dq_out + row * D + 16 * dt + 4 * g) = acc;
    }
  }

  // dk[dt][v], dv[dt][v]: key 16 wave + 4v + g, feature 16 dt + n.
  const double scale = a.scale;
  if (c.nseg > 1) {
    double* sk = reinterpret_cast<double*>(a.seg_scratch) +
                 (static_cast<int64_t>(blockIdx.y) * (a.scratch_cap / 2) + c.scratch) * 2 * BS * D;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int at = (wave * 16 + 4 * v + g) * D + 16 * dt + n;
        sk[at] = dk[dt][v] * scale;
        sk[BS * D + at] = dv[dt][v];
      }
    return;
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int key = wave * 16 + 4 * v + g;
    if (key >= key_lim) continue;
    const int64_t off = ((c.tok0 + key) * a.h_kv + c.hk) * D + n;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      static_cast<float*>(a.dk)[off + 16 * dt] = static_cast<float>(dk[dt][v] * scale);
      static_cast<float*>(a.dv)[off + 16 * dt] = static_cast<float>(dv[dt][v]);
    }
  }
}

// dK / dV of the cut columns: the segments' float64 sums added in segment
// order and rounded once. Eight workgroups per cut column.
__global__ void __launch_bounds__(256) seg_finish_f32_kernel(AttnArgs a) {
  const int64_t rh = blockIdx.y;
  if (static_cast<int64_t>(blockIdx.x) >= a.seg_counts[2 * rh + 1]) return;
  const Column c = resolve_column(a, a.seg_split[rh * (a.seg_cap - a.n_blocks) + blockIdx.x], rh);
  const int64_t bsd = a.bs * a.D;
  const double* base = reinterpret_cast<const double*>(a.seg_scratch) +
                       (rh * (a.scratch_cap / 2) + c.scratch) * 2 * bsd;
  const int64_t n = (c.key_end - c.key0) * a.D;
  for (int64_t i = blockIdx.z * blockDim.x + threadIdx.x; i < n; i += gridDim.z * blockDim.x) {
    double sk = 0.0, sv = 0.0;
    for (int j = 0; j < c.nseg; ++j) {
      sk += base[j * 2 * bsd + i];
      sv += base[j * 2 * bsd + bsd + i];
    }
    const int64_t off = ((c.tok0 + i / a.D) * a.h_kv + c.hk) * a.D + i % a.D;
    static_cast<float*>(a.dk)[off] = static_cast<float>(sk);
    static_cast<float*>(a.dv)[off] = static_cast<float>(sv);
  }
}

// Rows are read and written in 16-byte pieces, (m, l) pairs in 8-byte ones.
bool aligned(const AttnArgs& a) {
  const uintptr_t wide = reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.k) |
                         reinterpret_cast<uintptr_t>(a.v) | reinterpret_cast<uintptr_t>(a.dout) |
                         reinterpret_cast<uintptr_t>(a.part_acc);
  const uintptr_t pair = reinterpret_cast<uintptr_t>(a.part_ml) | reinterpret_cast<uintptr_t>(a.lse_delta);
  return (wide & 15) == 0 && (pair & 7) == 0;
}

template <int D, int BS>
int launch_attend(const AttnArgs& a, int64_t n_cols, hipStream_t st) {
  const dim3 grid(column_programs(a, n_cols), static_cast<unsigned>(n_cols));
  hipLaunchKernelGGL((attend_f32_kernel<D, BS>), grid, dim3(64 * fwd_waves(D, BS)), 0, st, a);
  return check_launch("moba_attend (float32)");
}

template <int D, int BS>
int launch_bwd(const AttnArgs& args, int64_t n_cols, hipStream_t st) {
  AttnArgs a = args;
  // A cut column's segments need float64 scratch: twice the float32 slots
  // the segment list asks for, on an 8-byte boundary. Without it, whole
  // columns.
  if (a.seg && a.seg_cap > a.n_blocks &&
      (a.scratch_cap < 4 * (a.seg_cap - a.n_blocks) || (reinterpret_cast<uintptr_t>(a.seg_scratch) & 7)))
    a.seg = nullptr;
  const dim3 grid(column_programs(a, n_cols), static_cast<unsigned>(n_cols));
  hipLaunchKernelGGL((bwd_f32_kernel<D, BS>), grid, dim3(4 * BS), 0, st, a);
  const int rc = check_launch("moba_bwd (float32)");
  if (rc || !a.seg || a.seg_cap == a.n_blocks) return rc;
  hipLaunchKernelGGL(seg_finish_f32_kernel,
                     dim3(static_cast<unsigned>(a.seg_cap - a.n_blocks), static_cast<unsigned>(n_cols), 8),
                     dim3(256), 0, st, a);
  return check_launch("moba_bwd (float32, cut columns)");
}

}  // namespace

int attend_f32(const AttnArgs& a, int dtype, int acc_dtype, int64_t n_cols, hipStream_t st) {
  if (dtype != MOBA_FP32 || acc_dtype != MOBA_FP32 || !aligned(a)) return MOBA_ERR_UNSUPPORTED;
  if (a.D == 64) {
    if (a.bs == 128) return launch_attend<64, 128>(a, n_cols, st);
    if (a.bs == 64) return launch_attend<64, 64>(a, n_cols, st);
    if (a.bs == 32) return launch_attend<64, 32>(a, n_cols, st);
  } else if (a.D == 128) {
    if (a.bs == 128) return launch_attend<128, 128>(a, n_cols, st);
    if (a.bs == 64) return launch_attend<128, 64>(a, n_cols, st);
    if (a.bs == 32) return launch_attend<128, 32>(a, n_cols, st);
  }
  return MOBA_ERR_UNSUPPORTED;
}

int bwd_f32(const AttnArgs& a, int dtype, int acc_dtype, int64_t n_cols, hipStream_t st) {
  if (dtype != MOBA_FP32 || acc_dtype != MOBA_FP32 || !aligned(a)) return MOBA_ERR_UNSUPPORTED;
  if (a.D == 64) {
    if (a.bs == 128) return launch_bwd<64, 128>(a, n_cols, st);
    if (a.bs == 64) return launch_bwd<64, 64>(a, n_cols, st);
    if (a.bs == 32) return launch_bwd<64, 32>(a, n_cols, st);
  } else if (a.D == 128) {
    if (a.bs == 128) return launch_bwd<128, 128>(a, n_cols, st);
    if (a.bs == 64) return launch_bwd<128, 64>(a, n_cols, st);
    if (a.bs == 32) return launch_bwd<128, 32>(a, n_cols, st);
  }
  return MOBA_ERR_UNSUPPORTED;
}

}  // namespace moba
