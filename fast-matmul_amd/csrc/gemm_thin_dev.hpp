// gemm_thin_dev.hpp -- the strip products of dynamic peeling (gemm_thin.hip), as
// device functions: also run beside the W stage of small problems.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "gemm_thin.hpp"
#include "gmem.hpp"

namespace fm_thin {

// Tiles.  Right strip: 128-byte
// runs of rows (16 FP64, 32 FP32), the rest of the work group on K segments.
// Bottom strip: 4 columns per wave, K over the wave's lanes, so each A value
// a lane fetches (a cache line of its own) serves 4 columns.
// A short K does not fill those segments or lanes: as many of them as take K in
// one round of loads work on it, the others take further rows (columns).
// Strips of strassen one level, all segments and lanes on K -> as many as K
// fills: FP64 1000001 x 8 x 5 151 -> 23 us, 300001 x 64 x 65 93 -> 69, 65 x 64 x 300001
// 115 -> 53; whole call FP32 5 x 8 x 1000001 550 -> 386.
constexpr int BOT_COLS = 4, BOT_WAVES = FM_THIN_THREADS / 64;
constexpr int STRIP_LOADS = 8, BOT_LOADS = 4;  // K values in flight per lane
constexpr int BOT_LOG = 6;                     // lanes over K at most, as a power of two
template <typename T>
constexpr int strip_log() {  // K segments at most, as a power of two
  return sizeof(T) == 8 ? 4 : 3;
}
// powers of two: K segments of a right strip, lanes over K of a bottom strip
__host__ __device__ __forceinline__ int strip_segs(int max_log, int K) {
  int l = 0;
  while (l < max_log && (STRIP_LOADS << l) < K) ++l;
  return l;
}
__host__ __device__ __forceinline__ int bot_lanes(int K) {
  int l = 0;
  while (l < BOT_LOG && (BOT_LOADS << l) < K) ++l;
  return l;
}

// p = alpha * sum + beta * p, in the roundings of the K update (see thin_k)
template <typename T>
__device__ __forceinline__ void put(fm_gptr<T> p, T alpha, T beta, T sum) {
  T r = alpha * sum;
  if (beta != T(0)) r = fma(beta, (T)*p, r);
  *p = r;
}

// ALL: every segment on K, the number of them a constant (W and strips of strassen
// 257 x 500 x 55: 4.25 us, 4.42 with it found at run time).
template <typename T, int NT, bool ALL>
__device__ __forceinline__ void thin_n_segs(const FmThinDesc& d, int tm, fm_gptr<const T> A,
                                            fm_gptr<const T> B, fm_gptr<T> C, T* red) {
  constexpr int U = STRIP_LOADS, ML = strip_log<T>();
  const int64_t lda = d.a.ld, ldb = d.b.ld;
  const int K = d.K, tid = threadIdx.x;
  const int ls = ALL ? ML : strip_segs(ML, K), lr = 8 - ls;  // 2^ls segments, 2^lr rows
  const int r = tid & ((1 << lr) - 1), seg = tid >> lr, i0 = tm << lr;
  const fm_gptr<const T> Ai = A + min(i0 + r, d.M - 1);  // rows past M: row M - 1, not stored
  T acc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) acc[j] = T(0);
  for (int k0 = seg; k0 < K; k0 += U << ls) {
    T a[U], b[U][NT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(k0 + (u << ls), K - 1);
      a[u] = Ai[k * lda];
#pragma unroll
      for (int j = 0; j < NT; ++j) b[u][j] = B[k + j * ldb];
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < NT; ++j)
        acc[j] = k0 + (u << ls) < K ? fma(a[u], b[u][j], acc[j]) : acc[j];
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) red[j * FM_THIN_THREADS + tid] = acc[j];
  __syncthreads();
  for (int e = tid; e < NT << lr; e += FM_THIN_THREADS) {
    const int j = e >> lr, rr = e & ((1 << lr) - 1);
    if (i0 + rr >= d.M) continue;
    const T* p = red + j * FM_THIN_THREADS + rr;
    T s = T(0);
#pragma unroll
    for (int q = 0; q < 1 << ls; ++q) s += p[q << lr];
    put<T>(C + i0 + rr + j * d.c.ld, (T)d.alpha, (T)d.beta, s);
  }
}

template <typename T, int NT>
__device__ __forceinline__ void thin_n(const FmThinDesc& d, int tm, fm_gptr<const T> A,
                                       fm_gptr<const T> B, fm_gptr<T> C, T* red) {
  if (d.K > STRIP_LOADS << (strip_log<T>() - 1))
    thin_n_segs<T, NT, true>(d, tm, A, B, C, red);
  else
    thin_n_segs<T, NT, false>(d, tm, A, B, C, red);
}

template <typename T, int MT, bool ALL>
__device__ __forceinline__ void thin_m_lanes(const FmThinDesc& d, int tn, fm_gptr<const T> A,
                                             fm_gptr<const T> B, fm_gptr<T> C) {
  constexpr int U = BOT_LOADS;
  const int K = d.K, lk = ALL ? BOT_LOG : bot_lanes(K);  // 2^lk lanes over K
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int kl = lane & ((1 << lk) - 1), ng = 64 >> lk;  // ng columns side by side
  // column c of this lane: j0 + c * ng
  const int jw = (tn * BOT_WAVES + wave) * (BOT_COLS * ng), j0 = jw + (lane >> lk);
  if (jw >= d.N) return;
  const int64_t lda = d.a.ld, ldb = d.b.ld;
  fm_gptr<const T> Bj[BOT_COLS];
#pragma unroll
  for (int c = 0; c < BOT_COLS; ++c) Bj[c] = B + (int64_t)min(j0 + c * ng, d.N - 1) * ldb;
  T acc[BOT_COLS][MT];
#pragma unroll
  for (int c = 0; c < BOT_COLS; ++c)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[c][i] = T(0);
  for (int k0 = kl; k0 < K; k0 += U << lk) {
    T a[U][MT], b[U][BOT_COLS];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(k0 + (u << lk), K - 1);
#pragma unroll
      for (int c = 0; c < BOT_COLS; ++c) b[u][c] = Bj[c][k];
#pragma unroll
      for (int i = 0; i < MT; ++i) a[u][i] = A[i + k * lda];
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int c = 0; c < BOT_COLS; ++c)
#pragma unroll
        for (int i = 0; i < MT; ++i)
          acc[c][i] = k0 + (u << lk) < K ? fma(a[u][i], b[u][c], acc[c][i]) : acc[c][i];
  }
#pragma unroll
  for (int o = (1 << lk) >> 1; o > 0; o >>= 1)
#pragma unroll
    for (int c = 0; c < BOT_COLS; ++c)
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[c][i] += __shfl_xor(acc[c][i], o);
  // the lanes of a column's group take turns: value v goes to lane v of the group
  if constexpr (ALL) {
    T mine = T(0);
#pragma unroll
    for (int c = 0; c < BOT_COLS; ++c)
#pragma unroll
      for (int i = 0; i < MT; ++i)
        if (lane == c * MT + i) mine = acc[c][i];
    const int c = lane / MT, i = lane - c * MT;
    if (c < BOT_COLS && j0 + c < d.N)
      put<T>(C + i + (int64_t)(j0 + c) * d.c.ld, (T)d.alpha, (T)d.beta, mine);
  } else {
#pragma unroll
    for (int c = 0; c < BOT_COLS; ++c)
#pragma unroll
      for (int i = 0; i < MT; ++i)
        if (kl == ((c * MT + i) & ((1 << lk) - 1)) && j0 + c * ng < d.N)
          put<T>(C + i + (int64_t)(j0 + c * ng) * d.c.ld, (T)d.alpha, (T)d.beta, acc[c][i]);
  }
}

template <typename T, int MT>
__device__ __forceinline__ void thin_m(const FmThinDesc& d, int tn, fm_gptr<const T> A,
                                       fm_gptr<const T> B, fm_gptr<T> C) {
  if (d.K > BOT_LOADS << (BOT_LOG - 1))
    thin_m_lanes<T, MT, true>(d, tn, A, B, C);
  else
    thin_m_lanes<T, MT, false>(d, tn, A, B, C);
}

// f(std::integral_constant) for the thin dimension's value 1 .. MAX
template <int MAX, int V = 1, class F>
__device__ __forceinline__ void thin_dispatch(int v, F&& f) {
  if constexpr (V <= MAX) {
    if (v == V)
      f(std::integral_constant<int, V>());
    else
      thin_dispatch<MAX, V + 1>(v, f);
  }
}

}  // namespace fm_thin
