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
constexpr int BOT_COLS = 4, BOT_WAVES = FM_THIN_THREADS / 64;
template <typename T>
constexpr int strip_rows() {
  return 128 / (int)sizeof(T);
}

// p = alpha * sum + beta * p, in the roundings of the K update (see thin_k)
template <typename T>
__device__ __forceinline__ void put(fm_gptr<T> p, T alpha, T beta, T sum) {
  T r = alpha * sum;
  if (beta != T(0)) r = fma(beta, (T)*p, r);
  *p = r;
}

template <typename T, int NT>
__device__ __forceinline__ void thin_n(const FmThinDesc& d, int tm, fm_gptr<const T> A,
                                       fm_gptr<const T> B, fm_gptr<T> C, T* red) {
  constexpr int TR = strip_rows<T>(), SEG = FM_THIN_THREADS / TR, U = 8;
  const int r = threadIdx.x % TR, seg = threadIdx.x / TR;
  const int i = tm * TR + r;
  const int64_t lda = d.a.ld, ldb = d.b.ld;
  const int K = d.K;
  const fm_gptr<const T> Ai = A + min(i, d.M - 1);  // rows past M: row M - 1, not stored
  T acc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) acc[j] = T(0);
  for (int k0 = seg; k0 < K; k0 += U * SEG) {
    T a[U], b[U][NT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(k0 + u * SEG, K - 1);
      a[u] = Ai[k * lda];
#pragma unroll
      for (int j = 0; j < NT; ++j) b[u][j] = B[k + j * ldb];
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < NT; ++j)
        acc[j] = k0 + u * SEG < K ? fma(a[u], b[u][j], acc[j]) : acc[j];
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) red[(j * SEG + seg) * TR + r] = acc[j];
  __syncthreads();
  for (int e = threadIdx.x; e < NT * TR; e += FM_THIN_THREADS) {
    const int j = e / TR, rr = e - j * TR;
    if (tm * TR + rr >= d.M) continue;
    T s = T(0);
#pragma unroll
    for (int q = 0; q < SEG; ++q) s += red[(j * SEG + q) * TR + rr];
    put<T>(C + tm * TR + rr + j * d.c.ld, (T)d.alpha, (T)d.beta, s);
  }
}

template <typename T, int MT>
__device__ __forceinline__ void thin_m(const FmThinDesc& d, int tn, fm_gptr<const T> A,
                                       fm_gptr<const T> B, fm_gptr<T> C) {
  constexpr int U = 4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int j0 = (tn * BOT_WAVES + wave) * BOT_COLS;
  if (j0 >= d.N) return;
  const int64_t lda = d.a.ld, ldb = d.b.ld;
  const int K = d.K;
  fm_gptr<const T> Bj[BOT_COLS];
#pragma unroll
  for (int c = 0; c < BOT_COLS; ++c) Bj[c] = B + (int64_t)min(j0 + c, d.N - 1) * ldb;
  T acc[BOT_COLS][MT];
#pragma unroll
  for (int c = 0; c < BOT_COLS; ++c)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[c][i] = T(0);
  for (int k0 = lane; k0 < K; k0 += U * 64) {
    T a[U][MT], b[U][BOT_COLS];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(k0 + u * 64, K - 1);
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
          acc[c][i] = k0 + u * 64 < K ? fma(a[u][i], b[u][c], acc[c][i]) : acc[c][i];
  }
  T mine = T(0);
#pragma unroll
  for (int c = 0; c < BOT_COLS; ++c)
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      T s = acc[c][i];
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
      if (lane == c * MT + i) mine = s;
    }
  const int c = lane / MT, i = lane - c * MT;
  if (c < BOT_COLS && j0 + c < d.N)
    put<T>(C + i + (int64_t)(j0 + c) * d.c.ld, (T)d.alpha, (T)d.beta, mine);
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
