// gemm_thin.hip -- dynamic-peeling products (linalg/linalg.hpp:201-244): the
// rows, columns and K slices left over by a floor split into blocks.
//
// Each product is bound by memory: it reads the one large operand once (the
// right strip of C reads A, the bottom strip B) or updates C once, at 2 to 14
// flops an element, while its thin dimension (1 to FM_THIN_MAX) fills a
// sixteenth of a matrix instruction.  On 64 x 64 matrix-core tiles a strip
// had one work group per 64 rows walking all of K through LDS, 16 deep at a
// time: a serial chain of loads and barriers, 0.25 us per unit of K whatever
// the machine could stream.  Here K is spread over the lanes of a work group
// (up to 16 or 8 K segments in the right strip, 64 lanes in the bottom strip) with 8
// (4) loads in flight per lane, and the segments' sums meet once at the end,
// in a fixed order that depends on the product alone.
// Measured on MI355X (peeling per multiply, before -> after):
// smirnov333 one level 4799^3 FP64 1190 -> 250 us; grey333_23_152 two levels
// 4009 x 2800 x 2489 FP64 630 -> 234 us; strassen 257 x 500 x 55 FP64
// 41 -> 7 us.
#include <hip/hip_runtime.h>

#include "gemm_thin_dev.hpp"

using namespace fm_thin;

namespace {

// Update of C: one row per lane, 16 columns.
constexpr int UPD_COLS = 16;

// KT: K, or 0 for a K beyond FM_THIN_MAX, read column by column; the sums run
// over K in the same order.
template <typename T, int KT>
__device__ __forceinline__ void thin_k(const FmThinDesc& d, int tm, int tn, fm_gptr<const T> A,
                                       fm_gptr<const T> B, fm_gptr<T> C) {
  const int i = tm * FM_THIN_THREADS + (int)threadIdx.x, j0 = tn * UPD_COLS;
  if (i >= d.M) return;
  const T alpha = (T)d.alpha, beta = (T)d.beta;
  const int64_t ldb = d.b.ld, ldc = d.c.ld;
  T a[KT > 0 ? KT : 1], sum[UPD_COLS];
  if constexpr (KT > 0) {
#pragma unroll
    for (int q = 0; q < KT; ++q) a[q] = A[i + q * d.a.ld];
  } else {
#pragma unroll
    for (int u = 0; u < UPD_COLS; ++u) sum[u] = T(0);
    for (int q = 0; q < d.K; ++q) {
      a[0] = A[i + q * d.a.ld];
#pragma unroll
      for (int u = 0; u < UPD_COLS; ++u)
        sum[u] = fma(a[0], (T)B[q + (int64_t)min(j0 + u, d.N - 1) * ldb], sum[u]);
    }
  }
  C += i;
  // columns past N read column N - 1 again and are not stored: every load of
  // the tile is in flight at once
  T c[UPD_COLS];
  if (beta != T(0)) {
#pragma unroll
    for (int u = 0; u < UPD_COLS; ++u) c[u] = C[(int64_t)min(j0 + u, d.N - 1) * ldc];
  }
#pragma unroll
  for (int u = 0; u < UPD_COLS; ++u) {
    const int j = j0 + u;
    if (j >= d.N) break;
    T s = T(0);
    if constexpr (KT > 0) {
#pragma unroll
      for (int q = 0; q < KT; ++q) s = fma(a[q], (T)B[q + (int64_t)j * ldb], s);
    } else {
      s = sum[u];
    }
    T r = alpha * s;
    if (beta != T(0)) r = fma(beta, c[u], r);
    C[(int64_t)j * ldc] = r;
  }
}

template <typename T>
__global__ void __launch_bounds__(FM_THIN_THREADS) fm_thin_kernel(FmThinArgs args) {
  __shared__ T red[FM_THIN_MAX * FM_THIN_THREADS];
  const int t = blockIdx.x;
  int g;
  if (args.uniform) {
    const int q = t >= args.t0[2] ? 2 : t >= args.t0[1] ? 1 : 0;
    g = args.d0[q] + (t - args.t0[q]) / args.per[q];
  } else {
    int lo = 0, hi = args.ndesc - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (args.descs[mid].tile_begin <= t)
        lo = mid;
      else
        hi = mid - 1;
    }
    g = lo;
  }
  const FmThinDesc d = args.descs[g];
  const int local = t - d.tile_begin;
  const int tn = local / d.tiles_m, tm = local - tn * d.tiles_m;
  const fm_gptr<const T> A = fm_global(reinterpret_cast<const T*>(fm_base(args.bases, d.a.role)) + d.a.off);
  const fm_gptr<const T> B = fm_global(reinterpret_cast<const T*>(fm_base(args.bases, d.b.role)) + d.b.off);
  const fm_gptr<T> C = fm_global(reinterpret_cast<T*>(fm_base(args.bases, d.c.role)) + d.c.off);
  if (d.kind == FM_THIN_K && d.K > FM_THIN_MAX)
    thin_k<T, 0>(d, tm, tn, A, B, C);
  else if (d.kind == FM_THIN_K)
    thin_dispatch<FM_THIN_MAX>(d.K, [&](auto v) { thin_k<T, decltype(v)::value>(d, tm, tn, A, B, C); });
  else if (d.kind == FM_THIN_N)
    thin_dispatch<FM_THIN_MAX>(d.N, [&](auto v) { thin_n<T, decltype(v)::value>(d, tm, A, B, C, red); });
  else
    thin_dispatch<FM_THIN_MAX>(d.M, [&](auto v) { thin_m<T, decltype(v)::value>(d, tn, A, B, C); });
}

}  // namespace

void fm_thin_tile(int dtype_f64, int kind, int K, int* rows, int* cols) {
  *rows = FM_THIN_MAX;
  *cols = FM_THIN_MAX;
  if (kind == FM_THIN_K) {
    *rows = FM_THIN_THREADS;
    *cols = UPD_COLS;
  } else if (kind == FM_THIN_N) {
    *rows = FM_THIN_THREADS >> strip_segs(dtype_f64 ? strip_log<double>() : strip_log<float>(), K);
  } else {
    *cols = BOT_WAVES * BOT_COLS * (64 >> bot_lanes(K));
  }
}

hipError_t fm_thin_launch(int dtype_f64, const FmThinArgs& a, hipStream_t s) {
  if (a.total_tiles <= 0) return hipSuccess;
  if (dtype_f64)
    hipLaunchKernelGGL(fm_thin_kernel<double>, dim3(a.total_tiles), dim3(FM_THIN_THREADS), 0, s, a);
  else
    hipLaunchKernelGGL(fm_thin_kernel<float>, dim3(a.total_tiles), dim3(FM_THIN_THREADS), 0, s, a);
  return hipGetLastError();
}
