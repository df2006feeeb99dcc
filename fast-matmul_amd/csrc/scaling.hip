// scaling.hip -- diagonal scaling around the fast multiply
// (scaling/scaling.hpp:105-196 of the reference).
//
// Outer scaling divides the rows of A by their largest magnitude x_i and the
// columns of B by theirs y_j (the factors accumulate in r and s); inner
// scaling multiplies column k of A by 1/z_k and row k of B by z_k with
// z_k = sqrt(max|A[:,k]| / max|B[k,:]|).  After the multiply,
// PostProcessScaling multiplies row i of the product by r_i and column j by
// s_j.  Each pass is the reference's: the factor vector is formed first
// (1/x rounded, sqrt rounded), then every element is multiplied by it, one
// rounding per pass, in the reference's pass order.  A row or column that is
// all zeros keeps factor 1 (the reference would divide by zero).
//
// Every pass is bound by memory, so a scaling step does not store its
// intermediate matrices: the second pass's maxima are taken over the
// products with the first pass's factors formed on the fly, and one last
// pass multiplies by both factors, in order, and writes the copies.  A and B
// share each launch.  A step reads each matrix three times and writes it
// once, in 6 launches (it was 5 reads, 3 writes and 17 launches, and the row
// maxima ran on 256 work groups): strassen one level 4096^3 FP32, all of
// the scaling 490 -> 136 us, the call 1435 -> 1109 us.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "gmem.hpp"
#include "scaling.hpp"

namespace {

template <typename T>
struct Bits;
template <>
struct Bits<double> {
  typedef unsigned long long U;
  __device__ static U of(double v) { return (U)__double_as_longlong(v); }
  __device__ static double val(U u) { return __longlong_as_double((long long)u); }
};
template <>
struct Bits<float> {
  typedef unsigned int U;
  __device__ static U of(float v) { return __float_as_uint(v); }
  __device__ static float val(U u) { return __uint_as_float(u); }
};

// separately rounded products and sums (no contraction into FMA)
__device__ __forceinline__ double mul_rn(double a, double b) { return __dmul_rn(a, b); }
__device__ __forceinline__ float mul_rn(float a, float b) { return __fmul_rn(a, b); }
__device__ __forceinline__ double add_rn(double a, double b) { return __dadd_rn(a, b); }
__device__ __forceinline__ float add_rn(float a, float b) { return __fadd_rn(a, b); }

// A work group's lanes take 16 bytes of rows each.  Where a matrix has fewer rows
// than they cover, 2^lr of them (of a wave's, in the column maxima) go along the
// rows and the others take further columns.  With all lanes along the rows a B of
// 7 rows kept 2 of 256 lanes busy, and every 32 columns ended in their own atomics
// on the same 7 maxima: whole call, strassen one level, 5 x 7 x 1000000 FP32 2300 ->
// 471 us, FP64 1800 -> 689; 64 x 64 x 100000 354 -> 124, 303 -> 194.
constexpr int SC_THREADS = 256;
constexpr int SC_COLS = 32;        // columns a lane takes in a row-maxima tile
constexpr int SC_SHORT_COLS = 16;  // the same where lanes share the columns
constexpr int SC_WCOLS = 8;        // columns a lane takes in a write tile
constexpr int SC_SEGMENT = 8192;   // rows of a column-maxima segment (one wave)
constexpr int ROW_LOG = 8, COL_LOG = 6;  // lr where all lanes go along the rows
template <typename T>
constexpr int sc_vl() {
  return 16 / (int)sizeof(T);
}

// VL consecutive rows of a column at the alignment of an element (rows past
// the end read as zero)
template <typename T>
struct Rows {
  static constexpr int VL = 16 / (int)sizeof(T);
  typedef T vec_t __attribute__((ext_vector_type(VL))) __attribute__((aligned(sizeof(T))));
  T v[VL];
  __device__ __forceinline__ void load(const T* p, int n) {
    if (n >= VL) {
      const vec_t x = *(fm_gptr<const vec_t>)p;
#pragma unroll
      for (int e = 0; e < VL; ++e) v[e] = x[e];
    } else {
#pragma unroll
      for (int e = 0; e < VL; ++e) v[e] = e < n ? p[e] : T(0);
    }
  }
  __device__ __forceinline__ void store(T* p, int n) const {
    if (n >= VL) {
      vec_t x;
#pragma unroll
      for (int e = 0; e < VL; ++e) x[e] = v[e];
      *(fm_gptr<vec_t>)p = x;
    } else {
#pragma unroll
      for (int e = 0; e < VL; ++e)
        if (e < n) p[e] = v[e];
    }
  }
};

// One matrix of a maxima launch: `out` gets the largest magnitude of every
// row (rowwise) or column of X, each element first multiplied by the factor
// of its column (rowwise) or row where `pre` is given.  Partial maxima meet
// in an integer atomicMax on the bit pattern (non-negative floats order like
// their bits); `out` starts as zeros.
template <typename T>
struct MaxArgs {
  const T* X;
  int64_t ld;
  int rows, cols, rowwise;
  const T* pre;
  typename Bits<T>::U* out;
  int tiles_r, tiles;  // tiles along the rows, all tiles
  int lr;              // lanes along the rows, as a power of two
};

// All lanes along the rows: the layout a constant, uniform trip counts (1000^3
// FP32, whole call: 66 us, 83 with the layout read at run time).
template <typename T>
__device__ __forceinline__ void row_max_tile(const MaxArgs<T>& a, int t) {
  constexpr int VL = Rows<T>::VL;
  const int tr = t % a.tiles_r, tc = t / a.tiles_r;
  const int64_t i0 = ((int64_t)tr * SC_THREADS + (int)threadIdx.x) * VL;
  if (i0 >= a.rows) return;
  const int j0 = tc * SC_COLS, j1 = min(a.cols, j0 + SC_COLS), n = (int)(a.rows - i0);
  T mx[VL];
#pragma unroll
  for (int e = 0; e < VL; ++e) mx[e] = T(0);
#pragma unroll 8
  for (int j = j0; j < j1; ++j) {
    Rows<T> x;
    x.load(a.X + i0 + (int64_t)j * a.ld, n);
    const T f = a.pre ? a.pre[j] : T(1);
#pragma unroll
    for (int e = 0; e < VL; ++e) mx[e] = fmax(mx[e], fabs(a.pre ? mul_rn(x.v[e], f) : x.v[e]));
  }
#pragma unroll
  for (int e = 0; e < VL; ++e)
    if (e < n) atomicMax(a.out + i0 + e, Bits<T>::of(mx[e]));
}

template <typename T>
__device__ __forceinline__ void col_max_tile(const MaxArgs<T>& a, int t) {
  constexpr int VL = Rows<T>::VL;
  const int tr = t % a.tiles_r, tc = t / a.tiles_r;
  // one wave per column and segment of rows
  const int j = tc * (SC_THREADS / 64) + ((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (j >= a.cols) return;
  const int r0 = tr * SC_SEGMENT, len = min(a.rows - r0, SC_SEGMENT);
  const T* c = a.X + (int64_t)j * a.ld;
  T mx = T(0);
#pragma unroll 4
  for (int i = lane * VL; i < len; i += 64 * VL) {
    Rows<T> x;
    x.load(c + r0 + i, len - i);
    if (a.pre) {
      Rows<T> f;
      f.load(a.pre + r0 + i, len - i);
#pragma unroll
      for (int e = 0; e < VL; ++e) mx = fmax(mx, fabs(mul_rn(x.v[e], f.v[e])));
    } else {
#pragma unroll
      for (int e = 0; e < VL; ++e) mx = fmax(mx, fabs(x.v[e]));
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o));
  if (lane == 0) atomicMax(a.out + j, Bits<T>::of(mx));
}

// Short matrices.  Rows: lane r of 2^lr along the rows, g of ng column groups,
// whose maxima meet in the first group's lanes.
template <typename T>
__device__ __forceinline__ void row_max_short(const MaxArgs<T>& a, int t, T* red) {
  constexpr int VL = Rows<T>::VL;
  const int tid = threadIdx.x, lr = a.lr, ng = SC_THREADS >> lr, r = tid & ((1 << lr) - 1), g = tid >> lr;
  const int i0 = r * VL, n = a.rows - i0;  // one tile holds all rows
  const int64_t j0 = (int64_t)t * SC_SHORT_COLS * ng + g;
  T mx[VL];
#pragma unroll
  for (int e = 0; e < VL; ++e) mx[e] = T(0);
  if (n > 0) {
#pragma unroll 8
    for (int q = 0; q < SC_SHORT_COLS; ++q) {
      const int64_t j = j0 + q * ng;
      if (j >= a.cols) break;
      Rows<T> x;
      x.load(a.X + i0 + j * a.ld, n);
      const T f = a.pre ? a.pre[j] : T(1);
#pragma unroll
      for (int e = 0; e < VL; ++e) mx[e] = fmax(mx[e], fabs(a.pre ? mul_rn(x.v[e], f) : x.v[e]));
    }
  }
#pragma unroll
  for (int e = 0; e < VL; ++e) red[e * SC_THREADS + tid] = mx[e];
  __syncthreads();
  if (g > 0) return;
  for (int q = 1; q < ng; ++q)
#pragma unroll
    for (int e = 0; e < VL; ++e) mx[e] = fmax(mx[e], red[e * SC_THREADS + (q << lr) + r]);
#pragma unroll
  for (int e = 0; e < VL; ++e)
    if (e < n) atomicMax(a.out + i0 + e, Bits<T>::of(mx[e]));
}

// Columns: 2^lr lanes of a wave per column, one vector each.
template <typename T>
__device__ __forceinline__ void col_max_short(const MaxArgs<T>& a, int t) {
  constexpr int VL = Rows<T>::VL;
  const int tid = threadIdx.x, lr = a.lr, i = (tid & ((1 << lr) - 1)) * VL;
  const int64_t j = (int64_t)t * (SC_THREADS >> lr) + (tid >> lr);
  if (j >= a.cols) return;
  T mx = T(0);
  if (i < a.rows) {
    Rows<T> x, f;
    x.load(a.X + i + j * a.ld, a.rows - i);
    if (a.pre) f.load(a.pre + i, a.rows - i);
#pragma unroll
    for (int e = 0; e < VL; ++e) mx = fmax(mx, fabs(a.pre ? mul_rn(x.v[e], f.v[e]) : x.v[e]));
  }
  for (int o = (1 << lr) >> 1; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o));
  if (i == 0) atomicMax(a.out + j, Bits<T>::of(mx));
}

template <typename T, bool SHORT>
__device__ __forceinline__ void max_tile(const MaxArgs<T>& a, int t, T* red) {
  if (a.rowwise) {
    if (!SHORT || a.lr == ROW_LOG)
      row_max_tile(a, t);
    else
      row_max_short(a, t, red);
  } else {
    if (!SHORT || a.lr == COL_LOG)
      col_max_tile(a, t);
    else
      col_max_short(a, t);
  }
}

// A and B in one launch.  SHORT: A or B is short (1000^3 FP32, whole call: 65.8 us
// without, 67.2 with those paths beside the others in one kernel).
template <typename T, bool SHORT>
__global__ void __launch_bounds__(SC_THREADS) fm_max_kernel(MaxArgs<T> a, MaxArgs<T> b) {
  __shared__ T red[SHORT ? SC_THREADS * Rows<T>::VL : 1];
  const int t = blockIdx.x;
  if (t < a.tiles)
    max_tile<T, SHORT>(a, t, red);
  else
    max_tile<T, SHORT>(b, t - a.tiles, red);
}

// Factor arithmetic follows the reference's types: the maxima are doubles
// (MaxAbsRow / MaxAbsCol return double), 1/x and sqrt(a/b) are evaluated in
// double and stored as Scalar (InverseVector, InnerScaling), and the running
// products r, s are Scalar (UpdateVals).  The factors replace the maxima they
// come from.

// outer-scaling factors: f[i] = 1 / x[i] (1 for x = 0), r[i] *= x[i] (x = 0: unchanged)
template <typename T>
__device__ __forceinline__ void outer_factor(T* f, T* r, int i) {
  const T x = f[i];
  if (x > T(0)) {
    f[i] = (T)(1.0 / (double)x);
    r[i] = mul_rn(r[i], x);
  } else {
    f[i] = T(1);
  }
}
template <typename T>
__global__ void fm_outer_factors(T* f, T* r, int m, T* f2, T* s, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < m) outer_factor(f, r, i);
  if (i < n) outer_factor(f2, s, i);
}

// inner-scaling factors: z = sqrt(ca / rb) (1 where either is 0), zi = 1 / z;
// ca becomes zi (the factor of A's columns), rb becomes z
template <typename T>
__global__ void fm_inner_factors(T* ca, T* rb, int n) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k >= n) return;
  const double a = (double)ca[k], b = (double)rb[k];
  T v = T(1);
  if (a > 0.0 && b > 0.0) v = (T)sqrt(a / b);
  rb[k] = v;
  ca[k] = (T)(1.0 / (double)v);
}

// zero the maxima of a step; the first step also sets r and s to ones
template <typename T>
__global__ void fm_scale_init(T* f, T* r, int m, T* f2, T* s, int n, T* u1, T* u2, int k, int first) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < m) f[i] = T(0);
  if (i < n) f2[i] = T(0);
  if (i < k) u1[i] = u2[i] = T(0);
  if (first && i < m) r[i] = T(1);
  if (first && i < n) s[i] = T(1);
}

// One matrix of the write launch: Y[i, j] = X[i, j] times its row's factor rf
// and its column's factor cf (where given; rf first when row_first), one
// rounding per factor; Y may alias X.
template <typename T>
struct WriteArgs {
  const T* X;
  int64_t ldx;
  T* Y;
  int64_t ldy;
  int rows, cols;
  const T *rf, *cf;
  int row_first;
  int tiles_r, tiles, lr;  // as in MaxArgs
};

// This lane's place in tile t of a write launch: its first row, its first column
// and the distance to the next.
template <bool ALL>
using ColIdx = typename std::conditional<ALL, int, int64_t>::type;  // (tall: few columns fit)
template <typename T, bool ALL>
__device__ __forceinline__ void write_place(int t, int tiles_r, int some, int64_t* i0, ColIdx<ALL>* j0, int* step) {
  const int tr = t % tiles_r, tc = t / tiles_r, tid = threadIdx.x, lr = ALL ? ROW_LOG : some;
  *step = ALL ? 1 : SC_THREADS >> lr;
  *i0 = (((int64_t)tr << lr) + (ALL ? tid : tid & ((1 << lr) - 1))) * Rows<T>::VL;
  *j0 = ALL ? tc * SC_WCOLS : (ColIdx<ALL>)tc * SC_WCOLS * *step + (tid >> lr);
}

template <typename T, bool ALL>
__device__ __forceinline__ void write_tile_lanes(const WriteArgs<T>& a, int t) {
  constexpr int VL = Rows<T>::VL;
  int64_t i0;
  ColIdx<ALL> j0;
  int step;
  write_place<T, ALL>(t, a.tiles_r, a.lr, &i0, &j0, &step);
  if (i0 >= a.rows) return;
  const int n = (int)(a.rows - i0);
  Rows<T> rf;
  if (a.rf) rf.load(a.rf + i0, n);
  Rows<T> x[SC_WCOLS];
#pragma unroll
  for (int u = 0; u < SC_WCOLS; ++u)  // columns past the end read the last one, not stored
    x[u].load(a.X + i0 + (int64_t)min(j0 + u * step, (ColIdx<ALL>)(a.cols - 1)) * a.ldx, n);
#pragma unroll
  for (int u = 0; u < SC_WCOLS; ++u) {
    const ColIdx<ALL> j = j0 + u * step;
    if (j >= a.cols) break;
    const T c = a.cf ? a.cf[j] : T(1);
#pragma unroll
    for (int e = 0; e < VL; ++e) {
      T v = x[u].v[e];
      if (a.row_first && a.rf) v = mul_rn(v, rf.v[e]);
      if (a.cf) v = mul_rn(v, c);
      if (!a.row_first && a.rf) v = mul_rn(v, rf.v[e]);
      x[u].v[e] = v;
    }
    x[u].store(a.Y + i0 + (int64_t)j * a.ldy, n);
  }
}

template <typename T, bool SHORT>
__device__ __forceinline__ void write_tile(const WriteArgs<T>& a, int t) {
  if (!SHORT || a.lr == ROW_LOG)
    write_tile_lanes<T, true>(a, t);
  else
    write_tile_lanes<T, false>(a, t);
}

template <typename T, bool SHORT>
__global__ void __launch_bounds__(SC_THREADS) fm_write_kernel(WriteArgs<T> a, WriteArgs<T> b) {
  const int t = blockIdx.x;
  if (t < a.tiles)
    write_tile<T, SHORT>(a, t);
  else
    write_tile<T, SHORT>(b, t - a.tiles);
}

// C[i, j] = alpha * ((P[i, j] * r[i]) * s[j]) + beta * C[i, j]; P may be C
template <typename T, bool ALL>
__global__ void __launch_bounds__(SC_THREADS) fm_post_kernel(const T* P, int64_t ldp, T* C, int64_t ldc,
                                                             int rows, int cols, const T* r, const T* s,
                                                             T alpha, T beta, int tiles_r, int lr) {
  constexpr int VL = Rows<T>::VL;
  int64_t i0;
  ColIdx<ALL> j0;
  int step;
  write_place<T, ALL>(blockIdx.x, tiles_r, lr, &i0, &j0, &step);
  if (i0 >= rows) return;
  const int n = (int)(rows - i0);
  Rows<T> rf, x[SC_WCOLS];
  rf.load(r + i0, n);
#pragma unroll
  for (int u = 0; u < SC_WCOLS; ++u) x[u].load(P + i0 + (int64_t)min(j0 + u * step, (ColIdx<ALL>)(cols - 1)) * ldp, n);
#pragma unroll
  for (int u = 0; u < SC_WCOLS; ++u) {
    const ColIdx<ALL> j = j0 + u * step;
    if (j >= cols) break;
    const T c = s[j];
    T* out = C + i0 + (int64_t)j * ldc;
    Rows<T> old;
    if (beta != T(0)) old.load(out, n);
#pragma unroll
    for (int e = 0; e < VL; ++e) {
      T v = mul_rn(mul_rn(x[u].v[e], rf.v[e]), c);
      if (alpha != T(1)) v = mul_rn(alpha, v);
      if (beta != T(0)) v = add_rn(v, mul_rn(beta, old.v[e]));
      x[u].v[e] = v;
    }
    x[u].store(out, n);
  }
}

inline unsigned blocks_for(int n) { return (unsigned)((n + 255) / 256); }

// lanes along `rows` rows, as a power of two up to max_log
template <typename T>
int row_lanes(int rows, int max_log) {
  int l = 0;
  while (l < max_log && ((int64_t)sc_vl<T>() << l) < rows) ++l;
  return l;
}

template <typename T>
MaxArgs<T> max_args(const T* X, int64_t ld, int rows, int cols, int rowwise, const T* pre, T* out) {
  MaxArgs<T> a{X, ld, rows, cols, rowwise, pre, reinterpret_cast<typename Bits<T>::U*>(out), 0, 0, 0};
  a.lr = row_lanes<T>(rows, rowwise ? ROW_LOG : COL_LOG);
  const int groups = SC_THREADS >> a.lr;
  const int64_t tile_r = rowwise ? sc_vl<T>() << a.lr : SC_SEGMENT;
  const int64_t tile_c = rowwise ? (groups > 1 ? SC_SHORT_COLS : SC_COLS) * groups : groups;
  a.tiles_r = (int)((rows + tile_r - 1) / tile_r);
  a.tiles = a.tiles_r * (int)((cols + tile_c - 1) / tile_c);
  return a;
}

template <typename T>
int write_tiles(int rows, int cols, int* tiles_r, int* lr) {
  *lr = row_lanes<T>(rows, ROW_LOG);
  const int64_t tile_r = sc_vl<T>() << *lr, tile_c = SC_WCOLS * (SC_THREADS >> *lr);
  *tiles_r = (int)((rows + tile_r - 1) / tile_r);
  return *tiles_r * (int)((cols + tile_c - 1) / tile_c);
}

// Scaled copies of A and B, r and s.
template <typename T>
hipError_t run_scaling(const FmScaleArgs& a, hipStream_t st) {
  const int m = a.m, k = a.k, n = a.n;
  T *A = reinterpret_cast<T*>(a.A), *B = reinterpret_cast<T*>(a.B);
  T *r = reinterpret_cast<T*>(a.r), *s = reinterpret_cast<T*>(a.s);
  // maxima, then factors: rows of A, columns of B (outer); columns of A, rows of B (inner)
  T *fa = reinterpret_cast<T*>(a.f), *fb = reinterpret_cast<T*>(a.f2);
  T *ga = reinterpret_cast<T*>(a.u1), *gb = reinterpret_cast<T*>(a.u2);
  const int longest = m > n ? (m > k ? m : k) : (n > k ? n : k);
  // the first step reads the caller's matrices, later ones the scaled copies
  const T *X = reinterpret_cast<const T*>(a.srcA), *Y = reinterpret_cast<const T*>(a.srcB);
  int64_t ldx = a.ld_srcA, ldy = a.ld_srcB;
  const bool outer_first = a.type == 0 || a.type == 3, outer = a.type != 2, inner = a.type != 3;
  auto maxima = [&](bool out, bool second) {
    // the second pass sees the products with the first pass's factors
    const T* pa = !second ? nullptr : out ? ga : fa;
    const T* pb = !second ? nullptr : out ? gb : fb;
    const MaxArgs<T> ma = max_args<T>(X, ldx, m, k, out, pa, out ? fa : ga);
    const MaxArgs<T> mb = max_args<T>(Y, ldy, k, n, !out, pb, out ? fb : gb);
    const bool whole = ma.lr == (ma.rowwise ? ROW_LOG : COL_LOG) && mb.lr == (mb.rowwise ? ROW_LOG : COL_LOG);
    auto* kernel = whole ? &fm_max_kernel<T, false> : &fm_max_kernel<T, true>;
    hipLaunchKernelGGL(kernel, dim3(ma.tiles + mb.tiles), dim3(SC_THREADS), 0, st, ma, mb);
    if (out)
      hipLaunchKernelGGL(fm_outer_factors<T>, dim3(blocks_for(m > n ? m : n)), dim3(256), 0, st, fa, r, m,
                         fb, s, n);
    else
      hipLaunchKernelGGL(fm_inner_factors<T>, dim3(blocks_for(k)), dim3(256), 0, st, ga, gb, k);
  };
  auto write = [&](const T* ra, const T* ca, const T* rb, const T* cb) {
    WriteArgs<T> wa{X, ldx, A, a.lda, m, k, ra, ca, outer_first, 0, 0, 0};
    WriteArgs<T> wb{Y, ldy, B, a.ldb, k, n, rb, cb, !outer_first, 0, 0, 0};
    wa.tiles = write_tiles<T>(m, k, &wa.tiles_r, &wa.lr);
    wb.tiles = write_tiles<T>(k, n, &wb.tiles_r, &wb.lr);
    auto* kernel = wa.lr == ROW_LOG && wb.lr == ROW_LOG ? &fm_write_kernel<T, false> : &fm_write_kernel<T, true>;
    hipLaunchKernelGGL(kernel, dim3(wa.tiles + wb.tiles), dim3(SC_THREADS), 0, st, wa, wb);
  };
  auto init = [&](int first) {
    hipLaunchKernelGGL(fm_scale_init<T>, dim3(blocks_for(longest)), dim3(256), 0, st, fa, r, m, fb, s, n, ga,
                       gb, k, first);
  };
  if (a.steps == 0) {
    init(1);
    write(nullptr, nullptr, nullptr, nullptr);
  }
  for (int it = 0; it < a.steps; ++it) {
    init(it == 0);
    if (outer && outer_first) maxima(true, false);
    if (inner) maxima(false, a.type == 0);
    if (outer && !outer_first) maxima(true, true);
    write(outer ? fa : nullptr, inner ? ga : nullptr, inner ? gb : nullptr, outer ? fb : nullptr);
    X = A;
    Y = B;
    ldx = a.lda;
    ldy = a.ldb;
  }
  return hipGetLastError();
}

}  // namespace

hipError_t fm_scaling_run(int dtype_f64, const FmScaleArgs& a, hipStream_t s) {
  return dtype_f64 ? run_scaling<double>(a, s) : run_scaling<float>(a, s);
}

template <typename T>
static void post(const void* P, int64_t ldp, void* C, int64_t ldc, int rows, int cols, const void* r,
                 const void* sv, double alpha, double beta, hipStream_t s) {
  int tiles_r, lr;
  const int tiles = write_tiles<T>(rows, cols, &tiles_r, &lr);
  auto* kernel = lr == ROW_LOG ? &fm_post_kernel<T, true> : &fm_post_kernel<T, false>;
  hipLaunchKernelGGL(kernel, dim3(tiles), dim3(SC_THREADS), 0, s, reinterpret_cast<const T*>(P), ldp,
                     reinterpret_cast<T*>(C), ldc, rows, cols, reinterpret_cast<const T*>(r),
                     reinterpret_cast<const T*>(sv), (T)alpha, (T)beta, tiles_r, lr);
}

hipError_t fm_scaling_post(int dtype_f64, const void* P, int64_t ldp, void* C, int64_t ldc,
                           int rows, int cols, const void* r, const void* sv, double alpha,
                           double beta, hipStream_t s) {
  if (dtype_f64)
    post<double>(P, ldp, C, ldc, rows, cols, r, sv, alpha, beta, s);
  else
    post<float>(P, ldp, C, ldc, rows, cols, r, sv, alpha, beta, s);
  return hipGetLastError();
}
