// gemm_thin.hpp -- dynamic-peeling products: one dimension is the remainder of
// a block split, the others are a node's full size.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "alg_desc.hpp"

// Largest thin dimension the kernels are built for: the remainder of a split into
// FM_THIN_MAX + 1 blocks, the finest of the shipped tables.  Wider strips are
// several products; a K beyond it is summed by a loop.  (Each further value costs
// every FP64 strip registers: built up to 7, 182 of them, two waves a SIMD.)
constexpr int FM_THIN_MAX = 5;
// the largest thin dimension of a split into s blocks, as the kernels take it
constexpr int fm_thin_limit(int s) { return s <= 1 ? 1 : s - 1 > FM_THIN_MAX ? FM_THIN_MAX : s - 1; }
constexpr int FM_THIN_THREADS = 256;

// which dimension is thin, i.e. which of the three peeling products it is
enum FmThinKind : int32_t {
  FM_THIN_K = 0,  // C (+)= A B with a thin K: an update of all of C
  FM_THIN_N = 1,  // N <= FM_THIN_MAX columns: reads A once
  FM_THIN_M = 2,  // M <= FM_THIN_MAX rows: reads B once
};

// One product C = alpha * A * B + beta * C (linalg/linalg.hpp:201-244).
struct FmThinDesc {
  FmOp a, b, c;
  int32_t M, N, K;
  int32_t kind;
  int32_t tiles_m;     // tiles along M (kind M: 1)
  int32_t tile_begin;  // first tile of this product in the launch
  double alpha, beta;
};

struct FmThinArgs {
  FmBases bases;
  const FmThinDesc* descs;  // ordered by kind
  int32_t ndesc, total_tiles;
  // uniform: the products of each kind have one shape, and a tile finds its
  // product by division: kind q starts at tile t0[q] and product d0[q], with
  // per[q] tiles a product (per = 1 where the kind is absent)
  int32_t uniform;
  int32_t t0[3], d0[3], per[3];
};

// output tile of a product of each kind and depth: rows x columns of C per work group
void fm_thin_tile(int dtype_f64, int kind, int K, int* rows, int* cols);
hipError_t fm_thin_launch(int dtype_f64, const FmThinArgs& a, hipStream_t s);
