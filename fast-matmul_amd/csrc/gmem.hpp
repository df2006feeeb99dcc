// gmem.hpp -- global-memory pointers for device code.
//
// Operand addresses reach the kernels through descriptor tables, so the
// compiler cannot tell that they point to global memory and emits flat
// loads and stores.  A flat access counts against the LDS wait counter as
// well as the vector-memory one, and may complete out of order with LDS
// reads, so every wait for an LDS read then also waits for all global
// loads in flight: a GEMM's register prefetch of the next K slice stalls
// the first MFMAs that follow it.  Casting to the global address space
// gives global_load/global_store, which only the vector-memory counter
// tracks.
#pragma once

#include <hip/hip_runtime.h>

template <typename T>
using fm_gptr = __attribute__((address_space(1))) T*;

template <typename T>
__device__ __forceinline__ fm_gptr<T> fm_global(T* p) {
  return (fm_gptr<T>)p;
}

// fm_ptr<G, T>: T* in the global address space when G, generic otherwise
// (for kernels whose measured speed decides the form per element type).
template <bool G, typename T>
struct fm_ptr_sel {
  using type = T*;
};
template <typename T>
struct fm_ptr_sel<true, T> {
  using type = fm_gptr<T>;
};
template <bool G, typename T>
using fm_ptr = typename fm_ptr_sel<G, T>::type;

// Map a work-group id to a tile id.  The 8 XCDs receive work groups round-robin
// and each has its own L2, so an XCD's consecutive work groups take
// consecutive tiles, which share A/B panels: with chunk == 0 each XCD walks one
// eighth of the tiles, otherwise every eighth run of `chunk` tiles (64: the
// tiles an XCD's 32 CUs hold at a time).  A launch whose products differ in
// depth takes chunks, deepest products first: eighths of equal tile count are
// not equal work (64 FP32 problems of 512 to 4096 a side: 103 -> 136 TFLOP/s),
// and the last tiles to start are then short ones.
__device__ __forceinline__ int fm_xcd_tile(int wg, int nwg, int chunk) {
  if (chunk == 0) {
    const int full = nwg & ~7;
    return wg < full ? (wg & 7) * (full >> 3) + (wg >> 3) : wg;
  }
  const int round = 8 * chunk, full = nwg / round * round;
  if (wg >= full) return wg;
  const int i = wg >> 3;  // position among this XCD's work groups
  return (i / chunk * 8 + (wg & 7)) * chunk + i % chunk;
}
