// Weights of the grid transfers (device code).
#pragma once
#include "common.hpp"

namespace et {

__device__ __forceinline__ double pw(int d) {  // 2^-|d| for d in {-1, 0, 1}
  return d == 0 ? 1.0 : 0.5;
}

// 1/tw(c) as a product of per-axis factors (2/3 on the boundary, 1/2 inside),
// in the working precision: no division in the transfer kernels
template <typename T, int DIM>
__device__ __forceinline__ T inv_tw_of(const Grid& gc, int i, int j, int k) {
  const T bnd = T(2.0 / 3.0), mid = T(0.5);
  T t = (i == 0 || i == gc.nx() - 1) ? bnd : mid;
  t *= (j == 0 || j == gc.ny() - 1) ? bnd : mid;
  if (DIM == 3) t *= (k == 0 || k == gc.nz() - 1) ? bnd : mid;
  return t;
}

}  // namespace et
