// 2-D fine-grid operator y = A_hat(E) x, fused with its epilogue (modes as in op_tiled.hpp):
//
//   TM_Y y = A x; TM_RES y = b - A x; TM_JAC y = x + w D^-1 (b - A x); TM_JAC_ADD the same + xadd;
//   TM_YDOT y = A x and per-workgroup sums of x.y; TM_JAC0 the first two Jacobi sweeps from the
//   zero guess (x = w D^-1 b formed while staging); TM_JAC_ADD_DOT TM_JAC_ADD and per-workgroup
//   sums of bdot.y (bdot in FP64 also beside FP32 sweeps: r.z loses nothing to r's FP32 copy).
//
// A_hat = M K(E) M + I_c with any symmetric or unsymmetric 8 x 8 K0 (core/_templated_cuda.cu:782-834
// for Q4 elements).  One thread owns one node of a 32 x 8 tile and sums its four elements in the
// reference's order, so every output is written once and the order is fixed.
//
// What bounds it is load latency: nodes run fastest in x and elements fastest in y, so gathering E
// per node touches a cache line per lane and element, in four dependent rounds.  Here the tile's
// nodes (masked by the constraints) and its elements are staged in LDS by loads that are all in
// flight at once, with the epilogue's operands, behind one barrier.  FP64 y = A x at 1024 x 512:
// 28.4 -> 13.2 us (22 MB, 1.7 TB/s); FP32 Jacobi sweep at 512 x 256: 10.9 -> 5.8 us.  Two nodes per
// thread keep K0's 64 entries beside two sums and spill scalars (17.4 us); 32 x 16 tiles measured
// the same, K0 read from LDS 14.6 us.
#include "blas.hpp"
#include "common.hpp"
#include "op_tiled.hpp"
#include "stiffness.hpp"

namespace et {

namespace {

constexpr int kTX = 32, kTY = 8;  // nodes per tile, one per thread

template <typename T, int MODE>
__global__ __launch_bounds__(256) void op2d_kernel(const Grid g, const T* __restrict__ K0, const T* __restrict__ E,
                                                   const uint8_t* __restrict__ cons, const T* __restrict__ x,
                                                   const T* __restrict__ b, const T* __restrict__ Dinv,
                                                   const double* __restrict__ omega, double wscale,
                                                   const T* __restrict__ xadd, T* __restrict__ y,
                                                   const double* __restrict__ bdot, double* __restrict__ part) {
  constexpr int PX = kTX + 2, PY = kTY + 2, EX = kTX + 1, EY = kTY + 1;
  constexpr bool kJac = MODE == TM_JAC || MODE == TM_JAC_ADD || MODE == TM_JAC0 || MODE == TM_JAC_ADD_DOT;
  constexpr bool kAdd = MODE == TM_JAC_ADD || MODE == TM_JAC_ADD_DOT;
  __shared__ T su[2][PY * PX];
  __shared__ T sE[EX * EY];  // y fastest; EY is odd, so lanes along x fall into different banks
  const int tid = threadIdx.x, tx = tid & 31, ty = tid >> 5;
  const int nx = g.nx(), ny = g.ny(), ntx = (nx + kTX - 1) / kTX;
  const int x0 = blockIdx.x % ntx * kTX, y0 = blockIdx.x / ntx * kTY;
  const T w = kJac ? (T)((omega != nullptr ? *omega : 1.0) * wscale) : T(0);

  // the own node's operands (clamped to the grid: every lane loads)
  const int i = x0 + tx, j = y0 + ty;
  T ob[2], od[2], oa[2], ox[2];
  double ot[2];
  bool fixed[2];
  {
    const int d = 2 * (min(j, ny - 1) * nx + min(i, nx - 1));
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      if (MODE != TM_Y && MODE != TM_YDOT) ob[c] = b[d + c];
      if (kJac) od[c] = Dinv[d + c];
      if (kAdd) oa[c] = xadd[d + c];
      if (MODE == TM_JAC_ADD_DOT) ot[c] = bdot[d + c];
      if (MODE != TM_JAC0) ox[c] = x[d + c];
      fixed[c] = cons != nullptr && cons[d + c] != 0;
    }
  }
#pragma unroll
  for (int q = 0; q < (PX * PY + 255) / 256; ++q) {
    const int t = tid + 256 * q;
    const int si = x0 - 1 + t % PX, sj = y0 - 1 + t / PX;
    const bool in = si >= 0 && si < nx && sj >= 0 && sj < ny;
    const int d = 2 * (min(max(sj, 0), ny - 1) * nx + min(max(si, 0), nx - 1));
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const T v = MODE == TM_JAC0 ? w * Dinv[d + c] * b[d + c] : x[d + c];
      const bool fx = cons != nullptr && cons[d + c] != 0;
      if (t < PX * PY) su[c][t] = in && !fx ? v : T(0);
    }
  }
#pragma unroll
  for (int q = 0; q < (EX * EY + 255) / 256; ++q) {
    const int t = tid + 256 * q;
    const int ex = x0 - 1 + t / EY, ey = y0 - 1 + t % EY;
    const T v = E[min(max(ex, 0), g.ex - 1) * g.ey + min(max(ey, 0), g.ey - 1)];
    if (t < EX * EY) sE[t] = v;
  }
  __syncthreads();

  T acc[2] = {T(0), T(0)};
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    T s[2] = {T(0), T(0)};
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const T u = su[c][(ty + 1 - qy(a) + qy(nb)) * PX + tx + 1 - qx(a) + qx(nb)];
        s[0] += K0[(2 * a) * 8 + 2 * nb + c] * u;
        s[1] += K0[(2 * a + 1) * 8 + 2 * nb + c] * u;
      }
    const int ex = i - qx(a), ey = j - qy(a);
    const bool in = ex >= 0 && ex < g.ex && ey >= 0 && ey < g.ey;
    const T e = sE[(tx + 1 - qx(a)) * EY + ty + 1 - qy(a)];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const T v = acc[c] + e * s[c];
      acc[c] = in ? v : acc[c];
    }
  }

  double dot = 0.0;
  if (i < nx && j < ny) {
    const int d = 2 * (j * nx + i);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const T xv = MODE == TM_JAC0 ? rounded(w * od[c] * ob[c]) : ox[c];
      const T ax = fixed[c] ? xv : acc[c];
      T v;
      if (MODE == TM_Y || MODE == TM_YDOT)
        v = ax;
      else if (MODE == TM_RES)
        v = ob[c] - ax;
      else
        v = xv + w * od[c] * (ob[c] - ax);
      if (kAdd) v += oa[c];
      y[d + c] = v;
      if (MODE == TM_YDOT) dot += (double)xv * (double)v;
      if (MODE == TM_JAC_ADD_DOT) dot += ot[c] * (double)v;
    }
  }
  if (MODE == TM_YDOT || MODE == TM_JAC_ADD_DOT) {
    dot = block_sum256(dot);
    if (tid == 0) part[blockIdx.x] = dot;
  }
}

}  // namespace

int op2d_partials(const Grid& g) {
  return ((g.nx() + kTX - 1) / kTX) * ((g.ny() + kTY - 1) / kTY);
}

template <typename T>
int op2d(int mode, const Grid& g, const T* K0, const T* E, const uint8_t* cons, const T* x, const T* b, const T* Dinv,
         const double* omega, double wscale, const T* xadd, T* y, const double* bdot, double* part, hipStream_t s) {
  const unsigned grid = op2d_partials(g);
#define ET_OP2(M) \
  op2d_kernel<T, M><<<grid, 256, 0, s>>>(g, K0, E, cons, x, b, Dinv, omega, wscale, xadd, y, bdot, part)
  switch (mode) {
    case TM_Y: ET_OP2(TM_Y); break;
    case TM_RES: ET_OP2(TM_RES); break;
    case TM_JAC: ET_OP2(TM_JAC); break;
    case TM_YDOT: ET_OP2(TM_YDOT); break;
    case TM_JAC0: ET_OP2(TM_JAC0); break;
    case TM_JAC_ADD_DOT: ET_OP2(TM_JAC_ADD_DOT); break;
    default: ET_OP2(TM_JAC_ADD); break;
  }
#undef ET_OP2
  ET_CHECK_LAUNCH();
  return ET_OK;
}

template int op2d<double>(int, const Grid&, const double*, const double*, const uint8_t*, const double*, const double*,
                          const double*, const double*, double, const double*, double*, const double*, double*,
                          hipStream_t);
template int op2d<float>(int, const Grid&, const float*, const float*, const uint8_t*, const float*, const float*,
                         const float*, const double*, double, const float*, float*, const double*, double*,
                         hipStream_t);

}  // namespace et
