// 2-D V(2,2) cycles, two launches per level instead of six.
//
// A 2-D hierarchy is small (a level has at most a few hundred thousand nodes): each kernel of a
// V-cycle is a launch and one round of dependent loads, about 3 us whatever its size, and the
// cycle is a chain of them.  Per level (CuMultiGrid's cycle, solvers/_multigrid_cuda.py:133-186)
//
//   down  x0 = w D^-1 b, x1 = x0 + w D^-1 (b - A x0), r = b - A x1, b_c = R r
//   up    e0 = P x_c, e1 = e0 + w D^-1 (r - A e0), x = x1 + e1 + w D^-1 (r - A e1)
//
// are each one kernel: a workgroup owns 16 x 16 nodes and computes the earlier stages on a halo
// that shrinks by one node per stage (down 21, 19, 17 nodes wide; up 20, 18, 16), in LDS.  The halo
// is recomputed, 1.3 times the sweeps' work, which is far from what bounds them.  512 threads, so
// that every stage is one round.  A is the element operator on level 0 (any K0, constrained rows
// identity) and the half-stored block stencil below (layout in solver.hip); a thread keeps one node
// through the stages, so the stencil's 36 values are loaded once, ahead of the first stage (6.4 ->
// 5.2 us for a leg down in FP32, 6.2 -> 5.2 in FP64).  Sums run in the order of the single kernels.
// The convergence test of the PCG iteration is part of the first leg down: every workgroup sums r.r
// (up to 1024 partials) while its operands are on their way (512 x 256: the leg takes 9.2 us with it,
// 7.2 without), instead of a launch of 4 us between the update of r and the cycle.
// Six launches per level -> two: 120 x 40 FP64 solve 3.47 -> 2.76 ms.  The legs also read each vector
// once where the single kernels read it up to three times, so they stay ahead on large grids: a PCG
// iteration takes 143 us at 1024 x 512, mixed, and 855 us at 2048 x 2048, FP64, where six launches
// of per-node gathers took 270 and 1730.
#include "blas.hpp"
#include "common.hpp"
#include "mg_weights.hpp"
#include "op_tiled.hpp"
#include "pcg_check.hpp"
#include "stiffness.hpp"
#include "vcycle_2d.hpp"

namespace et {

namespace {

constexpr int kW = 16;           // output nodes per tile side
constexpr int kThreads = 512;

// LDS field of two components on a square of side P, lower corner at (-H, -H) of the tile
template <typename T, int P>
struct Field {
  T v[2][P * P];
};

// (A u)(i, j): u at local (lx, ly) of a field of side P.  Level 0: elements of the tile in sE (side
// PE, local element (ex, ey) covers nodes ex .. ex + 1 of the field's numbering shifted by
// `shift`); u is zero on constrained DOFs and outside the grid, as E is.
template <typename T, int P, int PE>
__device__ __forceinline__ void apply_elements(const T* __restrict__ K0, const T* sE, int ex0, int ey0,
                                               const Field<T, P>& u, int lx, int ly, T (&acc)[2]) {
  acc[0] = acc[1] = T(0);
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    T s[2] = {T(0), T(0)};
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const T uv = u.v[c][(ly - qy(a) + qy(nb)) * P + lx - qx(a) + qx(nb)];
        s[0] += K0[(2 * a) * 8 + 2 * nb + c] * uv;
        s[1] += K0[(2 * a + 1) * 8 + 2 * nb + c] * uv;
      }
    // element whose corner a is the node; elements run fastest in y, and so does sE
    const T e = sE[(ex0 - qx(a)) * PE + ey0 - qy(a)];
#pragma unroll
    for (int c = 0; c < 2; ++c) acc[c] += e * s[c];
  }
}

// Coarse levels: the node's 36 stencil values, requested at the start of a kernel and kept for both
// of its stages.  A neighbour outside the grid reads the node itself and meets u = 0.
template <typename T>
struct Stencil {
  T f[5][2][2], b[5][2][2];

  __device__ __forceinline__ void load(const T* __restrict__ S, int N, int nx, int ny, int i, int j) {
    const int n = j * nx + i;
#pragma unroll
    for (int h = 0; h < 5; ++h) {
      const int o = 4 + h, oi = o / 3 - 1, oj = o % 3 - 1;
      const bool in = i - oi >= 0 && i - oi < nx && j - oj >= 0 && j - oj < ny;
      const int m = in ? n - (oj * nx + oi) : n;
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          f[h][r][c] = S[((h * 2 + r) * 2 + c) * N + n];
          if (h > 0) b[h][r][c] = S[((h * 2 + c) * 2 + r) * N + m];
        }
    }
  }

  template <int P>
  __device__ __forceinline__ void apply(const Field<T, P>& u, int lx, int ly, T (&acc)[2]) const {
    acc[0] = acc[1] = T(0);
#pragma unroll
    for (int h = 0; h < 5; ++h) {
      const int o = 4 + h, oi = o / 3 - 1, oj = o % 3 - 1;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const T uf = u.v[c][(ly + oj) * P + lx + oi];
#pragma unroll
        for (int r = 0; r < 2; ++r) acc[r] += f[h][r][c] * uf;
      }
      if (h > 0) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const T ub = u.v[c][(ly - oj) * P + lx - oi];
#pragma unroll
          for (int r = 0; r < 2; ++r) acc[r] += b[h][r][c] * ub;
        }
      }
    }
  }
};

// elements (x0 - H .. x0 - H + PE - 1) x (y0 - H ..) into sE[ex][ey], zero outside the grid
template <typename T, int PE>
__device__ __forceinline__ void stage_elements(const Grid& g, const T* __restrict__ E, int x0, int y0, T* sE) {
  for (int t = threadIdx.x; t < PE * PE; t += kThreads) {
    const int ex = x0 + t / PE, ey = y0 + t % PE;
    const bool in = ex >= 0 && ex < g.ex && ey >= 0 && ey < g.ey;
    const T v = E[min(max(ex, 0), g.ex - 1) * g.ey + min(max(ey, 0), g.ey - 1)];
    sE[t] = in ? v : T(0);
  }
}

template <typename T, bool L0>
__global__ __launch_bounds__(kThreads) void down2_kernel(const Grid g, const Grid gc, const T* __restrict__ op,
                                                         const T* __restrict__ E, const uint8_t* __restrict__ cons,
                                                         const T* __restrict__ b, const T* __restrict__ Dinv,
                                                         const double* __restrict__ omega, double wscale,
                                                         T* __restrict__ x1, T* __restrict__ r, T* __restrict__ bc,
                                                         const PcgCheck ck) {
  constexpr int P0 = kW + 5, P1 = kW + 3, P2 = kW + 1, PE = kW + 4;
  __shared__ Field<T, P0> fb, fd, u0;
  __shared__ Field<T, P1> u1, v1;  // x1 with constrained DOFs zeroed, and as it is (level 0)
  __shared__ Field<T, P2> fr;
  __shared__ T sE[L0 ? PE * PE : 1];
  __shared__ uint8_t fx[L0 ? P0 * P0 : 1];
  const int nx = g.nx(), ny = g.ny(), N = nx * ny;
  const int ntx = (nx + kW - 1) / kW;
  const int x0 = blockIdx.x % ntx * kW, y0 = blockIdx.x / ntx * kW;
  const int tid = threadIdx.x;

  // a thread's node of the second and third stage (x0 - 2 + lx, ...): one node, so that a coarse
  // level's stencil is loaded once
  const int t1 = min(tid, P1 * P1 - 1), lx = t1 % P1, ly = t1 / P1, i1 = x0 - 2 + lx, j1 = y0 - 2 + ly;
  const bool in1 = tid < P1 * P1 && i1 >= 0 && i1 < nx && j1 >= 0 && j1 < ny;
  Stencil<T> st1;
  if (!L0) st1.load(op, N, nx, ny, min(max(i1, 0), nx - 1), min(max(j1, 0), ny - 1));
  // operands of the first stage (clamped: every lane loads)
  const int t0 = min(tid, P0 * P0 - 1), i0 = x0 - 3 + t0 % P0, j0 = y0 - 3 + t0 / P0;
  const bool in0 = i0 >= 0 && i0 < nx && j0 >= 0 && j0 < ny;
  const int d0 = 2 * (min(max(j0, 0), ny - 1) * nx + min(max(i0, 0), nx - 1));
  T b0[2], dv0[2];
  bool f0[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    b0[c] = b[d0 + c];
    dv0[c] = Dinv[d0 + c];
    f0[c] = L0 && cons[d0 + c] != 0;
  }
  if (L0) stage_elements<T, PE>(g, E, x0 - 3, y0 - 3, sE);
  T w;
  if (L0 && ck.sc != nullptr) {
    // every workgroup sums r.r in the same order and takes omega from it; the first one records the
    // test.  Once the loop has stopped, omega does not matter: nothing of this cycle is used.
    __shared__ double srr[kThreads / 64];
    const PcgState st = pcg_state(ck.sc);
    double rr = 0.0;
    for (int t = tid; t < ck.n_rr; t += kThreads) rr += ck.rr_part[t];
    rr = wave_sum(rr);
    if ((tid & 63) == 0) srr[tid >> 6] = rr;
    __syncthreads();
    rr = 0.0;
#pragma unroll
    for (int k = 0; k < kThreads / 64; ++k) rr += srr[k];
    w = (T)(pcg_omega(sqrt(rr) / sqrt(st.bb), ck.tol, ck.wmin, ck.dw) * wscale);
    // by the last wavefront, which has no part in the next stages
    if (blockIdx.x == 0 && tid == kThreads - 1) pcg_check(ck, st, rr);
  } else {
    w = (T)(*omega * wscale);
  }
  if (tid < P0 * P0) {
    int m = 0;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      m |= f0[c] ? 1 << c : 0;
      fb.v[c][tid] = in0 ? b0[c] : T(0);
      fd.v[c][tid] = in0 ? dv0[c] : T(0);
      u0.v[c][tid] = in0 && !f0[c] ? w * dv0[c] * b0[c] : T(0);
    }
    if (L0) fx[tid] = (uint8_t)m;
  }
  __syncthreads();
  const int at = (ly + 1) * P0 + lx + 1;
  if (tid < P1 * P1) {
    T v[2] = {T(0), T(0)};
    if (in1) {
      T ax[2];
      if constexpr (L0)
        apply_elements<T, P0, PE>(op, sE, lx + 1, ly + 1, u0, lx + 1, ly + 1, ax);
      else
        st1.template apply<P0>(u0, lx + 1, ly + 1, ax);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const T bv = fb.v[c][at], dv = fd.v[c][at], xv = rounded(w * dv * bv);
        if (L0 && ((fx[at] >> c) & 1)) ax[c] = xv;
        v[c] = xv + w * dv * (bv - ax[c]);
        if (lx >= 2 && lx < kW + 2 && ly >= 2 && ly < kW + 2) x1[2 * (j1 * nx + i1) + c] = v[c];
      }
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      u1.v[c][tid] = L0 && ((fx[at] >> c) & 1) ? T(0) : v[c];
      if (L0) v1.v[c][tid] = v[c];
    }
  }
  __syncthreads();
  if (tid < P1 * P1 && lx >= 1 && lx <= P2 && ly >= 1 && ly <= P2) {
    T v[2] = {T(0), T(0)};
    if (in1) {
      T ax[2];
      if constexpr (L0)
        apply_elements<T, P1, PE>(op, sE, lx + 1, ly + 1, u1, lx, ly, ax);
      else
        st1.template apply<P1>(u1, lx, ly, ax);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        if (L0 && ((fx[at] >> c) & 1)) ax[c] = v1.v[c][tid];
        v[c] = fb.v[c][at] - ax[c];
        if (lx >= 2 && ly >= 2) r[2 * (j1 * nx + i1) + c] = v[c];
      }
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) fr.v[c][(ly - 1) * P2 + lx - 1] = v[c];
  }
  __syncthreads();
  if (L0 && ck.sc != nullptr && blockIdx.x == 0 && tid == kThreads - 1) __threadfence_system();
  // restriction to the coarse nodes whose fine node lies in the tile (r is zero outside the grid)
  constexpr int HC = kW / 2;
  if (tid < HC * HC) {
    const int cx = tid % HC, cy = tid / HC, ci = x0 / 2 + cx, cj = y0 / 2 + cy;
    if (ci < gc.nx() && cj < gc.ny()) {
      T acc[2] = {T(0), T(0)};
#pragma unroll
      for (int dj = -1; dj <= 1; ++dj)
#pragma unroll
        for (int di = -1; di <= 1; ++di) {
          const bool in = 2 * cj + dj >= 0 && 2 * cj + dj < ny && 2 * ci + di >= 0 && 2 * ci + di < nx;
          const T wgt = in ? (T)(pw(di) * pw(dj)) : T(0);
#pragma unroll
          for (int c = 0; c < 2; ++c) acc[c] += wgt * fr.v[c][(2 * cy + 1 + dj) * P2 + 2 * cx + 1 + di];
        }
      const T inv = inv_tw_of<T, 2>(gc, ci, cj, 0);
#pragma unroll
      for (int c = 0; c < 2; ++c) bc[2 * (cj * gc.nx() + ci) + c] = acc[c] * inv;
    }
  }
}

// DOT: also per-workgroup sums of bdot.x, bdot in FP64 (r.z with r's FP32 copy cost the mixed 2-D
// solver a quarter more iterations at 512 x 256)
template <typename T, bool L0, bool DOT>
__global__ __launch_bounds__(kThreads) void up2_kernel(const Grid g, const Grid gc, const T* __restrict__ op,
                                                       const T* __restrict__ E, const uint8_t* __restrict__ cons,
                                                       const T* __restrict__ xc, const T* __restrict__ r,
                                                       const T* __restrict__ x1, const T* __restrict__ Dinv,
                                                       const double* __restrict__ omega, double wscale,
                                                       T* __restrict__ x, const double* __restrict__ bdot,
                                                       double* __restrict__ part) {
  constexpr int P0 = kW + 4, P1 = kW + 2, PE = kW + 3;
  __shared__ Field<T, P0> u0, v0;
  __shared__ Field<T, P1> u1, v1;
  __shared__ T sE[L0 ? PE * PE : 1];
  __shared__ uint8_t fx[L0 ? P0 * P0 : 1];
  __shared__ double wsum[kThreads / 64];
  const int nx = g.nx(), ny = g.ny(), N = nx * ny, cnx = gc.nx(), cny = gc.ny();
  const int ntx = (nx + kW - 1) / kW;
  const int x0 = blockIdx.x % ntx * kW, y0 = blockIdx.x / ntx * kW;
  const T w = (T)(*omega * wscale);
  const int tid = threadIdx.x;
  // a thread's node (x0 - 1 + lx, ...) is the same in both sweeps: its operands and, on coarse
  // levels, its stencil are on their way while e0 is formed
  const int t1 = min(tid, P1 * P1 - 1), lx = t1 % P1, ly = t1 / P1, i1 = x0 - 1 + lx, j1 = y0 - 1 + ly;
  const bool in1 = tid < P1 * P1 && i1 >= 0 && i1 < nx && j1 >= 0 && j1 < ny;
  const bool in2 = in1 && lx >= 1 && lx <= kW && ly >= 1 && ly <= kW;
  const int ic1 = min(max(i1, 0), nx - 1), jc1 = min(max(j1, 0), ny - 1), d1 = 2 * (jc1 * nx + ic1);
  Stencil<T> st1;
  if (!L0) st1.load(op, N, nx, ny, ic1, jc1);
  T r1[2], dd1[2], xa[2];
  double bt[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    r1[c] = r[d1 + c];
    dd1[c] = Dinv[d1 + c];
    xa[c] = x1[d1 + c];
    bt[c] = DOT ? bdot[d1 + c] : 0.0;
  }
  if (L0) stage_elements<T, PE>(g, E, x0 - 2, y0 - 2, sE);
  if (tid < P0 * P0) {
    const int i = x0 - 2 + tid % P0, j = y0 - 2 + tid / P0;
    const bool in = i >= 0 && i < nx && j >= 0 && j < ny;
    const int ic = min(max(i, 0), nx - 1), jc = min(max(j, 0), ny - 1), ci = ic >> 1, cj = jc >> 1;
    // mean of the parents, each over its total weight, in j, i order
    const bool two_i = (ic & 1) && ci + 1 < cnx, two_j = (jc & 1) && cj + 1 < cny;
    T acc[2] = {T(0), T(0)};
#pragma unroll
    for (int pj = 0; pj < 2; ++pj)
#pragma unroll
      for (int pi = 0; pi < 2; ++pi) {
        const int pc = min(ci + pi, cnx - 1), qc = min(cj + pj, cny - 1);
        const T inv = inv_tw_of<T, 2>(gc, pc, qc, 0);
        const bool use = (pj == 0 || two_j) && (pi == 0 || two_i);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const T v = xc[2 * (qc * cnx + pc) + c] * inv;
          acc[c] += use ? v : T(0);
        }
      }
    const T scl = T(1) / (T)((two_i ? 2 : 1) * (two_j ? 2 : 1));
    int m = 0;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const bool f = L0 && cons[2 * (jc * nx + ic) + c] != 0;
      m |= f ? 1 << c : 0;
      const T v = in ? acc[c] * scl : T(0);
      u0.v[c][tid] = f ? T(0) : v;
      if (L0) v0.v[c][tid] = v;
    }
    if (L0) fx[tid] = (uint8_t)m;
  }
  __syncthreads();
  const int at = (ly + 1) * P0 + lx + 1;
  if (tid < P1 * P1) {
    T v[2] = {T(0), T(0)};
    if (in1) {
      T ax[2];
      if constexpr (L0)
        apply_elements<T, P0, PE>(op, sE, lx + 1, ly + 1, u0, lx + 1, ly + 1, ax);
      else
        st1.template apply<P0>(u0, lx + 1, ly + 1, ax);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const T e = L0 ? v0.v[c][at] : u0.v[c][at];
        if (L0 && ((fx[at] >> c) & 1)) ax[c] = e;
        v[c] = e + w * dd1[c] * (r1[c] - ax[c]);
      }
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      u1.v[c][tid] = L0 && ((fx[at] >> c) & 1) ? T(0) : v[c];
      if (L0) v1.v[c][tid] = v[c];
    }
  }
  __syncthreads();
  double dot = 0.0;
  if (in2) {
    T ax[2];
    if constexpr (L0)
      apply_elements<T, P1, PE>(op, sE, lx + 1, ly + 1, u1, lx, ly, ax);
    else
      st1.template apply<P1>(u1, lx, ly, ax);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const T e = L0 ? v1.v[c][tid] : u1.v[c][tid];
      if (L0 && ((fx[at] >> c) & 1)) ax[c] = e;
      T v = e + w * dd1[c] * (r1[c] - ax[c]);
      v += xa[c];
      x[d1 + c] = v;
      if (DOT) dot += bt[c] * (double)v;
    }
  }
  if (DOT) {
    dot = wave_sum(dot);
    if ((tid & 63) == 0) wsum[tid >> 6] = dot;
    __syncthreads();
    if (tid == 0) {
      double s = 0.0;
#pragma unroll
      for (int k = 0; k < kThreads / 64; ++k) s += wsum[k];
      part[blockIdx.x] = s;
    }
  }
}

}  // namespace

int vcycle2_tiles(const Grid& g) { return ((g.nx() + kW - 1) / kW) * ((g.ny() + kW - 1) / kW); }

template <typename T>
int vcycle2_down(const Grid& g, bool level0, const T* op, const T* E, const uint8_t* cons, const T* b, const T* Dinv,
                 const double* omega, double wscale, T* x1, T* r, T* bc, const PcgCheck* ck, hipStream_t s) {
  const int n = vcycle2_tiles(g);
  const PcgCheck c = ck != nullptr ? *ck : PcgCheck{};
  if (level0)
    down2_kernel<T, true><<<n, kThreads, 0, s>>>(g, g.coarse(), op, E, cons, b, Dinv, omega, wscale, x1, r, bc, c);
  else
    down2_kernel<T, false><<<n, kThreads, 0, s>>>(g, g.coarse(), op, E, cons, b, Dinv, omega, wscale, x1, r, bc, c);
  ET_CHECK_LAUNCH();
  return ET_OK;
}

template <typename T>
int vcycle2_up(const Grid& g, bool level0, const T* op, const T* E, const uint8_t* cons, const T* xc, const T* r,
               const T* x1, const T* Dinv, const double* omega, double wscale, T* x, const double* bdot, double* part,
               hipStream_t s) {
  const int n = vcycle2_tiles(g);
  const Grid gc = g.coarse();
  if (!level0)
    up2_kernel<T, false, false><<<n, kThreads, 0, s>>>(g, gc, op, E, cons, xc, r, x1, Dinv, omega, wscale, x, bdot, part);
  else if (part == nullptr)
    up2_kernel<T, true, false><<<n, kThreads, 0, s>>>(g, gc, op, E, cons, xc, r, x1, Dinv, omega, wscale, x, bdot, part);
  else
    up2_kernel<T, true, true><<<n, kThreads, 0, s>>>(g, gc, op, E, cons, xc, r, x1, Dinv, omega, wscale, x, bdot, part);
  ET_CHECK_LAUNCH();
  return ET_OK;
}

#define ET_V2(T)                                                                                                    \
  template int vcycle2_down<T>(const Grid&, bool, const T*, const T*, const uint8_t*, const T*, const T*,           \
                               const double*, double, T*, T*, T*, const PcgCheck*, hipStream_t);                    \
  template int vcycle2_up<T>(const Grid&, bool, const T*, const T*, const uint8_t*, const T*, const T*, const T*,   \
                             const T*, const double*, double, T*, const double*, double*, hipStream_t);
ET_V2(double)
ET_V2(float)
#undef ET_V2

}  // namespace et
