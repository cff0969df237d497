// Matrix-free operator of the first coarse multigrid level.
//
// With even fine element counts every fine element is one of the 8 children
// t of a coarse element C, and the Galerkin operator A_1 = R A_hat R^T
// (R = D^-1 P^T, D the total weights tw) splits into
//     A_1 = D^-1 ( sum_C Q_C^T K_C Q_C ) D^-1 + dA,   K_C = sum_t E_t M_t,
// where M_t = W_t^T K0 W_t and dA collects everything constrained fine DOFs
// change (masked children and the identity rows); dA is non-zero only at the
// coarse nodes of coarse elements with a constrained child, whose rows of A_1
// are stored whole.
//
// Element product in the corner Walsh-Hadamard basis (8-point transform H per
// displacement component): reflecting child 0 onto child t is diagonal there,
// so  H K_C H / 64 = Mh o Eh  with a fixed 24 x 24 matrix Mh (279 structural
// non-zeros, level1_terms.hpp) and Eh[(M,c),(N,d)] = (H E_C)[M^N^e_c^e_d],
// H E_C being the transform of the 8 children's densities (computed once per
// solve).  Per coarse element: one forward transform of the tw-scaled corner
// values, 279 + 150 FMAs, one inverse transform.
//
// One launch per application, no atomics, fixed summation order:
//   tiles    a workgroup owns a tile of (cx - 1) x (cy - 1) node columns (all of z, or zl nodes of it)
//            and the cx x cy element columns around it.  The nodes' x / tw are staged in LDS; a lane
//            computes one element (whole columns side by side in a wavefront), its top (bz = 1)
//            results move one lane up, and the four node sums are added to LDS accumulators one face
//            corner after the other, so no two columns add to one node at a time; then the mode's
//            epilogue (y = Ax, b - Ax, Jacobi, Jacobi + add), every output written once;
//   rows     nodes of coarse elements with a constrained child take their operator row, stored at
//            setup from the Galerkin stencil, in workgroups of their own at the front of the grid.
// Small grids are bound by latency, above all by the chain of 279 scalar coefficients: there a
// wavefront computes one of the three output components, three wavefronts to an element.  Large ones
// are bound by VALU issue, cx cy / ((cx - 1)(cy - 1)) times the grid's elements.  Per application
// (before: an element, a node and a correction kernel, the corrections as A_1 - sum_C):
//   FP64 61 x 29 x 25 nodes 24 -> 13 us, FP32 33 x 17 x 17 17 -> 8 us, FP32 129 x 65 x 65 39 -> 29 us,
//   FP64 129 x 65 x 65 57 -> 53 us.
// Capping the registers for two workgroups per compute unit spills (FP32 129 x 65 x 65: 36 us).
#include <cmath>
#include <vector>

#include "common.hpp"
#include "galerkin_elem.hpp"
#include "level1.hpp"
#include "level1_terms.hpp"

namespace et {

static int g_level1_mf = 1;
void set_level1_mf(int on) { g_level1_mf = on ? 1 : 0; }
int get_level1_mf() { return g_level1_mf; }

bool level1_supported(const Grid& g0, int n_level) {
  return g0.dim == 3 && n_level >= 2 && galerkin_elem_supported(g0);
}

// corner-bit order (beta = bx + 2 by + 4 bz) -> H8 local corner index
__host__ __device__ constexpr int l1_corner(int beta) {
  return (beta & 4 ? 4 : 0) + ((beta & 2) ? ((beta & 1) ? 2 : 3) : ((beta & 1) ? 1 : 0));
}

// 1/tw of a node in the working precision, as a product of per-axis factors
template <typename T>
__device__ __forceinline__ T l1_inv_tw_t(const Grid& g, int i, int j, int k) {
  const T bnd = T(2.0 / 3.0), mid = T(0.5);
  T t = (i == 0 || i == g.nx() - 1) ? bnd : mid;
  t *= (j == 0 || j == g.ny() - 1) ? bnd : mid;
  t *= (k == 0 || k == g.nz() - 1) ? bnd : mid;
  return t;
}

// ------------------------------------------------------------ setup ----

template <typename T>
__global__ void l1_eh_kernel(const Grid g0, const Grid g1, const double* __restrict__ E,
                             const uint8_t* __restrict__ eflag, T* __restrict__ Eh,
                             uint8_t* __restrict__ special) {
  const int C = blockIdx.x * blockDim.x + threadIdx.x;
  if (C >= (int)g1.n_elem()) return;
  const int K = C % g1.ez, IJ = C / g1.ez, J = IJ % g1.ey, I = IJ / g1.ey;
  double v[8];
  uint8_t sp = 0;
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const int64_t e = ((int64_t)(2 * I + (t & 1)) * g0.ey + 2 * J + ((t >> 1) & 1)) * g0.ez + 2 * K + (t >> 2);
    v[t] = E[e];
    sp |= eflag[e];
  }
  wht8(v);
#pragma unroll
  for (int m = 0; m < 8; ++m) Eh[(int64_t)C * 8 + m] = (T)v[m];
  special[C] = sp ? 1 : 0;
}

__global__ void l1_affected_kernel(const Grid g1, const uint8_t* __restrict__ special,
                                   int* __restrict__ aidx, int* __restrict__ alist, int* __restrict__ count) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= (int)g1.n_nodes()) return;
  const int k = n % g1.nz(), ij = n / g1.nz(), i = ij % g1.nx(), j = ij / g1.nx();
  bool hit = false;
  for (int beta = 0; beta < 8; ++beta) {
    const int I = i - (beta & 1), J = j - ((beta >> 1) & 1), K = k - (beta >> 2);
    if (I < 0 || I >= g1.ex || J < 0 || J >= g1.ey || K < 0 || K >= g1.ez) continue;
    if (special[(I * g1.ey + J) * g1.ez + K]) hit = true;
  }
  int idx = -1;
  if (hit) {
    idx = atomicAdd(count, 1);
    alist[idx] = n;
  }
  aidx[n] = idx;
}

// Operator rows [27][3][3] of the listed nodes, from the true Galerkin stencil S1.
template <typename T>
__global__ void l1_rows_kernel(const Grid g1, const double* __restrict__ S1, const int* __restrict__ alist, int n_aff,
                               T* __restrict__ rows) {
  const int tid = blockIdx.x * blockDim.x + threadIdx.x;
  if (tid >= n_aff * 27) return;
  const int o = tid / n_aff, a = tid - o * n_aff, n = alist[a];
  const int nx = g1.nx(), ny = g1.ny(), nz = g1.nz();
  const int k = n % nz + o % 3 - 1, ij = n / nz, i = ij % nx + o / 9 - 1, j = ij / nx + (o / 3) % 3 - 1;
  const bool in = i >= 0 && i < nx && j >= 0 && j < ny && k >= 0 && k < nz;
  const int64_t N = g1.n_nodes();
#pragma unroll
  for (int e = 0; e < 9; ++e) {
    const double v = S1[(int64_t)(o * 9 + e) * N + n];
    rows[(int64_t)a * 243 + o * 9 + e] = in ? (T)v : T(0);
  }
}

// ------------------------------------------------------------ apply ----

constexpr int kL1FixNodes = 2;  // corrected nodes per 32 lanes
// FP32 grids below this take one output component per wavefront: 12.4 against 13.5 us at 44 225 nodes,
// 15.7 against 11.6 us at 99 225.  FP64 needs the split for its registers.
constexpr int64_t kL1SplitNodes = 65536;

struct L1Args {
  Grid g;
  L1Plan p;
};

// t / d for t < 2^16 by the reciprocal: (t + 1/2) / d is at least 1 / (2 d) from an integer, d <= 66
// or a tile's column count, and the product's rounding is below t / d * 2^-22
__device__ __forceinline__ int l1_div(int t, float inv) { return (int)(((float)t + 0.5f) * inv); }

// y at one degree of freedom from ax = (A x)_d
template <typename T, int MODE>
__device__ __forceinline__ T l1_epilogue(T ax, T xv, T bv, T dv, T w, T av) {
  if (MODE == 0) return ax;
  if (MODE == 1) return bv - ax;
  const T v = xv + w * dv * (bv - ax);
  return MODE == 3 ? v + av : v;
}

template <typename T, int MODE, bool SPLIT>
__global__ __launch_bounds__(SPLIT ? 768 : 1024) void l1_tile_kernel(
    const L1Args A, const T* __restrict__ cf, const T* __restrict__ Eh, const int* __restrict__ aidx,
    const int* __restrict__ alist, int n_aff, int n_fix, const T* __restrict__ rows, const T* __restrict__ x,
    const T* __restrict__ b, const T* __restrict__ Dinv, const double* __restrict__ omega, double wscale,
    const T* __restrict__ xadd, T* __restrict__ y) {
  extern __shared__ __align__(16) unsigned char l1_lds[];
  constexpr int kThreads = SPLIT ? 768 : 1024, kSlots = SPLIT ? 4 : 16;
  const Grid& g = A.g;
  const int nx = g.nx(), ny = g.ny(), nz = g.nz();
  const int tid = threadIdx.x;
  const T w = MODE >= 2 ? (T)((omega != nullptr ? *omega : 1.0) * wscale) : T(0);

  if ((int)blockIdx.x < n_fix) {
    // corrected nodes: 32 lanes a node, lane o < 27 the block of neighbour o
    const int o = tid & 31, oc = min(o, 26);
    for (int m = 0; m < kL1FixNodes; ++m) {
      const int a0 = (blockIdx.x * kL1FixNodes + m) * (kThreads / 32) + (tid >> 5), a = min(a0, n_aff - 1);
      const int n = alist[a];
      const int k = n % nz, ij = n / nz, i = ij % nx, j = ij / nx;
      const int mi = i + oc / 9 - 1, mj = j + (oc / 3) % 3 - 1, mk = k + oc % 3 - 1;
      const bool in = mi >= 0 && mi < nx && mj >= 0 && mj < ny && mk >= 0 && mk < nz;
      const int nb = in ? (mj * nx + mi) * nz + mk : n;
      const T* R = rows + (int64_t)a * 243 + oc * 9;
      T v[3] = {T(0), T(0), T(0)};
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const T xv = o < 27 && in ? x[nb * 3 + c] : T(0);
#pragma unroll
        for (int r = 0; r < 3; ++r) v[r] += R[r * 3 + c] * xv;
      }
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int h = 16; h > 0; h >>= 1) v[r] += __shfl_xor(v[r], h, 32);
      if (o < 3 && a0 < n_aff) {
        const int d = n * 3 + o;
        const T ax = o == 0 ? v[0] : o == 1 ? v[1] : v[2];
        y[d] = l1_epilogue<T, MODE>(ax, MODE >= 2 ? x[d] : T(0), MODE >= 1 ? b[d] : T(0), MODE >= 2 ? Dinv[d] : T(0),
                                    w, MODE == 3 ? xadd[d] : T(0));
      }
    }
    return;
  }

  const L1Plan& P = A.p;
  const int CX = P.cx, CY = P.cy;
  const int tile = blockIdx.x - n_fix;
  const int tx = tile % P.ntx, tyz = tile / P.ntx, ty = tyz % P.nty, tz = tyz / P.nty;
  const int X0 = tx * (CX - 1), Y0 = ty * (CY - 1), z0 = tz * P.zl, z1 = min(z0 + P.zl, nz);
  const int e0 = max(z0 - 1, 0), nle = min(z1, g.ez) - e0;  // elements of a column in this tile
  const int zs = P.lpc + 1;                                 // staged nodes of a column
  const int ncol = (CX + 1) * (CY + 1), ocol = (CX - 1) * (CY - 1);
  T* su = reinterpret_cast<T*>(l1_lds);  // [column][z][3], x / tw
  T* sa = su + 3 * ncol * zs;            // [output column][z][3]
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int slot = SPLIT ? wave / 3 : wave, comp = SPLIT ? wave - 3 * slot : 0;
  const int lcol = lane / P.lpc, lez = lane - lcol * P.lpc;
  const int kel = min(e0 + lez, g.ez - 1);

  // transformed densities of the lane's element of round q0; zero off the grid
  T eh[8];
  auto load_eh = [&](int q0) {
    const int q = min(q0 + slot * P.cpw + lcol, CX * CY - 1), cj = q / CX, ci = q - cj * CX;
    const int I = X0 - 1 + ci, J = Y0 - 1 + cj;
    const bool in = I >= 0 && I < g.ex && J >= 0 && J < g.ey;
    const int C = in ? (I * g.ey + J) * g.ez + kel : 0;
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const T v = Eh[(int64_t)C * 8 + m];
      eh[m] = in ? v : T(0);
    }
  };
  load_eh(0);

  // stage: loads are unconditional (clamped to the grid), four nodes of a thread in flight
  constexpr int kSC = 4;
  const float inv_zs = 1.0f / (float)zs, inv_cx1 = 1.0f / (float)(CX + 1);
  for (int t0 = tid; t0 < ncol * zs; t0 += kSC * kThreads) {
    T v[kSC][3];
#pragma unroll
    for (int m = 0; m < kSC; ++m) {
      const int t = min(t0 + m * kThreads, ncol * zs - 1);
      const int c = l1_div(t, inv_zs), z = e0 + t - c * zs, cj = l1_div(c, inv_cx1), i = X0 - 1 + c - cj * (CX + 1), j = Y0 - 1 + cj;
      const bool in = i >= 0 && i < nx && j >= 0 && j < ny && z < nz;
      const int ic = min(max(i, 0), nx - 1), jc = min(max(j, 0), ny - 1), zc = min(z, nz - 1);
      const T sw = l1_inv_tw_t<T>(g, ic, jc, zc);
      const int n = (jc * nx + ic) * nz + zc;
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        const T u = x[n * 3 + r];
        v[m][r] = in ? u * sw : T(0);
      }
    }
#pragma unroll
    for (int m = 0; m < kSC; ++m) {
      const int t = t0 + m * kThreads;
      if (t < ncol * zs)
#pragma unroll
        for (int r = 0; r < 3; ++r) su[t * 3 + r] = v[m][r];
    }
  }
  for (int t = tid; t < 3 * ocol * P.zl; t += kThreads) sa[t] = T(0);
  __syncthreads();

  for (int q0 = 0; q0 < CX * CY; q0 += kSlots * P.cpw) {
    const int q = q0 + slot * P.cpw + lcol;
    const bool valid = lcol < P.cpw && q < CX * CY && lez < nle;
    const int qc = min(q, CX * CY - 1), cj = qc / CX, ci = qc - cj * CX;
    const T* uc = su + ((cj * (CX + 1) + ci) * zs + min(lez, zs - 2)) * 3;
    T xh[3][8];
#pragma unroll
    for (int beta = 0; beta < 8; ++beta)
#pragma unroll
      for (int c = 0; c < 3; ++c)
        xh[c][beta] = uc[(((beta & 1) + ((beta >> 1) & 1) * (CX + 1)) * zs + (beta >> 2)) * 3 + c];
#pragma unroll
    for (int c = 0; c < 3; ++c) wht8(xh[c]);
    // node sums at the bottom face corners f = bx + 2 by, and the unmoved top results
    constexpr int NC = SPLIT ? 1 : 3;
    T sum[4][NC], top[4][NC];
    auto faces = [&](T (&v)[8], int s) {
      wht8(v);
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const T moved = lane_shr(v[f + 4]);
        sum[f][s] = v[f] + (lez > 0 ? moved : T(0));
        top[f][s] = v[f + 4];
      }
    };
    // the coefficients are wave-uniform: scalar loads that the compiler may not hoist
    const __attribute__((address_space(4))) T* k4 = (const __attribute__((address_space(4))) T*)(const void*)cf;
    asm volatile("" : "+s"(k4));
    auto coef = [&](int k) -> T { return k4[k]; };
    if constexpr (SPLIT) {
      T yh[3][8];
      if (comp == 0) {
        level1_product(xh, eh, coef, yh);
        faces(yh[0], 0);
      } else if (comp == 1) {
        level1_product(xh, eh, coef, yh);
        faces(yh[1], 0);
      } else {
        level1_product(xh, eh, coef, yh);
        faces(yh[2], 0);
      }
    } else {
      T yh[3][8];
      level1_product(xh, eh, coef, yh);
#pragma unroll
      for (int c = 0; c < NC; ++c) faces(yh[c], c);
    }
    load_eh(q0 + kSlots * P.cpw);
    // one face corner after the other: the columns of a round reach different nodes
    const bool last = lez == nle - 1 && e0 + nle < z1;
    const int zk = e0 + lez - z0;  // node below the element, -1 on the layer shared with the tile below
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      const int ti = ci + (f & 1) - 1, tj = cj + (f >> 1) - 1;
      if (valid && ti >= 0 && ti < CX - 1 && tj >= 0 && tj < CY - 1) {
        T* d = sa + ((tj * (CX - 1) + ti) * P.zl + zk) * 3 + comp;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          if (zk >= 0) d[c] += sum[f][c];
          if (last) d[c + 3] += top[f][c];
        }
      }
      __syncthreads();
    }
  }

  // nodes: the operands of kSN nodes are requested together
  constexpr int kSN = 3;
  const float inv_zl = 1.0f / (float)P.zl, inv_ox = 1.0f / (float)(CX - 1);
  for (int t0 = tid; t0 < ocol * P.zl; t0 += kSN * kThreads) {
    T pb[kSN][3], pd[kSN][3], px[kSN][3], pa[kSN][3];
    int pn[kSN], corrected[kSN];
    bool live[kSN];
    T sc[kSN];
#pragma unroll
    for (int m = 0; m < kSN; ++m) {
      const int t = min(t0 + m * kThreads, ocol * P.zl - 1);
      const int c = l1_div(t, inv_zl), z = z0 + t - c * P.zl, tj = l1_div(c, inv_ox), i = X0 + c - tj * (CX - 1), j = Y0 + tj;
      live[m] = t0 + m * kThreads < ocol * P.zl && i < nx && j < ny && z < z1;
      const int ic = min(i, nx - 1), jc = min(j, ny - 1), zc = min(z, nz - 1), n = (jc * nx + ic) * nz + zc;
      sc[m] = l1_inv_tw_t<T>(g, ic, jc, zc);
      pn[m] = n;
      corrected[m] = aidx[n];
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        pb[m][r] = MODE >= 1 ? b[n * 3 + r] : T(0);
        pd[m][r] = MODE >= 2 ? Dinv[n * 3 + r] : T(0);
        px[m][r] = MODE >= 2 ? x[n * 3 + r] : T(0);
        pa[m][r] = MODE == 3 ? xadd[n * 3 + r] : T(0);
      }
    }
#pragma unroll
    for (int m = 0; m < kSN; ++m) {
      if (!live[m] || corrected[m] >= 0) continue;
#pragma unroll
      for (int r = 0; r < 3; ++r)
        y[pn[m] * 3 + r] = l1_epilogue<T, MODE>(sa[(t0 + m * kThreads) * 3 + r] * sc[m], px[m][r], pb[m][r], pd[m][r],
                                                w, pa[m][r]);
    }
  }
}

// ------------------------------------------------------------ host ----

namespace {
constexpr size_t kL1MaxLds = 160 * 1024;

size_t l1_lds_bytes(const L1Plan& p, size_t elem_bytes) {
  return elem_bytes * 3 * ((size_t)(p.cx + 1) * (p.cy + 1) * (p.lpc + 1) + (size_t)(p.cx - 1) * (p.cy - 1) * p.zl);
}

// The tile with the least time on the busiest compute unit (one workgroup at a time), its ends
// (staging, epilogue) counted as one round of element columns; among equals the least work.
L1Plan l1_plan_of(const Grid& g, size_t elem_bytes, bool split) {
  L1Plan best{};
  int64_t cost = INT64_MAX;
  for (int ntz = (g.nz() + 62) / 63 > 2 ? (g.nz() + 62) / 63 : 1; ntz <= (g.nz() + 7) / 8; ++ntz) {
    L1Plan p{};
    p.split = split;
    p.zl = (g.nz() + ntz - 1) / ntz;
    p.ntz = (g.nz() + p.zl - 1) / p.zl;
    p.lpc = p.ntz == 1 ? g.ez : p.zl + 1;
    if (p.lpc > 64) continue;
    p.cpw = 64 / p.lpc;
    const int round = (split ? 4 : 16) * p.cpw;
    for (p.cx = 2; p.cx <= 12; ++p.cx)
      for (p.cy = 2; p.cy <= 12; ++p.cy) {
        if (l1_lds_bytes(p, elem_bytes) > kL1MaxLds) continue;
        p.ntx = (g.nx() + p.cx - 2) / (p.cx - 1);
        p.nty = (g.ny() + p.cy - 2) / (p.cy - 1);
        const int64_t tiles = (int64_t)p.ntx * p.nty * p.ntz;
        const int64_t rounds = (p.cx * p.cy + round - 1) / round;
        const int64_t c = ((tiles + 255) / 256 * (rounds + 1) << 20) + tiles * rounds;
        if (c < cost) {
          cost = c;
          best = p;
        }
      }
  }
  return best;
}

L1Plan l1_plan(const Grid& g, bool mixed) {
  return l1_plan_of(g, mixed ? sizeof(float) : sizeof(double), !mixed || g.n_nodes() < kL1SplitNodes);
}

inline int l1_at(int B, int c, int D, int d) { return ((B * 3 + c) * 8 + D) * 3 + d; }

// Mh = H M_0 H / 64, M_0 = W_0^T K0 W_0 in corner-bit order, [M][c][N][d]
std::vector<double> level1_mh(const double* K0_host) {
  double Kb[8][3][8][3];
  for (int b = 0; b < 8; ++b)
    for (int b2 = 0; b2 < 8; ++b2)
      for (int c = 0; c < 3; ++c)
        for (int d = 0; d < 3; ++d) Kb[b][c][b2][d] = K0_host[(3 * l1_corner(b) + c) * 24 + 3 * l1_corner(b2) + d];
  double W[8][8];  // child 0: [child corner b][coarse corner B]
  for (int b = 0; b < 8; ++b)
    for (int B = 0; B < 8; ++B) {
      double w = 1.0;
      for (int d = 0; d < 3; ++d) {
        const int f = (b >> d) & 1, cpos = 2 * ((B >> d) & 1);
        w *= std::fmax(0.0, 1.0 - std::fabs((double)(f - cpos)) / 2.0);
      }
      W[b][B] = w;
    }
  std::vector<double> M0(8 * 3 * 8 * 3, 0.0), Mh(8 * 3 * 8 * 3, 0.0);
  for (int B = 0; B < 8; ++B)
    for (int c = 0; c < 3; ++c)
      for (int D = 0; D < 8; ++D)
        for (int d = 0; d < 3; ++d) {
          double v = 0.0;
          for (int b = 0; b < 8; ++b)
            for (int b2 = 0; b2 < 8; ++b2) v += W[b][B] * Kb[b][c][b2][d] * W[b2][D];
          M0[l1_at(B, c, D, d)] = v;
        }
  auto h = [](int m, int b) { return (__builtin_popcount(m & b) & 1) ? -1.0 : 1.0; };
  for (int M = 0; M < 8; ++M)
    for (int c = 0; c < 3; ++c)
      for (int N = 0; N < 8; ++N)
        for (int d = 0; d < 3; ++d) {
          double v = 0.0;
          for (int B = 0; B < 8; ++B)
            for (int D = 0; D < 8; ++D) v += h(M, B) * M0[l1_at(B, c, D, d)] * h(N, D);
          Mh[l1_at(M, c, N, d)] = v / 64.0;
        }
  return Mh;
}
}  // namespace

bool level1_terms_cover(const double* K0_host, double rtol) {
  const std::vector<double> Mh = level1_mh(K0_host);
  std::vector<char> kept(Mh.size(), 0);
  for (int t = 0; t < kL1Terms; ++t) kept[l1_at(kL1Term[t][1], kL1Term[t][0], kL1Term[t][3], kL1Term[t][2])] = 1;
  double mx = 0.0;
  for (double v : Mh) mx = std::fmax(mx, std::fabs(v));
  for (size_t i = 0; i < Mh.size(); ++i)
    if (!kept[i] && std::fabs(Mh[i]) > rtol * mx) return false;
  return true;
}

int Level1MF::init(const Grid& fine, const double* K0_host, bool mixed_, hipStream_t s) {
  g0 = fine;
  g1 = fine.coarse();
  mixed = mixed_;
  plan = l1_plan(g1, mixed);
  ET_REQUIRE(plan.cx > 0, "level-1 operator: no tile fits");
  const std::vector<double> Mh = level1_mh(K0_host);
  auto at = l1_at;
  std::vector<double> cd(kL1Terms);
  std::vector<float> cfl(kL1Terms);
  for (int t = 0; t < kL1Terms; ++t) {
    cd[t] = Mh[at(kL1Term[t][1], kL1Term[t][0], kL1Term[t][3], kL1Term[t][2])];
    cfl[t] = (float)cd[t];
  }
  const size_t ts = mixed ? sizeof(float) : sizeof(double);
  ET_CHECK_HIP(hipMalloc(&cf, kL1Terms * ts));
  ET_CHECK_HIP(hipMemcpy(cf, mixed ? (const void*)cfl.data() : (const void*)cd.data(), kL1Terms * ts,
                         hipMemcpyHostToDevice));
  const int64_t ne1 = g1.n_elem(), nn1 = g1.n_nodes();
  ET_CHECK_HIP(hipMalloc(&Eh, ne1 * 8 * ts));
  ET_CHECK_HIP(hipMalloc(&special, ne1));
  ET_CHECK_HIP(hipMalloc(&aidx, nn1 * sizeof(int)));
  ET_CHECK_HIP(hipMalloc(&alist, nn1 * sizeof(int)));
  ET_CHECK_HIP(hipMalloc(&acount, sizeof(int)));
  ET_CHECK_HIP(hipHostMalloc(&acount_h, sizeof(int)));
  (void)s;
  return ET_OK;
}

int Level1MF::setup(const double* E, const uint8_t* eflag, const double* S1, hipStream_t s) {
  const int64_t ne1 = g1.n_elem(), nn1 = g1.n_nodes();
  if (mixed)
    l1_eh_kernel<float><<<grid_for(ne1), kBlock, 0, s>>>(g0, g1, E, eflag, (float*)Eh, special);
  else
    l1_eh_kernel<double><<<grid_for(ne1), kBlock, 0, s>>>(g0, g1, E, eflag, (double*)Eh, special);
  ET_CHECK_LAUNCH();
  ET_CHECK_HIP(hipMemsetAsync(acount, 0, sizeof(int), s));
  l1_affected_kernel<<<grid_for(nn1), kBlock, 0, s>>>(g1, special, aidx, alist, acount);
  ET_CHECK_LAUNCH();
  ET_CHECK_HIP(hipMemcpyAsync(acount_h, acount, sizeof(int), hipMemcpyDeviceToHost, s));
  ET_CHECK_HIP(hipStreamSynchronize(s));
  n_aff = *acount_h;
  if (n_aff == 0) return ET_OK;
  if (n_aff > rows_cap) {
    if (rows) (void)hipFree(rows);
    rows = nullptr;
    rows_cap = 0;
    ET_CHECK_HIP(hipMalloc(&rows, (size_t)n_aff * 243 * (mixed ? sizeof(float) : sizeof(double))));
    rows_cap = n_aff;
  }
  const unsigned grid = grid_for((int64_t)n_aff * 27);
  if (mixed)
    l1_rows_kernel<float><<<grid, kBlock, 0, s>>>(g1, S1, alist, n_aff, (float*)rows);
  else
    l1_rows_kernel<double><<<grid, kBlock, 0, s>>>(g1, S1, alist, n_aff, (double*)rows);
  ET_CHECK_LAUNCH();
  return ET_OK;
}

namespace {
template <typename T, int MODE, bool SPLIT>
void l1_launch(const L1Args& A, size_t lds, int n_fix, hipStream_t s, const Level1MF& L, const T* x, const T* b,
               const T* Dinv, const double* omega, double wscale, const T* xadd, T* y) {
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&l1_tile_kernel<T, MODE, SPLIT>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)kL1MaxLds);
  (void)attr;
  l1_tile_kernel<T, MODE, SPLIT><<<n_fix + A.p.ntx * A.p.nty * A.p.ntz, SPLIT ? 768 : 1024, lds, s>>>(
      A, (const T*)L.cf, (const T*)L.Eh, L.aidx, L.alist, L.n_aff, n_fix, (const T*)L.rows, x, b, Dinv, omega, wscale,
      xadd, y);
}
}  // namespace

template <typename T>
int Level1MF::apply(int mode, const T* x, const T* b, const T* Dinv, const double* omega, double wscale,
                    const T* xadd, T* y, hipStream_t s) const {
  ET_REQUIRE((sizeof(T) == sizeof(float)) == mixed, "level-1 operator: precision mismatch");
  const int per = (plan.split ? 768 : 1024) / 32 * kL1FixNodes;
  const int n_fix = (n_aff + per - 1) / per;
  const L1Args A{g1, plan};
  const size_t lds = l1_lds_bytes(plan, sizeof(T));
#define ET_L1(M)                                                                          \
  do {                                                                                    \
    if constexpr (sizeof(T) == sizeof(float)) {                                           \
      if (!plan.split) {                                                                  \
        l1_launch<T, M, false>(A, lds, n_fix, s, *this, x, b, Dinv, omega, wscale, xadd, y); \
        break;                                                                            \
      }                                                                                   \
    }                                                                                     \
    l1_launch<T, M, true>(A, lds, n_fix, s, *this, x, b, Dinv, omega, wscale, xadd, y);   \
  } while (0)
  switch (mode) {
    case 0: ET_L1(0); break;
    case 1: ET_L1(1); break;
    case 2: ET_L1(2); break;
    default: ET_L1(3); break;
  }
#undef ET_L1
  ET_CHECK_LAUNCH();
  return ET_OK;
}
template int Level1MF::apply<float>(int, const float*, const float*, const float*, const double*, double,
                                    const float*, float*, hipStream_t) const;
template int Level1MF::apply<double>(int, const double*, const double*, const double*, const double*, double,
                                     const double*, double*, hipStream_t) const;

void Level1MF::release() {
  for (void* p : {cf, Eh, (void*)special, (void*)aidx, (void*)alist, (void*)acount, rows})
    if (p) (void)hipFree(p);
  if (acount_h) (void)hipHostFree(acount_h);
  cf = Eh = rows = nullptr;
  special = nullptr;
  aidx = alist = acount = acount_h = nullptr;
  n_aff = rows_cap = 0;
}

}  // namespace et
