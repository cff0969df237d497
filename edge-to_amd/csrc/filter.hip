// Linear-hat density filter on structured element grids: normaliser, forward
// (normalised weighted average over in-bounds neighbours), exact transpose, and
// the SIMP adjoint fused with the transpose.
//
// 3-D: a workgroup owns a tile of TY x 64 element columns (TY 8 or 4, a wavefront per row along
// z) and marches along x through a chunk of planes (4 to 32, as many as keep about two
// workgroups per compute unit busy).  Each step stages one element plane of the tile with its
// y/z halo into one of two LDS planes and adds it to the 2R + 1 outputs of its column that it
// reaches, which wait in registers: an LDS value is read once per thread and not once per tap.
// At 256 x 128 x 128, radius 1, that took the forward from 51 to 23 us (67 MB, 2.9 TB/s) and the
// transpose from 51 to 26 us (100 MB, 3.9 TB/s) against one LDS read per tap and weight; what is
// left is load and barrier latency at 4 wavefronts per SIMD (128 VGPRs at radius 2).
// 2-D: one workgroup stages one tile with its halo and sums it, 4 x 64 outputs on small grids, which
// are bound by launch and load latency (120 x 40: 9 us with a plane march, 4.4 us with one tile), and
// 32 x 64 on large ones.
// Every output is written once, with no atomics, and sums follow the offset table's order, so
// results are deterministic; the forward pass is bitwise the reference's (out-of-grid taps add
// an exact 0.0).  The forward's denominator depends only on the output's distances to the six
// faces clipped to the radius, so each 3-D workgroup tabulates it once per boundary class.
//
//   forward    y_i = (sum_k w_k x_{i+o_k}) / (sum_k [i+o_k in grid] w_k)
//              (apply_filter_{2D,3D}_kernel, core/_templated_cuda.cu:1526-1583)
//   transpose  y_j = sum_k w_k (v / N)_{j+o_k}, the offsets being symmetric; v / N is
//              formed once per staged value, not once per tap
//              (apply_filter_{2D,3D}_transpose_kernel, core/_templated_cuda.cu:1632-1679)
//   adjoint    y_j = sum_k w_k s_{j+o_k} / N_{j+o_k} with the SIMP sensitivity
//              s_e = p clip(xt_e, void, 1)^(p-1) (-u_e^T K0 u_e) computed while staging
//              (process_dk + SingleMaterial.__backward__ + the transpose of
//              CuTopOpt.solve_and_process, TopOpt/_cuda.py:293-300), in one kernel.
//
// In 3-D the element energy is evaluated in the corner Walsh-Hadamard basis,
// u^T K0 u = sum over the kept couplings of uh[M][c] G[M][c][d] uh[M^e_c^e_d][d]
// with uh = H u_e and G = H K0 H / 64 (about 140 flops instead of 1152).  The
// host picks that form only for element matrices with the brick's reflection
// structure (k0_structure); any other K0 takes the full product.
//
// The march needs a radius of at most kMaxR per axis and a table in ascending (dx, dy, dz) order
// with weights even in each of them (every table the meshes build up to rmin 3); any other table
// of that radius is summed tap by tap from a ring of LDS planes.  The 2-D tile takes any table with a
// radius of at most kR2.  Each workgroup checks that on the device, where the table is; wider
// tables are gathered from memory tap by tap (the adjoint then recomputes the neighbour's
// sensitivity per tap).
#include "common.hpp"
#include "op_tiled.hpp"
#include "stiffness.hpp"

namespace et {

constexpr int kMaxOff = 1024;
constexpr int kMaxR = 2;     // halo radius per axis of the 3-D march (rmin <= 3)
constexpr int kMaxTaps = 512;  // taps held in LDS (rmin up to about 4.9)
constexpr int kMaxCX = 32;   // x planes per workgroup, at most

template <int DIM>
__device__ __forceinline__ void elem_coords(const Grid& g, int64_t e, int& i, int& j, int& k) {
  if (DIM == 3) {
    i = (int)(e / ((int64_t)g.ey * g.ez));
    const int r = (int)(e % ((int64_t)g.ey * g.ez));
    j = r / g.ez;
    k = r % g.ez;
  } else {
    i = (int)(e / g.ey);
    j = (int)(e % g.ey);
    k = 0;
  }
}

// One thread per element (normaliser; fallback for wide stencils).
// MODE 0: normaliser, 1: forward, 2: transpose
template <int DIM, int MODE>
__global__ __launch_bounds__(256) void filter_kernel(const Grid g, int n_off,
                                                     const int32_t* __restrict__ off,
                                                     const double* __restrict__ w,
                                                     const double* __restrict__ norm,
                                                     const double* __restrict__ x,
                                                     double* __restrict__ y) {
  __shared__ int s_off[kMaxOff * DIM];
  __shared__ double s_w[kMaxOff];
  for (int t = threadIdx.x; t < n_off; t += blockDim.x) {
    for (int d = 0; d < DIM; ++d) s_off[t * DIM + d] = off[t * DIM + d];
    s_w[t] = w[t];
  }
  __syncthreads();
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= g.n_elem()) return;
  int i, j, k;
  elem_coords<DIM>(g, e, i, j, k);
  double sv = 0.0, sw = 0.0;
  for (int t = 0; t < n_off; ++t) {
    const int a = i + s_off[t * DIM], b = j + s_off[t * DIM + 1];
    const int c = DIM == 3 ? k + s_off[t * DIM + 2] : 0;
    bool ok = a >= 0 && a < g.ex && b >= 0 && b < g.ey;
    if (DIM == 3) ok = ok && c >= 0 && c < g.ez;
    if (!ok) continue;
    const int64_t q = DIM == 3 ? ((int64_t)a * g.ey + b) * g.ez + c : (int64_t)a * g.ey + b;
    if (MODE == 0) {
      sw += s_w[t];
    } else if (MODE == 1) {
      sv += s_w[t] * x[q];
      sw += s_w[t];
    } else {
      sv += (s_w[t] / norm[q]) * x[q];
    }
  }
  if (MODE == 0)
    y[e] = sw;
  else if (MODE == 1)
    y[e] = sw > 0.0 ? sv / sw : 0.0;
  else
    y[e] = sv;
}

// ------------------------------------------------------- stencil geometry ---

// element grid seen as (X, Y, Z) with index (x * Y + y) * Z + z
struct SGrid {
  int X, Y, Z;
};

__host__ inline SGrid sgrid(const Grid& g) {
  if (g.dim == 3) return SGrid{g.ex, g.ey, g.ez};
  return SGrid{g.ex, 1, g.ey};  // 2-D: (i, j) -> x = i, z = j
}

struct AdjArgs {
  const double* K0;
  const double* U;
  const double* xt;
  double penal, vmin;
  const double* norm;
};

// corner-bit order beta = bx + 2 by + 4 bz of the H8 corners
__device__ __forceinline__ int fcorner(int beta) { return h8_corner(beta & 1, (beta >> 1) & 1, beta >> 2); }

// -u_e^T K0 u_e of element (x, y, z) of a 3-D grid: transformed basis or full product
template <bool WHT>
__device__ __forceinline__ double elem_energy3(const Grid& g, int ex, int ey, int ez, const double* __restrict__ U,
                                               const double* K0, const double* sG) {
  const int nx = g.nx(), nz = g.nz();
  // node index of corner-bit beta = bx + 2 by + 4 bz
  const int64_t m0 = ((int64_t)ey * nx + ex) * nz + ez;
  const int64_t sx = nz, sy = (int64_t)nx * nz;
  double e = 0.0;
  if (WHT) {
    // one displacement component at a time: its 8 corner values, then their
    // 8-point Walsh-Hadamard transform (the memory clobber keeps the three
    // components' loads from being scheduled together: fewer live registers)
    double uh[3][8];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      double a[8];
#pragma unroll
      for (int b = 0; b < 8; ++b) a[b] = U[(m0 + (b & 1) * sx + ((b >> 1) & 1) * sy + (b >> 2)) * 3 + c];
#pragma unroll
      for (int h = 1; h < 8; h <<= 1)
#pragma unroll
        for (int b = 0; b < 8; ++b)
          if (!(b & h)) {
            const double p = a[b], q = a[b | h];
            a[b] = p + q;
            a[b | h] = p - q;
          }
#pragma unroll
      for (int M = 0; M < 8; ++M) uh[c][M] = a[M];
      asm volatile("" ::: "memory");
    }
#pragma unroll
    for (int M = 1; M < 8; ++M) {
      // the coefficients of one M at a time (a clobber per M bounds the loads in flight)
      asm volatile("" ::: "memory");
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int d = 0; d < 3; ++d)
          if (wht_nz(M, c, d)) e = fma(uh[c][M] * sG[(M - 1) * 9 + c * 3 + d], uh[d][M ^ (1 << c) ^ (1 << d)], e);
    }
  } else {
    // full product in the element's own DOF order
    double u[8][3];  // corner-bit order
#pragma unroll
    for (int beta = 0; beta < 8; ++beta)
#pragma unroll
      for (int c = 0; c < 3; ++c)
        u[beta][c] = U[(m0 + (beta & 1) * sx + ((beta >> 1) & 1) * sy + (beta >> 2)) * 3 + c];
#pragma unroll 1
    for (int p = 0; p < 24; ++p) {
      const int ap = p / 3, cp = p % 3;
      double v = 0.0;
#pragma unroll
      for (int q = 0; q < 24; ++q) {
        const int aq = q / 3, cq = q % 3;
        v += K0[p * 24 + q] * u[hx(aq) + 2 * hy(aq) + 4 * hz(aq)][cq];
      }
      // u[corner of p][component of p], selected without dynamic register indexing
      double up = 0.0;
#pragma unroll
      for (int b = 0; b < 8; ++b)
#pragma unroll
        for (int c = 0; c < 3; ++c)
          up = (b == hx(ap) + 2 * hy(ap) + 4 * hz(ap) && c == cp) ? u[b][c] : up;
      e += v * up;
    }
  }
  return -e;
}

__device__ inline double elem_energy2(const Grid& g, int ex, int ey, const double* __restrict__ U,
                                      const double* K0) {
  const int nx = g.nx();
  double ue[8];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int64_t m = (int64_t)(ey + qy(b)) * nx + ex + qx(b);
    ue[2 * b] = U[m * 2];
    ue[2 * b + 1] = U[m * 2 + 1];
  }
  double e = 0.0;
#pragma unroll
  for (int p = 0; p < 8; ++p) {
    double v = 0.0;
#pragma unroll
    for (int q = 0; q < 8; ++q) v += K0[p * 8 + q] * ue[q];
    e += v * ue[p];
  }
  return -e;
}

// out of line: pow's many registers stay out of the stencil loops
__device__ __attribute__((noinline)) double simp_pow(double x, double e) { return pow(x, e); }

// SIMP factor p x^(p-1); for the usual p = 3 (GP false, chosen on the host) x^2 = x * x,
// which is pow(x, 2) correctly rounded, and pow's registers stay out of the kernel
template <bool GP>
__device__ __forceinline__ double simp_factor(double x, double penal) {
  return GP ? penal * simp_pow(x, penal - 1.0) : penal * (x * x);
}

// value staged for element e at (xs, gy, gz) of the stencil grid:
// MODE 1 x_e, 2 v_e / N_e, 3 s_e / N_e (SIMP adjoint; EN 1 transformed-basis energy, 2 full)
template <int MODE, int DIM, int EN>
__device__ __forceinline__ double stencil_value(const Grid& g, const SGrid& sg, int xs, int gy, int gz,
                                                const double* __restrict__ x, const AdjArgs& adj,
                                                const double* sK, const double* sG) {
  const int64_t e = ((int64_t)xs * sg.Y + gy) * sg.Z + gz;
  if (MODE == 1) return x[e];
  if (MODE == 2) return x[e] / adj.norm[e];
  const double xe = fmin(fmax(adj.xt[e], adj.vmin), 1.0);
  const double en = DIM == 3 ? elem_energy3<(EN & 3) == 1>(g, xs, gy, gz, adj.U, sK, sG)
                             : elem_energy2(g, xs, gz, adj.U, sK);
  return simp_factor<(EN & 4) != 0>(xe, adj.penal) * en / adj.norm[e];
}

// The offset table in LDS, with what the kernels derive from it.
struct TapTable {
  double w[kMaxTaps];
  int d[kMaxTaps];      // dx, dy, dz + 8, 5 bits each (radii up to 7)
  double cube[125];     // weight at each position of the (2 rc + 1)^3 cube, 0 where there is no tap
  double bw[125];       // weight sum of every boundary class (forward)
  int r[3];             // radius per axis
  int odd;              // the march does not apply: order, duplicates or asymmetric weights
};

// One block-wide pass over the table.  Returns with the radii, and in 3-D with the cube of
// weights and `odd` set, behind a barrier.
template <int DIM, int NT>
__device__ __forceinline__ void load_taps(TapTable& T, int n_off, const int32_t* __restrict__ off,
                                          const double* __restrict__ w) {
  const int tid = threadIdx.x;
  if (tid < 3) T.r[tid] = 0;
  if (tid == 3) T.odd = 0;
  if (DIM == 3)
    for (int t = tid; t < 125; t += NT) T.cube[t] = 0.0;
  __syncthreads();
  for (int t = tid; t < n_off; t += NT) {
    const int dx = off[t * DIM];
    const int dy = DIM == 3 ? off[t * 3 + 1] : 0;
    const int dz = DIM == 3 ? off[t * 3 + 2] : off[t * 2 + 1];
    T.w[t] = w[t];
    T.d[t] = ((dx + 8) << 10) | ((dy + 8) << 5) | (dz + 8);
    if (dx != 0) atomicMax(&T.r[0], abs(dx));
    if (dy != 0) atomicMax(&T.r[1], abs(dy));
    if (dz != 0) atomicMax(&T.r[2], abs(dz));
  }
  __syncthreads();
  if (DIM != 3) return;
  const int rm = max(T.r[0], max(T.r[1], T.r[2]));
  if (rm > kMaxR) return;
  const int rc = max(rm, 1), wc = 2 * rc + 1;
  for (int t = tid; t < n_off; t += NT) {
    const int d = T.d[t];
    T.cube[(((d >> 10) - 8 + rc) * wc + ((d >> 5) & 31) - 8 + rc) * wc + (d & 31) - 8 + rc] = T.w[t];
    if (t > 0 && T.d[t - 1] >= d) T.odd = 1;
  }
  __syncthreads();
  for (int t = tid; t < wc * wc * wc; t += NT) {
    const int iz = t % wc, iy = (t / wc) % wc, ix = t / (wc * wc);
    const int m = (max(ix, 2 * rc - ix) * wc + max(iy, 2 * rc - iy)) * wc + max(iz, 2 * rc - iz);
    if (T.cube[t] != T.cube[m]) T.odd = 1;
  }
  __syncthreads();
}

// Boundary classes of one axis: an output's in-grid taps depend only on its distances to the two
// ends clipped to the radius.  S >= 2R + 1 positions fall into 2R + 1 classes, fewer into S.
__device__ __forceinline__ int axis_class(int o, int S, int R) {
  if (S <= 2 * R + 1) return o;
  return o < R ? o : (o > S - 1 - R ? 2 * R - (S - 1 - o) : R);
}
// (distance to the low end, distance to the high end), clipped, of class c
__device__ __forceinline__ void class_reach(int c, int S, int R, int& lo, int& hi) {
  const int o = S <= 2 * R + 1 ? c : (c <= R ? c : S - 1 - (2 * R - c));
  lo = min(o, R);
  hi = min(S - 1 - o, R);
}

// the value in a scalar register (every lane holds the same)
__device__ __forceinline__ double scalar_of(double v) {
  const int2 b = __builtin_bit_cast(int2, v);
  return __builtin_bit_cast(double, int2{__builtin_amdgcn_readfirstlane(b.x), __builtin_amdgcn_readfirstlane(b.y)});
}

// Weights by (|dx|, |dy|, |dz|) in scalar registers.
template <int R>
struct ClassWeights {
  static constexpr int W = R + 1;
  double w[W * W * W];
  __device__ __forceinline__ void load(const TapTable& T) {
    constexpr int C = 2 * R + 1;
#pragma unroll
    for (int k = 0; k < W * W * W; ++k)
      w[k] = scalar_of(T.cube[((R + k / (W * W)) * C + R + (k / W) % W) * C + R + k % W]);
  }
};

// Adds plane xs to the outputs xs - R .. xs + R held in a[0 .. 2R] (dx = R .. -R), the in-plane taps in
// ascending (dy, dz): together with the march along x every output sums its taps in the offset
// table's ascending order.  Each value is read from LDS once for its 2R + 1 outputs.  Cube positions
// without a tap add an exact zero while the values are finite; an output that is not finite is
// recomputed from the table's own taps (a zero weight times an infinity must not count).
template <int R, int PZ, bool ROWS = false>
__device__ __forceinline__ void add_plane(const double* me, const ClassWeights<R>& cw, double (&a)[2 * R + 1]) {
  constexpr int C = 2 * R + 1, W = R + 1;
#pragma unroll
  for (int iy = 0; iy < C; ++iy) {
    if (ROWS) asm volatile("" ::: "memory");  // one row's values in registers at a time
    const int ay = iy < R ? R - iy : iy - R;
#pragma unroll
    for (int iz = 0; iz < C; ++iz) {
      const int az = iz < R ? R - iz : iz - R;
      const double v = me[(iy - R) * PZ + iz - R];
#pragma unroll
      for (int j = 0; j < C; ++j) {
        const int ax = j < R ? R - j : j - R;
        a[j] = fma(cw.w[(ax * W + ay) * W + az], v, a[j]);
      }
    }
  }
}

// Taps beyond the LDS planes (radius above kMaxR): gathers from memory, the adjoint recomputing each
// tap's value.
template <int MODE, int DIM, int EN>
__device__ __forceinline__ void wide_taps(const Grid& g, const SGrid& sg, int x0, int x1, int oy, int oz, int n_off,
                                          const int32_t* __restrict__ off, const TapTable& T,
                                          const double* __restrict__ x, const AdjArgs& adj, const double* sK,
                                          const double* sG, double* __restrict__ y) {
#pragma unroll 1
  for (int xo = x0; xo < x1; ++xo) {
    double sv = 0.0, sw = 0.0;
#pragma unroll 1
    for (int t = 0; t < n_off; ++t) {
      const int dx = off[t * DIM];
      const int dy = DIM == 3 ? off[t * 3 + 1] : 0;
      const int dz = DIM == 3 ? off[t * 3 + 2] : off[t * 2 + 1];
      const int a = xo + dx, b = oy + dy, c = oz + dz;
      if (a < 0 || a >= sg.X || b < 0 || b >= sg.Y || c < 0 || c >= sg.Z) continue;
      if (MODE == 3) asm volatile("" ::: "memory");
      sv = fma(T.w[t], stencil_value<MODE, DIM, EN>(g, sg, a, b, c, x, adj, sK, sG), sv);
      sw += T.w[t];
    }
    const int64_t e = ((int64_t)xo * sg.Y + oy) * sg.Z + oz;
    y[e] = MODE == 1 ? (sw > 0.0 ? sv / sw : 0.0) : sv;
  }
}

// Any other table of radius R <= kMaxR (another order, duplicates, uneven weights), summed in the
// table's order: the planes an output reaches and the next one wait in a ring of kRing LDS planes, and
// a tap is one LDS read at an offset tabulated for each position of the ring (phase: the slot of the
// newest plane, the output's plus R).  128 x 64 x 64, 81 taps shuffled: forward 33 us, transpose 23,
// adjoint 37, against 75, 105 and 1480 gathered from memory, and 27, 17 and 33 for the ascending table.
constexpr int kRing = 2 * kMaxR + 2;

template <int R, int PZ, int PL, int NT>
__device__ __forceinline__ void load_phases(unsigned short (*phase)[kMaxTaps], const TapTable& T, int n_off) {
  for (int t = threadIdx.x; t < n_off; t += NT) {
    const int d = T.d[t];
    const int dx = (d >> 10) - 8, dy = ((d >> 5) & 31) - 8, dz = (d & 31) - 8;
    for (int p = 0; p < kRing; ++p) {
      const int slot = p - R + dx;  // >= p - 2R
      phase[p][t] = (unsigned short)((slot < 0 ? slot + kRing : slot) * PL + (dy + R) * PZ + dz + R);
    }
  }
  __syncthreads();
}
__device__ __forceinline__ double sum_taps(const double* me, const unsigned short* off, const double* w, int n_off) {
  double sv = 0.0;
  int t = 0;
#pragma unroll 1
  for (; t + 4 <= n_off; t += 4) {
    double wv[4], v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      wv[k] = w[t + k];
      v[k] = me[off[t + k]];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) sv = fma(wv[k], v[k], sv);
  }
  for (; t < n_off; ++t) sv = fma(w[t], me[off[t]], sv);
  return sv;
}

// ------------------------------------------------- 3-D forward, transpose ---

// Marches planes x0 - R .. x1 - 1 + R through two LDS planes.  A plane's loads are issued PD steps
// before it is stored, unconditionally (slots outside the grid read a clamped element and are
// zeroed at the store), so no wait but the store's own touches them.  Returns whether all of the
// thread's outputs are finite.  ODD: a table that add_plane does not take (always true: only the table's
// own taps are summed).
template <int MODE, int R, int TY, bool ODD>
__device__ __forceinline__ bool march(const SGrid& sg, int x0, int x1, int y0, int z0, int n_off, const TapTable& T,
                                      unsigned short (*phase)[kMaxTaps], double* planes,
                                      const double* __restrict__ x, const double* __restrict__ norm,
                                      double* __restrict__ y) {
  constexpr int NT = 64 * TY, PY = TY + 2 * R, PZ = 64 + 2 * R, PL = PY * PZ;
  constexpr int KP = (PL + NT - 1) / NT, PD = 4;
  const int tid = threadIdx.x, ty = tid >> 6, tz = tid & 63;
  const int oy = y0 + ty, oz = z0 + tz;
  const bool mine = oy < sg.Y && oz < sg.Z;
  ClassWeights<R> cw;
  if (ODD)
    load_phases<R, PZ, PL, NT>(phase, T, n_off);
  else
    cw.load(T);
  int qe[KP];  // element of the slot within a plane, -1 outside the grid
#pragma unroll
  for (int q = 0; q < KP; ++q) {
    const int t = tid + NT * q;
    const int gy = y0 - R + t / PZ, gz = z0 - R + t % PZ;
    qe[q] = t < PL && gy >= 0 && gy < sg.Y && gz >= 0 && gz < sg.Z ? gy * sg.Z + gz : -1;
  }
  const int YZ = sg.Y * sg.Z;
  double pre[PD][KP], prn[MODE == 2 ? PD : 1][KP];
  auto fetch = [&](double (&r)[KP], double (&rn)[KP], int xs) {
    const int base = min(max(xs, 0), sg.X - 1) * YZ;
#pragma unroll
    for (int q = 0; q < KP; ++q) {
      const int e = base + max(qe[q], 0);
      r[q] = x[e];
      if (MODE == 2) rn[q] = norm[e];
    }
  };
  int ph = 0;  // ODD: ring slot of plane xs
  auto put = [&](const double (&r)[KP], const double (&rn)[KP], int xs) {
    double* pl = planes + (ODD ? ph : xs & 1) * PL;
    const bool xin = xs >= 0 && xs < sg.X;
#pragma unroll
    for (int q = 0; q < KP; ++q) {
      const double v = MODE == 2 ? r[q] / rn[q] : r[q];
      if ((q + 1) * NT <= PL || tid + NT * q < PL) pl[tid + NT * q] = xin && qe[q] >= 0 ? v : 0.0;
    }
  };
  double a[2 * R + 1];
#pragma unroll
  for (int j = 0; j <= 2 * R; ++j) a[j] = 0.0;
  const int ncy = min(sg.Y, 2 * R + 1), ncz = min(sg.Z, 2 * R + 1);
  const int cyz = MODE == 1 && mine ? axis_class(oy, sg.Y, R) * ncz + axis_class(oz, sg.Z, R) : 0;
  bool fine = true;
  auto step = [&](int xs) {
    if (!ODD) add_plane<R, PZ>(planes + (xs & 1) * PL + (ty + R) * PZ + tz + R, cw, a);
    const int xo = xs - R;
    if (xo >= x0 && mine) {
      double out = ODD ? sum_taps(planes + ty * PZ + tz, phase[ph], T.w, n_off) : a[0];
      if (MODE == 1) {
        const double sw = T.bw[axis_class(xo, sg.X, R) * (ncy * ncz) + cyz];
        out = sw > 0.0 ? out / sw : 0.0;
      }
      y[xo * YZ + oy * sg.Z + oz] = out;
      fine = fine && isfinite(out);
    }
#pragma unroll
    for (int j = 0; j < 2 * R; ++j) a[j] = a[j + 1];
    a[2 * R] = 0.0;
  };
  const int xe = x1 + R;  // one past the last plane
#pragma unroll
  for (int k = 0; k < PD; ++k) {
    fetch(pre[k], prn[MODE == 2 ? k : 0], x0 - R + k);
    asm volatile("" ::: "memory");  // in plane order: the first store waits for its own plane's loads only
  }
  // groups of PD steps whose loads and stores have no conditions: every path issues the same ones
  for (int xb = x0 - R; xb < xe; xb += PD) {
#pragma unroll
    for (int k = 0; k < PD; ++k) {
      put(pre[k], prn[MODE == 2 ? k : 0], xb + k);
      __syncthreads();
      fetch(pre[k], prn[MODE == 2 ? k : 0], xb + k + PD);
      if (xb + k < xe) step(xb + k);
      ph = ph + 1 < kRing ? ph + 1 : 0;
    }
  }
  return ODD || fine;
}

// bw of every boundary class: the sum of the in-grid taps in table order, as the reference's loop adds
// them.  Visible behind the next barrier.
template <int NT>
__device__ __forceinline__ void class_sums(TapTable& T, const SGrid& sg, int rc, int n_off) {
  const int tid = threadIdx.x;
  const int nx = min(sg.X, 2 * rc + 1), ny = min(sg.Y, 2 * rc + 1), nz = min(sg.Z, 2 * rc + 1);
  for (int c = tid; c < nx * ny * nz; c += NT) {
    int lx, hx, ly, hy, lz, hz;
    class_reach(c / (ny * nz), sg.X, rc, lx, hx);
    class_reach((c / nz) % ny, sg.Y, rc, ly, hy);
    class_reach(c % nz, sg.Z, rc, lz, hz);
    double ws = 0.0;
    for (int t = 0; t < n_off; ++t) {
      const int d = T.d[t];
      const int dx = (d >> 10) - 8, dy = ((d >> 5) & 31) - 8, dz = (d & 31) - 8;
      ws += (dx >= -lx && dx <= hx && dy >= -ly && dy <= hy && dz >= -lz && dz <= hz) ? T.w[t] : 0.0;
    }
    T.bw[c] = ws;
  }
}

// MODE 1: forward, 2: transpose (values v / N).  Tile: TY x 64 outputs per plane, one per thread.
template <int MODE, int TY>
__global__ __launch_bounds__(64 * TY) __attribute__((amdgpu_waves_per_eu(4))) void march_kernel(
    const Grid g, const SGrid sg, int cx, int n_off, const int32_t* __restrict__ off, const double* __restrict__ w,
    const double* __restrict__ x, const double* __restrict__ norm, double* __restrict__ y) {
  constexpr int NT = 64 * TY;
  __shared__ TapTable T;
  __shared__ unsigned short phase[kRing][kMaxTaps];
  __shared__ double planes[kRing * (TY + 2 * kMaxR) * (64 + 2 * kMaxR)];  // two in use but for odd tables
  const int tid = threadIdx.x;
  load_taps<3, NT>(T, n_off, off, w);
  const int rm = max(T.r[0], max(T.r[1], T.r[2])), rc = max(rm, 1);
  const int y0 = blockIdx.x * TY, z0 = blockIdx.y * 64;
  const int x0 = blockIdx.z * cx, x1 = min(x0 + cx, sg.X);
  bool fine = false;
#define ET_MARCH(R, ODD) march<MODE, R, TY, ODD>(sg, x0, x1, y0, z0, n_off, T, phase, planes, x, norm, y)
  if (rm <= kMaxR && !T.odd) {
    if (MODE == 1) class_sums<NT>(T, sg, rc, n_off);
    fine = rc == 1 ? ET_MARCH(1, false) : ET_MARCH(2, false);
  } else if (rm <= kMaxR) {
    if (MODE == 1) class_sums<NT>(T, sg, rc, n_off);
    fine = rc == 1 ? ET_MARCH(1, true) : ET_MARCH(2, true);
  }
#undef ET_MARCH
  const int oy = y0 + (tid >> 6), oz = z0 + (tid & 63);
  if (!fine && oy < sg.Y && oz < sg.Z) {
    AdjArgs adj{};
    adj.norm = norm;
    wide_taps<MODE, 3, 0>(g, sg, x0, x1, oy, oz, n_off, off, T, x, adj, nullptr, nullptr, y);
  }
}

// ------------------------------------------------------- 3-D SIMP adjoint ---

// Energy coefficients of the transformed basis, G[M][c][c] at (M - 1) * 3 + c, then for each pair
// c < d (third axis t) the four couplings uh_c[M] uh_d[M ^ e_c ^ e_d], M in {e_c, e_d, e_c + e_t,
// e_d + e_t}, with both of K0's entries for them added up.
constexpr int kEnDiag = 21, kEnCoef = 33;
__host__ __device__ constexpr int en_pair_c(int p) { return p == 2 ? 1 : 0; }
__host__ __device__ constexpr int en_pair_d(int p) { return p == 0 ? 1 : 2; }
__host__ __device__ constexpr int en_pair_M(int p, int m) {
  const int c = 1 << en_pair_c(p), d = 1 << en_pair_d(p), t = 7 ^ c ^ d;
  return (m & 1 ? d : c) | (m & 2 ? t : 0);
}

// 4-point transform over (y, z) of one x face of an element: corner (by, bz) at 2 bz + by
struct Face {
  double f[3][4];
};
__device__ __forceinline__ void load_face(Face& f, const double* __restrict__ U, int m, int sy) {
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int c = 0; c < 3; ++c) f.f[c][b] = U[(m + (b & 1) * sy + (b >> 1)) * 3 + c];
}
__device__ __forceinline__ void face_transform(Face& f) {
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const double p = f.f[c][0] + f.f[c][1], q = f.f[c][0] - f.f[c][1];
    const double r = f.f[c][2] + f.f[c][3], s = f.f[c][2] - f.f[c][3];
    f.f[c][0] = p + r;
    f.f[c][1] = q + s;
    f.f[c][2] = p - r;
    f.f[c][3] = q - s;
  }
}
// -u^T K0 u from the transformed faces at x (lo) and x + 1 (hi)
__device__ __forceinline__ double face_energy(const Face& lo, const Face& hi, const double* sC) {
  double u[3][8];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      u[c][2 * k] = lo.f[c][k] + hi.f[c][k];
      u[c][2 * k + 1] = lo.f[c][k] - hi.f[c][k];
    }
  double e = 0.0;
#pragma unroll
  for (int M = 1; M < 8; ++M)
#pragma unroll
    for (int c = 0; c < 3; ++c) e = fma(sC[(M - 1) * 3 + c], u[c][M] * u[c][M], e);
#pragma unroll
  for (int p = 0; p < 3; ++p)
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      constexpr int kPair[3][2] = {{0, 1}, {0, 2}, {1, 2}};
      const int c = kPair[p][0], d = kPair[p][1], M = en_pair_M(p, m);
      e = fma(sC[kEnDiag + 4 * p + m], u[c][M] * u[d][M ^ (1 << c) ^ (1 << d)], e);
    }
  return -e;
}

// One staged value per thread and plane, s_e / N_e (about 120 FP64 operations: VALU bound, 34 to 21 us
// at 128 x 64 x 64 against 24 gathered displacements and 45 couplings per value).  In the transformed basis (EN & 3 == 1) a thread
// keeps its element column's x + 1 face for the next plane, so each node column is read once per
// plane; any other K0 takes the full product.
template <int EN, int R, int TY, bool ODD, int NT>
__device__ __forceinline__ bool march_adjoint(const Grid& g, const SGrid& sg, int x0, int x1, int y0, int z0,
                                              int n_off, const TapTable& T, unsigned short (*phase)[kMaxTaps],
                                              double* planes, const AdjArgs& adj, const double* sK, const double* sC,
                                              double* __restrict__ y) {
  constexpr int PY = TY + 2 * R, PZ = 64 + 2 * R, PL = PY * PZ;
  constexpr bool WHT = (EN & 3) == 1;
  const int tid = threadIdx.x, ty = tid >> 6, tz = tid & 63;
  const int oy = y0 + ty, oz = z0 + tz;
  const bool mine = ty < TY && oy < sg.Y && oz < sg.Z;
  const int gy = y0 - R + tid / PZ, gz = z0 - R + tid % PZ;
  const bool slot = tid < PL, in = slot && gy >= 0 && gy < sg.Y && gz >= 0 && gz < sg.Z;
  const int cy = min(max(gy, 0), sg.Y - 1), cz = min(max(gz, 0), sg.Z - 1);
  const int YZ = sg.Y * sg.Z, nz = g.nz(), sy = g.nx() * nz;
  const int q = cy * sg.Z + cz, m = cy * sy + cz;  // this slot's element in plane 0 and its first node
  ClassWeights<R> cw;
  if (ODD)
    load_phases<R, PZ, PL, NT>(phase, T, n_off);
  else
    cw.load(T);
  Face lo, hi;
  double xv = 0.0, nv = 1.0;
  // operands of plane xs: the face at xs + 1, the density and N (clamped to the grid)
  auto fetch = [&](int xs) {
    const int xc = min(max(xs, 0), sg.X - 1);
    if (WHT) load_face(hi, adj.U, m + (xc + 1) * nz, sy);
    xv = adj.xt[xc * YZ + q];
    nv = adj.norm[xc * YZ + q];
  };
  double a[2 * R + 1];
#pragma unroll
  for (int j = 0; j <= 2 * R; ++j) a[j] = 0.0;
  if (WHT) {
    load_face(lo, adj.U, m + min(max(x0 - R, 0), sg.X - 1) * nz, sy);
    face_transform(lo);
  }
  fetch(x0 - R);
  bool fine = true;
  int ph = 0;  // ODD: ring slot of plane xs
  for (int xs = x0 - R; xs < x1 + R; ++xs) {
    const bool xin = xs >= 0 && xs < sg.X;
    double v = 0.0;
    if (WHT) {
      if (xin) {
        face_transform(hi);
        v = face_energy(lo, hi, sC);
        lo = hi;
      }
    } else if (xin && in) {
      v = elem_energy3<false>(g, xs, gy, gz, adj.U, sK, nullptr);
    }
    const double xe = fmin(fmax(xv, adj.vmin), 1.0);
    v = simp_factor<(EN & 4) != 0>(xe, adj.penal) * v / nv;
    if (slot) planes[(ODD ? ph : xs & 1) * PL + tid] = xin && in ? v : 0.0;
    fetch(xs + 1);
    __syncthreads();
    if (ODD) {
      if (mine && xs - R >= x0)
        y[(xs - R) * YZ + oy * sg.Z + oz] = sum_taps(planes + ty * PZ + tz, phase[ph], T.w, n_off);
      ph = ph + 1 < kRing ? ph + 1 : 0;
    } else if (mine) {
      add_plane<R, PZ, (R > 1)>(planes + (xs & 1) * PL + (ty + R) * PZ + tz + R, cw, a);
      if (xs - R >= x0) {
        y[(xs - R) * YZ + oy * sg.Z + oz] = a[0];
        fine = fine && isfinite(a[0]);
      }
#pragma unroll
      for (int j = 0; j < 2 * R; ++j) a[j] = a[j + 1];
      a[2 * R] = 0.0;
    }
  }
  return ODD || fine;
}

// threads of the adjoint's workgroup: one staged slot each at the largest radius, whole wavefronts
__host__ __device__ constexpr int adjoint_threads(int ty) {
  return ((ty + 2 * kMaxR) * (64 + 2 * kMaxR) + 63) / 64 * 64;
}

// EN 1: the element energy in the transformed basis (element matrices with the brick's reflection
// structure, chosen on the host), 2: the full product; EN + 4: a penalty other than 3.
template <int EN, int TY>
__global__ __launch_bounds__(adjoint_threads(TY)) void adjoint_kernel(
    const Grid g, const SGrid sg, int cx, int n_off, const int32_t* __restrict__ off, const double* __restrict__ w,
    const AdjArgs adj, double* __restrict__ y) {
  constexpr int NT = adjoint_threads(TY);
  __shared__ TapTable T;
  __shared__ unsigned short phase[kRing][kMaxTaps];
  __shared__ double planes[kRing * (TY + 2 * kMaxR) * (64 + 2 * kMaxR)];  // two in use but for odd tables
  __shared__ double sK[576];
  __shared__ double sC[kEnCoef];
  __shared__ double sG[63];
  const int tid = threadIdx.x;
  for (int t = tid; t < 576; t += NT) sK[t] = adj.K0[t];
  load_taps<3, NT>(T, n_off, off, w);  // its barriers also cover sK
  if ((EN & 3) == 1) {
    if (tid < 63) {
      // kept couplings of G = H K0 H / 64
      const int M = 1 + tid / 9, c = (tid / 3) % 3, d = tid % 3;
      const int Mp = M ^ (1 << c) ^ (1 << d);
      double sum = 0.0;
      for (int bb = 0; bb < 8; ++bb)
        for (int bp = 0; bp < 8; ++bp) {
          const double k = sK[(3 * fcorner(bb) + c) * 24 + 3 * fcorner(bp) + d];
          sum += ((__builtin_popcount(M & bb) ^ __builtin_popcount(Mp & bp)) & 1) ? -k : k;
        }
      sG[tid] = wht_nz(M, c, d) ? sum / 64.0 : 0.0;
    }
    __syncthreads();
    if (tid < kEnDiag) sC[tid] = sG[tid / 3 * 9 + tid % 3 * 4];
    if (tid >= kEnDiag && tid < kEnCoef) {
      const int p = (tid - kEnDiag) / 4, M = en_pair_M(p, (tid - kEnDiag) % 4);
      const int c = en_pair_c(p), d = en_pair_d(p), Mp = M ^ (1 << c) ^ (1 << d);
      sC[tid] = sG[(M - 1) * 9 + c * 3 + d] + sG[(Mp - 1) * 9 + d * 3 + c];
    }
    __syncthreads();
  }
  const int rm = max(T.r[0], max(T.r[1], T.r[2]));
  const int y0 = blockIdx.x * TY, z0 = blockIdx.y * 64;
  const int x0 = blockIdx.z * cx, x1 = min(x0 + cx, sg.X);
  bool fine = false;
#define ET_MARCH(R, ODD) march_adjoint<EN, R, TY, ODD, NT>(g, sg, x0, x1, y0, z0, n_off, T, phase, planes, adj, sK, sC, y)
  if (rm <= kMaxR && T.odd)
    fine = rm <= 1 ? ET_MARCH(1, true) : ET_MARCH(2, true);
  else if (rm <= kMaxR)
    fine = rm <= 1 ? ET_MARCH(1, false) : ET_MARCH(2, false);
#undef ET_MARCH
  const int oy = y0 + (tid >> 6), oz = z0 + (tid & 63);
  if (!fine && tid < 64 * TY && oy < sg.Y && oz < sg.Z)
    wide_taps<3, 3, EN>(g, sg, x0, x1, oy, oz, n_off, off, T, nullptr, adj, sK, sG, y);
}

// -------------------------------------------------------------------- 2-D ---

constexpr int kR2 = 4;                  // halo radius of the 2-D tile (rmin <= 5)
constexpr int kTZ2 = 64;                // outputs of a tile along z

// MODE 1: forward, 2: transpose, 3: SIMP adjoint, on one staged tile of TX x 64 outputs with its
// halo, NO outputs of a column per thread (launch_filter2 says which).
template <int MODE, int EN, int TX, int NO>
__global__ __launch_bounds__(64 * TX / NO) void filter2_kernel(const Grid g, const SGrid sg, int n_off,
                                                      const int32_t* __restrict__ off,
                                                      const double* __restrict__ w, const double* __restrict__ x,
                                                      const AdjArgs adj, double* __restrict__ y) {
  constexpr int PZ = kTZ2 + 2 * kR2, NT = 64 * TX / NO;
  __shared__ TapTable T;
  __shared__ double tile[(TX + 2 * kR2) * PZ];
  __shared__ double sK[MODE == 3 ? 64 : 1];
  const int tid = threadIdx.x;
  if (MODE == 3 && tid < 64) sK[tid] = adj.K0[tid];
  load_taps<2, NT>(T, n_off, off, w);
  const int rx = T.r[0], rz = T.r[2];
  const int ntz = (sg.Z + kTZ2 - 1) / kTZ2, bx = blockIdx.x / ntz;
  const int x0 = bx * TX, z0 = (blockIdx.x - bx * ntz) * kTZ2;
  const int ox = x0 + (tid >> 6) * NO, oz = z0 + (tid & 63);
  if (rx > kR2 || rz > kR2) {
    if (oz < sg.Z)
      wide_taps<MODE, 2, EN>(g, sg, ox, min(ox + NO, sg.X), 0, oz, n_off, off, T, x, adj, sK, nullptr, y);
    return;
  }
  const int pz = kTZ2 + 2 * rz, pn = (TX + 2 * rx) * pz;
  if constexpr (MODE == 3 || TX == 4) {
    for (int t = tid; t < pn; t += NT) {
      const int lx = t / pz, lz = t - lx * pz;
      const int gx = x0 - rx + lx, gz = z0 - rz + lz;
      double v = 0.0;
      if (gx >= 0 && gx < sg.X && gz >= 0 && gz < sg.Z)
        v = stencil_value<MODE, 2, EN>(g, sg, gx, 0, gz, x, adj, sK, nullptr);
      tile[lx * PZ + lz] = v;
    }
  } else {
    // four slots of a thread at a time, loads unconditional (clamped to the grid): all in flight together
    const int dl = NT / pz, dr = NT - dl * pz;  // NT slots further on
    int lx = tid / pz, lz = tid - lx * pz;
#pragma unroll 1
    for (int t0 = tid; t0 < pn; t0 += NT * 4) {
      double v[4], nv[4];
      int at[4];
      bool in[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int gx = x0 - rx + lx, gz = z0 - rz + lz;
        in[k] = gx >= 0 && gx < sg.X && gz >= 0 && gz < sg.Z;
        at[k] = t0 + NT * k < pn ? lx * PZ + lz : -1;
        const int64_t e = (int64_t)min(max(gx, 0), sg.X - 1) * sg.Z + min(max(gz, 0), sg.Z - 1);
        v[k] = x[e];
        nv[k] = MODE == 2 ? adj.norm[e] : 1.0;
        lx += dl;
        lz += dr;
        if (lz >= pz) {
          lz -= pz;
          ++lx;
        }
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (MODE == 2) v[k] /= nv[k];
        if (at[k] >= 0) tile[at[k]] = in[k] ? v[k] : 0.0;
      }
    }
  }
  __syncthreads();
  if (oz >= sg.Z) return;
  const double* me = tile + ((tid >> 6) * NO + rx) * PZ + (tid & 63) + rz;
  double sv[NO], sw[NO];
#pragma unroll
  for (int r = 0; r < NO; ++r) sv[r] = sw[r] = 0.0;
  if (MODE != 1 || (x0 >= rx && x0 + TX + rx <= sg.X && z0 >= rz && z0 + kTZ2 + rz <= sg.Z)) {
    // every tap of every output lies in the grid: one sum of weights
#pragma unroll 4
    for (int t = 0; t < n_off; ++t) {
      const int d = T.d[t];
      const double wk = T.w[t];
      const double* p = me + ((d >> 10) - 8) * PZ + (d & 31) - 8;
#pragma unroll
      for (int r = 0; r < NO; ++r) sv[r] = fma(wk, p[r * PZ], sv[r]);
      if (MODE == 1) sw[0] += wk;
    }
#pragma unroll
    for (int r = 1; r < NO; ++r) sw[r] = sw[0];
  } else {
#pragma unroll(TX == 4 ? 4 : 1)
    for (int t = 0; t < n_off; ++t) {
      const int d = T.d[t];
      const int dx = (d >> 10) - 8, dz = (d & 31) - 8;
      const double wk = T.w[t];
      const bool in = oz + dz >= 0 && oz + dz < sg.Z;
#pragma unroll
      for (int r = 0; r < NO; ++r) {
        sv[r] = fma(wk, me[(dx + r) * PZ + dz], sv[r]);
        sw[r] += in && ox + r + dx >= 0 && ox + r + dx < sg.X ? wk : 0.0;
      }
    }
  }
#pragma unroll
  for (int r = 0; r < NO; ++r)
    if (ox + r < sg.X)
      y[(int64_t)(ox + r) * sg.Z + oz] = MODE == 1 ? (sw[r] > 0.0 ? sv[r] / sw[r] : 0.0) : sv[r];
}

// ------------------------------------------------------------------- host ---

template <int MODE>
static int launch_gather(const Grid& g, int n_off, const int32_t* off, const double* w, const double* norm,
                         const double* x, double* y, hipStream_t s) {
  const unsigned grid = grid_for(g.n_elem());
  if (g.dim == 3)
    filter_kernel<3, MODE><<<grid, kBlock, 0, s>>>(g, n_off, off, w, norm, x, y);
  else
    filter_kernel<2, MODE><<<grid, kBlock, 0, s>>>(g, n_off, off, w, norm, x, y);
  ET_CHECK_LAUNCH();
  return ET_OK;
}

// rows per 3-D tile, 4 or 8
static int g_stencil_ty = 8;
void set_stencil_rows(int ty) { g_stencil_ty = ty; }
int get_stencil_rows() { return g_stencil_ty; }

// x planes per workgroup: the longest chunk that still gives about 512 workgroups (two per compute unit)
static int chunk_planes(const SGrid& sg, int ty) {
  const int64_t tiles = (int64_t)((sg.Y + ty - 1) / ty) * ((sg.Z + 63) / 64);
  int cx = kMaxCX;
  while (cx > 4 && tiles * ((sg.X + cx - 1) / cx) < 512) cx /= 2;
  return cx;
}

static dim3 march_grid(const SGrid& sg, int ty, int cx) {
  return dim3((sg.Y + ty - 1) / ty, (sg.Z + 63) / 64, (sg.X + cx - 1) / cx);
}

// 2-D tiles.  A small grid is bound by launch and load latency: 4 x 64 outputs, one per thread.  A large
// one pays for the halo (2.1 staged values per output at radius 2; 1.2 with 32 x 64) and for the
// table, which every workgroup reads and every tap decodes: 32 x 64 outputs, 4 of a column per thread.
// The adjoint, whose energies take 168 registers and more, gains more from fewer threads: 8.
// Strips of a few rows fill too little of a tall tile (us, 4 / 32 rows, 16 x 200 000: forward 30 / 33,
// transpose 29 / 23, adjoint 81 / 53; 3 x 1 M: 34 / 128, 28 / 81, 79 / 125).
// us, 4 / 32 rows (and a march of 256-wide rows), radius 1: forward 7.6 / 7.6 (10) at 1024 x 512, 12.1 /
// 9.5 (14) at 1024 x 1024, 72 / 42 (41) at 4096 x 2048 (134 MB, 3.2 TB/s); transpose 6.5 / 6.0 (9.6), 10.4 /
// 7.6 (14), 62 / 43 (44); adjoint 14 / 12 (23), 28 / 17 (37), 215 / 120 (237); radius 2: forward 12 / 12
// (17), 20 / 15 (24), 125 / 73 (74).
constexpr int64_t kTall2 = (int64_t)1 << 20;

template <int MODE, int EN>
static void launch_filter2(const Grid& g, const SGrid& sg, int n_off, const int32_t* off, const double* w,
                           const double* x, const AdjArgs& adj, double* y, hipStream_t s) {
  constexpr int TX = 32, NO = MODE == 3 ? 8 : 4;
  const bool tall = (int64_t)sg.X * sg.Z >= kTall2 && sg.X >= (MODE == 3 ? 8 : 24);
  const int tx = tall ? TX : 4;
  const unsigned grid = (unsigned)((sg.Z + kTZ2 - 1) / kTZ2) * (unsigned)((sg.X + tx - 1) / tx);
  if (tall)
    filter2_kernel<MODE, EN, TX, NO><<<grid, 64 * TX / NO, 0, s>>>(g, sg, n_off, off, w, x, adj, y);
  else
    filter2_kernel<MODE, EN, 4, 1><<<grid, 256, 0, s>>>(g, sg, n_off, off, w, x, adj, y);
}

template <int MODE>
static int launch_filter(const Grid& g, int n_off, const int32_t* off, const double* w, const double* norm,
                         const double* x, double* y, hipStream_t s) {
  const SGrid sg = sgrid(g);
  AdjArgs adj{};
  adj.norm = norm;
  const int ty = g_stencil_ty, cx = chunk_planes(sg, ty);
  if (g.dim == 2)
    launch_filter2<MODE, 0>(g, sg, n_off, off, w, x, adj, y, s);
  else if (ty == 4)
    march_kernel<MODE, 4><<<march_grid(sg, ty, cx), 256, 0, s>>>(g, sg, cx, n_off, off, w, x, norm, y);
  else
    march_kernel<MODE, 8><<<march_grid(sg, ty, cx), 512, 0, s>>>(g, sg, cx, n_off, off, w, x, norm, y);
  ET_CHECK_LAUNCH();
  return ET_OK;
}

template <int EN>
static int launch_adjoint(const Grid& g, int n_off, const int32_t* off, const double* w, const AdjArgs& adj,
                          double* y, hipStream_t s) {
  const SGrid sg = sgrid(g);
  const int ty = g_stencil_ty, cx = chunk_planes(sg, ty);
  if (g.dim == 2) {
    if constexpr ((EN & 3) == 2) launch_filter2<3, EN>(g, sg, n_off, off, w, nullptr, adj, y, s);  // no basis in 2-D
  } else if (ty == 4)
    adjoint_kernel<EN, 4><<<march_grid(sg, ty, cx), adjoint_threads(4), 0, s>>>(g, sg, cx, n_off, off, w, adj, y);
  else
    adjoint_kernel<EN, 8><<<march_grid(sg, ty, cx), adjoint_threads(8), 0, s>>>(g, sg, cx, n_off, off, w, adj, y);
  ET_CHECK_LAUNCH();
  return ET_OK;
}

int filter_normalizer(const Grid& g, int n_off, const int32_t* off, const double* w, double* norm,
                      hipStream_t s) {
  ET_REQUIRE(n_off > 0 && n_off <= kMaxOff, "filter offset count out of range (1..1024)");
  return launch_gather<0>(g, n_off, off, w, nullptr, nullptr, norm, s);
}

int filter_fwd(const Grid& g, int n_off, const int32_t* off, const double* w, const double* x,
               double* y, hipStream_t s) {
  ET_REQUIRE(n_off > 0 && n_off <= kMaxOff, "filter offset count out of range (1..1024)");
  if (n_off > kMaxTaps) return launch_gather<1>(g, n_off, off, w, nullptr, x, y, s);
  return launch_filter<1>(g, n_off, off, w, nullptr, x, y, s);
}

int filter_adj(const Grid& g, int n_off, const int32_t* off, const double* w, const double* norm,
               const double* v, double* y, hipStream_t s) {
  ET_REQUIRE(n_off > 0 && n_off <= kMaxOff, "filter offset count out of range (1..1024)");
  if (n_off > kMaxTaps) return launch_gather<2>(g, n_off, off, w, norm, v, y, s);
  return launch_filter<2>(g, n_off, off, w, norm, v, y, s);
}

int simp_adjoint(const Grid& g, const double* K0, const double* U, const double* xt, double penal, double vmin,
                 int n_off, const int32_t* off, const double* w, const double* norm, int k0_flags, double* y,
                 hipStream_t s) {
  ET_REQUIRE(n_off > 0 && n_off <= kMaxTaps, "simp adjoint: filter offset count out of range (1..512)");
  const AdjArgs a{K0, U, xt, penal, vmin, norm};
  const bool wht = g.dim == 3 && (k0_flags & K0S_WHT);
  if (penal == 3.0)
    return wht ? launch_adjoint<1>(g, n_off, off, w, a, y, s)
               : launch_adjoint<2>(g, n_off, off, w, a, y, s);
  return wht ? launch_adjoint<5>(g, n_off, off, w, a, y, s)
             : launch_adjoint<6>(g, n_off, off, w, a, y, s);
}

}  // namespace et
