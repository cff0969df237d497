// Fine-grid H8 operator on one-shot tiles, for grids too small to march (op_wht.hip): the modes of
// op_tiled.hpp with the element product in the transformed basis (45 coefficients, element
// matrices with the brick's reflection structure) or with any 24 x 24 K0.
//
// The marching operator gives each of 256 persistent workgroups a range of node planes, with one
// extra element layer per range and a serial chain of planes; below about half a million nodes a
// range is one or two planes, so half of the work is the extra layer and the rest is latency.
// Here a workgroup owns a tile of CX x CY element columns (all of z, at most 63 elements: 64 nodes) once:
//   stage    the nodes of (CX + 1) x (CY + 1) columns (constrained DOFs zeroed) and the tile's E in LDS;
//   elements a lane computes one element (as many whole columns per wavefront as fit in 64 lanes),
//            the hz = 1 results move one lane up, and the 12 node sums are added to the LDS
//            accumulators of the inner (CX - 1) x (CY - 1) node columns.  The columns of a round add
//            in four colours (x and y parity) with a barrier between them, so no two add to one node
//            at a time and the order is fixed: no atomics, the same bits every run;
//   nodes    the epilogue of the mode, every output written once.
// The host picks CX and CY for the grid: the fewest element columns on the busiest compute unit.
// It is bound by VALU issue (CX CY / ((CX - 1)(CY - 1)) times the grid's elements) and the load
// latencies of the two ends (half of the time at 120 x 56 x 48).  FP64 y = A x, 97 x 45 x 51, any K0:
// 24 us a call; the marching kernel takes 26 us after the read-back of K0 that its structure check
// needs (78 us a call).
#include <algorithm>

#include "common.hpp"
#include "op_tiled.hpp"
#include "stiffness.hpp"

namespace et {

namespace {

struct T3Args {
  Grid g;
  int cx, cy;     // element columns per tile
  int ntx;        // tiles along x
  int cpw;        // element columns per wavefront
};

constexpr int kT3Threads = 1024;

template <typename T>
struct T3Table {
  T g[48];
};

// MODE as in op_tiled.hpp.  FULL: K0 (24 x 24, row-major) in place of the table.
template <typename T, int MODE, bool FULL>
__global__ __launch_bounds__(kT3Threads) void op_tile3_kernel(const T3Table<T> Gk, const T3Args A,
                                                              const T* __restrict__ K0, const T* __restrict__ E,
                                                              const uint8_t* __restrict__ cons,
                                                              const T* __restrict__ x, const T* __restrict__ b,
                                                              const T* __restrict__ Dinv,
                                                              const double* __restrict__ omega, double wscale,
                                                              const T* __restrict__ xadd, T* __restrict__ y,
                                                              double* __restrict__ part, const T* __restrict__ dotv) {
  extern __shared__ __align__(16) unsigned char t3_lds[];
  constexpr bool kAdd = MODE == TM_JAC_ADD || MODE == TM_JAC_ADD_DOT;
  constexpr bool kJac = MODE == TM_JAC || MODE == TM_JAC0 || kAdd;
  constexpr bool kProd = MODE == TM_Y || MODE == TM_YDOT;
  const Grid& g = A.g;
  const int nx = g.nx(), ny = g.ny(), nz = g.nz(), ez_n = g.ez;
  const int CX = A.cx, CY = A.cy;
  const int ncol = (CX + 1) * (CY + 1), span = ncol * nz;        // staged nodes
  const int ocol = (CX - 1) * (CY - 1), ospan = ocol * nz;       // output nodes
  T* su = reinterpret_cast<T*>(t3_lds);  // [3][span]
  T* sa = su + 3 * span;                 // [3][ospan]
  T* se = sa + 3 * ospan;                // [CY][CX][nelz]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int X0 = blockIdx.x % A.ntx * (CX - 1), Y0 = blockIdx.x / A.ntx * (CY - 1);  // first output node
  // without constraints every constraint byte is read at byte 0 of E and masked to zero
  const uint8_t* cp = cons != nullptr ? cons : reinterpret_cast<const uint8_t*>(E);
  const int cmask = cons != nullptr ? ~0 : 0;
  const uint8_t cbyte = cons != nullptr ? (uint8_t)0xff : (uint8_t)0;
  const T w = kJac ? (T)((omega != nullptr ? *omega : 1.0) * wscale) : T(0);

  // FULL: whether K0 takes a rigid translation to zero but for the rounding of its entries (each
  // row's sum per component within 32 units of rounding of the row's largest entry).  Then only
  // differences of displacements are multiplied: the entries' rounding, times displacements that are
  // large beside their differences, was most of the error (97 x 45 x 51 smooth FP64 field: 6.2e-16 of
  // the result without, 3.5e-16 with; the transformed basis has no translations either).  The loads
  // also bring K0 near before the element rounds read it through the scalar cache: 33.6 -> 24.2 us
  // a call on new operands at that size.
  __shared__ int s_loose[2];
  if (FULL && wave < 2) {
    const int q = min(tid, 71), row = q / 3, d = q - 3 * row;
    T sum = T(0), big = T(0);
#pragma unroll
    for (int t = 0; t < 24; ++t) {
      const T v = K0[row * 24 + t];
      big = max(big, abs(v));
      sum += t % 3 == d ? v : T(0);
    }
    constexpr T kRound = T(32) * (sizeof(T) == 8 ? T(2.220446049250313e-16) : T(1.1920929e-7f));
    const bool loose = !(abs(sum) <= kRound * big);
    if (__builtin_amdgcn_ballot_w64(loose) != 0) {
      if (lane == 0) s_loose[wave] = 1;
    } else if (lane == 0) {
      s_loose[wave] = 0;
    }
  }

  // Stage, a node or element column per wavefront (lane = z, so the column's indices are scalar).
  // Loads are unconditional (clamped to the grid) and masks are applied at the store, so the loads
  // of kSC columns are in flight together.
  constexpr int kSC = 4, kWaves = kT3Threads / 64;
  const int kn = min(lane, nz - 1), ke = min(lane, ez_n - 1);
  for (int c0 = wave; c0 < ncol; c0 += kSC * kWaves) {
    T pu[kSC][3], pd[MODE == TM_JAC0 ? kSC : 1][3], pe[kSC];
    uint8_t pc[kSC][3];
    bool pin[kSC], ein[kSC];
#pragma unroll
    for (int m = 0; m < kSC; ++m) {
      const int c = min(c0 + m * kWaves, ncol - 1);
      const int j = c / (CX + 1), i = X0 - 1 + c - j * (CX + 1), jj = Y0 - 1 + j;
      pin[m] = i >= 0 && i < nx && jj >= 0 && jj < ny;
      const int d = ((min(max(jj, 0), ny - 1) * nx + min(max(i, 0), nx - 1)) * nz + kn) * 3;
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        pu[m][r] = MODE == TM_JAC0 ? b[d + r] : x[d + r];
        if (MODE == TM_JAC0) pd[MODE == TM_JAC0 ? m : 0][r] = Dinv[d + r];
        pc[m][r] = cp[(d + r) & cmask] & cbyte;
      }
      // element column c: there are fewer of them than node columns
      const int ce = min(c, CX * CY - 1), je = ce / CX, ex = X0 - 1 + ce - je * CX, ey = Y0 - 1 + je;
      ein[m] = ex >= 0 && ex < g.ex && ey >= 0 && ey < g.ey;
      pe[m] = E[(min(max(ex, 0), g.ex - 1) * g.ey + min(max(ey, 0), g.ey - 1)) * ez_n + ke];
    }
#pragma unroll
    for (int m = 0; m < kSC; ++m) {
      const int c = c0 + m * kWaves;
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        const T v = MODE == TM_JAC0 ? w * pd[MODE == TM_JAC0 ? m : 0][r] * pu[m][r] : pu[m][r];
        if (c < ncol && lane < nz) su[r * span + c * nz + lane] = pin[m] && pc[m][r] == 0 ? v : T(0);
      }
      if (c < CX * CY && lane < ez_n) se[c * ez_n + lane] = ein[m] ? pe[m] : T(0);
    }
  }
  for (int t = tid; t < 3 * ospan; t += kT3Threads) sa[t] = T(0);
  __syncthreads();
  const bool loose = FULL && (s_loose[0] | s_loose[1]) != 0;

  // nz lanes per column: the last one holds no element and only takes the results moved to node nelz
  const int lcol = lane / nz, lez = lane - lcol * nz;
  for (int q0 = 0; q0 < CX * CY; q0 += kWaves * A.cpw) {
    {
      const int q = q0 + wave * A.cpw + lcol;
      const bool valid = lcol < A.cpw && q < CX * CY;
      const int qc = min(q, CX * CY - 1);
      const int cj = qc / CX, ci = qc - cj * CX;
      const T e = valid && lez < ez_n ? se[(cj * CX + ci) * ez_n + min(lez, ez_n - 1)] : T(0);
      const T* uc = su + (cj * (CX + 1) + ci) * nz + lez;
      T u[3][8];  // corner bits hx + 2 hy + 4 hz
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int h = 0; h < 8; ++h) u[c][h] = uc[c * span + ((h & 1) + ((h >> 1) & 1) * (CX + 1)) * nz + (h >> 2)];
      // node sums of this element at the face corners f = hx + 2 hy
      T sum[4][3];
      // component c of the results at face corner f (lo: hz = 0, up: hz = 1)
      auto add = [&](int f, int c, T lo, T up) {
        const T moved = lane_shr(up);
        sum[f][c] = (lez < ez_n ? lo : T(0)) + (lez > 0 ? moved : T(0));
      };
      if constexpr (FULL) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const T base = loose ? T(0) : T(0.5) * (u[c][0] + u[c][7]);  // about the element's middle
#pragma unroll
          for (int h = 0; h < 8; ++h) u[c][h] = (u[c][h] - base) * e;
        }
        // scalar loads that the compiler may not hoist out of the column loop
        const __attribute__((address_space(4))) T* k = (const __attribute__((address_space(4))) T*)(const void*)K0;
        asm volatile("" : "+s"(k));
#pragma unroll
        for (int f = 0; f < 4; ++f)
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            T v[2] = {T(0), T(0)};
#pragma unroll
            for (int top = 0; top < 2; ++top)
#pragma unroll
              for (int a = 0; a < 8; ++a)
#pragma unroll
                for (int d = 0; d < 3; ++d)
                  v[top] = fma(k[(3 * h8_corner(f & 1, f >> 1, top) + c) * 24 + 3 * a + d],
                               u[d][hx(a) + 2 * hy(a) + 4 * hz(a)], v[top]);
            add(f, c, v[0], v[1]);
          }
      } else {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          wht8(u[c]);
#pragma unroll
          for (int h = 0; h < 8; ++h) u[c][h] *= e;
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const __attribute__((address_space(4))) T* gq =
              (const __attribute__((address_space(4))) T*)__builtin_amdgcn_kernarg_segment_ptr() + 16 * c;
          asm volatile("" : "+s"(gq));
          T yc[8];
          yc[0] = T(0);
          int gi = 0;
#pragma unroll
          for (int M = 1; M < 8; ++M) {
            T s = T(0);
#pragma unroll
            for (int d = 0; d < 3; ++d)
              if (wht_nz(M, c, d)) s = fma(gq[gi++], u[d][M ^ (1 << c) ^ (1 << d)], s);
            yc[M] = s;
          }
          wht8(yc);
#pragma unroll
          for (int f = 0; f < 4; ++f) add(f, c, yc[f], yc[f + 4]);
        }
      }
      // one colour (x and y parity) after the other adds to the accumulators
      const int mine = (ci & 1) + 2 * (cj & 1);
      for (int colour = 0; colour < 4; ++colour) {
        if (valid && mine == colour) {
          T old[4][3];
          int at[4];
          bool in[4];
#pragma unroll
          for (int f = 0; f < 4; ++f) {
            const int ti = ci + (f & 1) - 1, tj = cj + (f >> 1) - 1;
            in[f] = ti >= 0 && ti < CX - 1 && tj >= 0 && tj < CY - 1;
            at[f] = in[f] ? (tj * (CX - 1) + ti) * nz + lez : 0;
#pragma unroll
            for (int c = 0; c < 3; ++c) old[f][c] = sa[c * ospan + at[f]];
          }
#pragma unroll
          for (int f = 0; f < 4; ++f)
#pragma unroll
            for (int c = 0; c < 3; ++c)
              if (in[f]) sa[c * ospan + at[f]] = old[f][c] + sum[f][c];
        }
        __syncthreads();
      }
    }
  }

  // Nodes, a column per wavefront: the operands of kSN columns are requested together.
  constexpr int kSN = 3;
  double dot = 0.0;
  for (int c0 = wave; c0 < ocol; c0 += kSN * kWaves) {
    T pb[kSN][3], pd[kSN][3], pa[kSN][3], pt[kSN][3];
    uint8_t pc[kSN][3];
    int pdof[kSN], pown[kSN];
    bool live[kSN];
#pragma unroll
    for (int m = 0; m < kSN; ++m) {
      const int c = min(c0 + m * kWaves, ocol - 1);
      const int tj = c / (CX - 1), ti = c - tj * (CX - 1), i = X0 + ti, j = Y0 + tj;
      live[m] = c0 + m * kWaves < ocol && i < nx && j < ny && lane < nz;
      const int d = ((min(j, ny - 1) * nx + min(i, nx - 1)) * nz + kn) * 3;
      pdof[m] = d;
      pown[m] = ((tj + 1) * (CX + 1) + ti + 1) * nz + kn;
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        pc[m][r] = cp[(d + r) & cmask] & cbyte;
        pb[m][r] = kProd ? T(0) : b[d + r];
        pd[m][r] = kJac ? Dinv[d + r] : T(0);
        pa[m][r] = kAdd ? xadd[d + r] : T(0);
        if (MODE == TM_JAC_ADD_DOT) pt[m][r] = dotv[d + r];
      }
    }
#pragma unroll
    for (int m = 0; m < kSN; ++m) {
      if (!live[m]) continue;
      const int d = pdof[m], t = (c0 + m * kWaves) * nz + lane;
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        const bool fx = pc[m][r] != 0;
        T xv = su[r * span + pown[m]];  // zero where constrained
        if (fx) xv = MODE == TM_JAC0 ? w * pd[m][r] * pb[m][r] : x[d + r];
        const T ax = fx ? xv : sa[r * ospan + t];
        T v;
        if (kProd)
          v = ax;
        else if (MODE == TM_RES)
          v = pb[m][r] - ax;
        else
          v = xv + w * pd[m][r] * (pb[m][r] - ax);
        if (kAdd) v += pa[m][r];
        if (MODE == TM_YDOT) dot += (double)xv * (double)v;
        if (MODE == TM_JAC_ADD_DOT) dot += (double)pt[m][r] * (double)v;
        y[d + r] = v;
      }
    }
  }
  if (MODE == TM_YDOT || MODE == TM_JAC_ADD_DOT) {
    // fixed order: lanes, then wavefronts (the staged nodes have been read)
    double* s = reinterpret_cast<double*>(t3_lds);
    dot = wave_sum(dot);
    __syncthreads();
    if (lane == 0) s[wave] = dot;
    __syncthreads();
    if (tid == 0) {
      double r = 0.0;
      for (int v = 0; v < kT3Threads / 64; ++v) r += s[v];
      part[blockIdx.x] = r;
    }
  }
}

constexpr size_t kT3MaxLds = 160 * 1024 - 64;  // 64: the kernel's own

size_t t3_lds_bytes(const Grid& g, int cx, int cy, size_t elem_bytes) {
  return elem_bytes * ((size_t)3 * g.nz() * ((cx + 1) * (cy + 1) + (cx - 1) * (cy - 1)) + (size_t)cx * cy * g.ez);
}

// The tile with the least time on the busiest compute unit, in the measured proportion of a
// workgroup's ends (staging, epilogue) to a round of one element column set per wavefront, 1 : 1.
// One workgroup per compute unit at a time: 1024 threads with up to 128 registers each fill it.
T3Args t3_args(const Grid& g, size_t elem_bytes) {
  T3Args best{g, 0, 0, 0, 0};
  best.cpw = 64 / g.nz();
  const int round = kT3Threads / 64 * best.cpw;  // element columns per round
  int64_t cost = INT64_MAX;
  for (int cx = 3; cx <= 12; ++cx)
    for (int cy = 3; cy <= 12; ++cy) {
      if (t3_lds_bytes(g, cx, cy, elem_bytes) > kT3MaxLds) continue;
      const int64_t ntx = (g.nx() + cx - 2) / (cx - 1), nty = (g.ny() + cy - 2) / (cy - 1);
      // rounds first, then the columns in them
      const int64_t c = (ntx * nty + 255) / 256 * (((cx * cy + round - 1) / round + 1) * 256 + cx * cy / best.cpw);
      if (c < cost) {
        cost = c;
        best.cx = cx;
        best.cy = cy;
        best.ntx = (int)ntx;
      }
    }
  return best;
}

int t3_tiles(const T3Args& A) { return A.ntx * ((A.g.ny() + A.cy - 2) / (A.cy - 1)); }

template <typename T, int MODE, bool FULL>
void t3_launch(const T3Args& A, const T3Table<T>& Gk, const T* K0, const T* E, const uint8_t* cons, const T* x,
               const T* b, const T* Dinv, const double* omega, double wscale, const T* xadd, T* y, double* part,
               const T* dotv, hipStream_t s) {
  // once; the batched engine launches from several host threads
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&op_tile3_kernel<T, MODE, FULL>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)kT3MaxLds);
  (void)attr;
  const size_t lds = std::max(t3_lds_bytes(A.g, A.cx, A.cy, sizeof(T)), (size_t)(kT3Threads / 64) * sizeof(double));
  op_tile3_kernel<T, MODE, FULL><<<t3_tiles(A), kT3Threads, lds, s>>>(Gk, A, K0, E, cons, x, b, Dinv, omega, wscale,
                                                                     xadd, y, part, dotv);
}

}  // namespace

// Largest grid (nodes) of the tile operator.  A single call on a grid up to this size costs 14 us
// (9 537 nodes) to 36 us (410 865 nodes) in FP64, against 68 to 85 us with the read-back of K0.
static int64_t g_tile3_nodes = (int64_t)1 << 19;
void set_tile3_nodes(int64_t n) { g_tile3_nodes = n; }
int64_t get_tile3_nodes() { return g_tile3_nodes; }

bool tile3_active(const Grid& g, size_t elem_bytes) {
  return g.dim == 3 && get_wht() && g.nz() <= 64 && g.n_nodes() <= g_tile3_nodes && t3_args(g, elem_bytes).cx > 0;
}

// With the table known, per PCG iteration of the FP64 solver: 64x32x32 252 -> 235 us, 96x48x48
// 316 -> 291, 128x64x48 385 -> 359, but 48x24x24 191 -> 199; FP32 sweeps, whose marching kernel
// runs 16 wavefronts, gain nothing (96x48x48 mixed 239 -> 235, 120x56x48 249 -> 263).
bool tile3_faster(const Grid& g, size_t elem_bytes) {
  return elem_bytes == 8 && g.n_nodes() >= 50000 && tile3_active(g, elem_bytes);
}

int tile3_partials(const Grid& g, size_t elem_bytes) { return t3_tiles(t3_args(g, elem_bytes)); }

template <typename T>
int op_tile3(int mode, const Grid& g, const T* K0, const WhtTable* tab, const T* E, const uint8_t* cons, const T* x,
             const T* b, const T* Dinv, const double* omega, double wscale, const T* xadd, T* y, const T* dotv,
             double* part, hipStream_t s) {
  const T3Args A = t3_args(g, sizeof(T));
  ET_REQUIRE(A.cx > 0 && g.nz() <= 64, "tile operator: grid not supported");
#define ET_T3(M, FULL)                                                                                            \
  case M:                                                                                                         \
    t3_launch<T, M, FULL>(A, Gk, K0, E, cons, x, b, Dinv, omega, wscale, xadd, y, part, dotv, s);                 \
    break;
  T3Table<T> Gk{};
  if (tab == nullptr) {
    // single calls
    switch (mode) {
      ET_T3(TM_Y, true)
      ET_T3(TM_RES, true)
      ET_T3(TM_JAC, true)
      default: ET_REQUIRE(false, "tile operator: this mode takes the transformed basis");
    }
  } else if constexpr (sizeof(T) == 8) {
    for (int i = 0; i < 48; ++i) Gk.g[i] = (T)tab->g[i];
    switch (mode) {
      ET_T3(TM_Y, false)
      ET_T3(TM_RES, false)
      ET_T3(TM_JAC, false)
      ET_T3(TM_JAC_ADD, false)
      ET_T3(TM_YDOT, false)
      ET_T3(TM_JAC0, false)
      ET_T3(TM_JAC_ADD_DOT, false)
      default: ET_REQUIRE(false, "tile operator: unknown mode");
    }
  } else {
    ET_REQUIRE(false, "tile operator: the transformed basis runs in FP64");  // see tile3_faster
  }
#undef ET_T3
  ET_CHECK_LAUNCH();
  return ET_OK;
}

template int op_tile3<double>(int, const Grid&, const double*, const WhtTable*, const double*, const uint8_t*,
                              const double*, const double*, const double*, const double*, double, const double*,
                              double*, const double*, double*, hipStream_t);
template int op_tile3<float>(int, const Grid&, const float*, const WhtTable*, const float*, const uint8_t*,
                             const float*, const float*, const float*, const double*, double, const float*, float*,
                             const float*, double*, hipStream_t);

}  // namespace et
